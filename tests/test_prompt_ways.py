"""How a prompt launch of the matrix-core attention goes, by its tiles, their keys and a window: near the best of those measured."""
import ctypes

import pytest

from ullm_amd.kernels import build
from ullm_amd.parts import StepShape
from ullm_amd.parts.attention import plan_attention_step


def _way(entries, nq, nkv, window=0, hd=128, units=256):
    f = plan_attention_step(StepShape(tuple(n for n, _ in entries), tuple(s for _, s in entries))).facts
    i, long = ctypes.c_int, ctypes.c_longlong
    return build.load("attention_mfma").ullm_attention_prefill_way(
        i(f["num_tiles"]), long(f["tile_keys_total"]), i(f["tile_keys_max"]), i(f["num_wide"]), long(f["wide_keys_total"]),
        i(f["wide_keys_max"]), i(nq), i(nkv), i(hd), i(window), i(units))


# (new tokens, keys before them) of the requests, heads, kv heads, window: us of the ways (1, 2: parts of the keys; 3: four; 4, 5: tiles of 64
# tokens, whole and in halves)
MEASURED = [([(130, 0)], 32, 8, 0, {1: 8.7, 2: 10.3}), ([(33, 287)], 16, 8, 0, {1: 13.7, 2: 12.7, 3: 13.8}),
            ([(33, 967)], 16, 8, 128, {1: 12.4, 2: 11.5, 3: 12.5}), ([(33, 967)], 16, 8, 200, {1: 13.3, 2: 12.5, 3: 12.2}),
            ([(130, 870)], 16, 8, 256, {1: 16.0, 2: 14.5, 3: 14.0, 4: 19.3, 5: 17.9}), ([(130, 870)], 32, 8, 256, {1: 16.9, 2: 15.8}),
            ([(2048, 0)], 16, 8, 256, {1: 19.9, 3: 28.2}), ([(2048, 0)], 16, 8, 512, {1: 28.5, 3: 34.3}),
            ([(300, 700)] * 16, 16, 8, 256, {1: 52.1, 2: 75.4, 3: 71.8, 4: 42.1, 5: 56.4}), ([(300, 0)] * 8, 16, 8, 0, {1: 20.4, 5: 23.3}),
            ([(700, 2100)], 16, 8, 0, {2: 57, 3: 40, 4: 87, 5: 59}), ([(2048, 0)], 16, 8, 0, {2: 53, 3: 43, 4: 66, 5: 47}),
            ([(3000, 0)], 16, 8, 0, {1: 92, 3: 83, 4: 93, 5: 63}), ([(8000, 0)], 16, 8, 0, {1: 523, 3: 402, 4: 304, 5: 321})]


@pytest.mark.parametrize("case", range(len(MEASURED)))
def test_near_the_best_of_those_measured(case):
    entries, nq, nkv, window, times = MEASURED[case]
    taken = times.get(_way(entries, nq, nkv, window))
    assert taken is not None and taken <= 1.03 * min(times.values())


def test_ways_of_other_heads():
    for entries in ([(300, 700)] * 16, [(8000, 0)], [(40, 280)], [(17, 0)]):
        assert _way(entries, 16, 8, hd=256) == 1 and _way(entries, 16, 8, hd=64) in (1, 2) and _way(entries, 32, 8) in (1, 2)
