"""Registers of the 32-bit tiled attention, as the compiled library states them: nothing in scratch memory (a word there is a
trip to memory every tile that also waits for the loads under way), and as many blocks of four waves a unit as each head size had
when its values were asked for only when they were needed."""
import re

from ullm_amd.kernels import build as kb

LANE_REGISTERS = 512            # of a SIMD, for a lane of each of its waves; one wave of a block on each of a unit's four


def compiled_kernels():
    with open(kb.compile_family("attention_generic", verbose=False), "rb") as f:
        text = f.read()
    number = rb"(?:[\x00-\x7f]|\xcc.|\xcd..)"
    for m in re.finditer(rb"\.name\xd9.(_Z\w+)\xbb\.private_segment_fixed_size(" + number + rb")(.*?)\xab\.vgpr_count(" + number + rb")", text, re.S):
        value = [int.from_bytes(v if v[0] < 0x80 else v[1:], "big") for v in (m.group(2), m.group(4))]
        yield m.group(1).decode(), value[0], value[1]


def test_no_scratch_and_no_fewer_blocks():
    seen = {}
    for name, scratch, registers in compiled_kernels():
        m = re.match(r"_Z28paged_attention_tiles_kernelI([ft])Li(\d+)ELb([01])E", name)
        if m:
            seen[m.group(1), int(m.group(2)), m.group(3)] = (scratch, LANE_REGISTERS // (-(-registers // 8) * 8))
    sizes = [1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16]
    assert sorted(seen) == sorted((t, k, p) for t in "ft" for k in sizes for p in "01")
    for (kind, chunks, _), (scratch, blocks) in seen.items():
        three, two = (2, 8) if kind == "f" else (4, 12)
        assert scratch == 0, (kind, chunks)
        assert blocks >= (3 if chunks <= three else 2 if chunks <= two else 1), (kind, chunks, blocks)
