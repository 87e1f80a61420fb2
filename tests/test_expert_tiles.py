"""Which tiles the experts' products take: thresholds on both sides, matrices that make too few blocks, inner sizes without whole
stages; and the router-independent promise that every size gets a tile the kernels know."""
import pytest

from ullm_amd.parts.moe import tile_rows_for


@pytest.mark.parametrize("experts,top,hidden,ff,expected", [
    (32, 4, 2048, 1024, {12: 16, 13: 64, 51: 64, 52: 128, 95: 128, 96: 128, 128: 256, 207: 256, 208: 128, 320: 256}),
    (8, 2, 1024, 512, {12: 16, 23: 16, 24: 32, 47: 32, 48: 64, 95: 64, 96: 128, 128: 256}),
    (32, 4, 2056, 1024, {13: 16, 24: 32, 52: 64, 96: 128, 320: 128}),
    (32, 4, 0, 0, {13: 16, 24: 32, 52: 64, 96: 128, 320: 128})])
def test_tiles_by_rows_an_expert(experts, top, hidden, ff, expected):
    for mean, rows in expected.items():
        assert tile_rows_for(mean * experts // top, top, experts, hidden, ff) == rows, mean
    assert all(tile_rows_for(t, top, experts, hidden, ff) in (16, 32, 64, 128, 256) for t in range(0, 5000, 7))
