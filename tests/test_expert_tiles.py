"""Which tiles the experts' products take: near the best of those measured, few experts and columns, inner sizes without whole
stages and float32 among them; and that every size gets a tile the kernels know."""
import pytest

from ullm_amd.parts.moe import product_rows_for, tile_rows_for

# microseconds of gate|up and down in tiles of 16, 32, 64, 128 and 256 rows, by the mean of rows an expert
MEASURED = {
    (32, 4, 2048, 1024): {6: (68, 73, 93, 98, 111), 18: (116, 84, 95, 101, 109), 47: (249, 170, 93, 102, 109), 96: (490, 326, 113, 105, 119),
                          160: (None, None, 155, 129, 122), 256: (None, None, 223, 174, 191), 1024: (None, None, 703, 501, 469),
                          # over twelve routings by chance: past 128 rows of one expert a second round of blocks begins
                          44: (None, None, 95, 102, 110), 50: (None, None, 104, 102, 111), 56: (None, None, 110, 103, 112), 64: (None, None, 112, 105, 114),
                          92: (None, None, 113, 108, 118), 104: (None, None, 119, 126, 119), 128: (None, None, 141, 133, 120), 208: (None, None, 189, 137, 131)},
    (8, 2, 1024, 512): {6: (11, 12, 18, 23, 33), 24: (16, 14, 18, 25, 34), 96: (38, 30, 20, 29, 39), 128: (49, 36, 21, 31, 40),
                        160: (None, None, 21, 30, 41), 320: (None, None, 29, 32, 45), 1024: (None, None, 56, 61, 51)},
    (16, 4, 1024, 512): {96: (70, 54, 22, 33, 42), 128: (89, 66, 29, 35, 44), 320: (None, None, 39, 36, 50)},
    (8, 2, 2048, 1024): {36: (53, 43, 38, 47, 69), 96: (119, 86, 39, 54, 73), 128: (150, 106, 48, 56, 75), 320: (None, None, 71, 56, 81)},
    (64, 8, 2048, 768): {6: (102, 111, 132, 140, 168), 47: (386, 276, 132, 148, 174), 160: (None, None, 237, 213, 195)},
    (16, 4, 5120, 1536): {70: (675, 439, 230, 168, 221)},
    (4, 1, 2048, 4096): {290: (None, None, 150, 126, 148)}}


@pytest.mark.parametrize("sizes", sorted(MEASURED))
def test_tiles_near_the_best_of_those_measured(sizes):
    experts, top, hidden, ff = sizes
    for mean, times in MEASURED[sizes].items():
        taken = times[(16, 32, 64, 128, 256).index(tile_rows_for(mean * experts // top, top, experts, hidden, ff))]
        assert taken is not None and taken <= 1.05 * min(t for t in times if t), mean


@pytest.mark.parametrize("hidden,ff", [(2056, 1024), (2048, 1000), (0, 0)])
def test_sizes_without_whole_stages_and_float32(hidden, ff):
    for mean, rows in {13: 16, 24: 32, 52: 64, 96: 128, 320: 128}.items():
        assert tile_rows_for(mean * 8, 4, 32, hidden, ff) == rows, mean


@pytest.mark.parametrize("experts,top,hidden,ff", [(32, 4, 2048, 1024), (8, 2, 1024, 512), (1, 1, 64, 64), (32, 4, 2056, 1024), (0, 2, 2048, 1024)])
def test_every_size_gets_a_tile_the_kernels_know(experts, top, hidden, ff):
    for tokens in (*range(0, 5000, 7), 65536, 10 ** 6):
        rows = tile_rows_for(tokens, top, experts, hidden, ff)
        assert rows in (16, 32, 64, 128, 256)
        if rows == 256:                                # what that kernel's 32-bit offsets reach
            assert hidden % 64 == ff % 64 == 0 and (tokens * top + 256 * experts) * max(hidden, ff) < 2 ** 31


# us of gate|up and down in the tiles named, the mean over routings by chance, unequal experts and very unequal ones (up to 0.35 and 0.7 of
# the scores' spread apart).  Tiles of 256 were once taken from 16 rows on, which only routings by chance bear out
UNEQUAL = {
    (32, 4, 2048, 1024): {36: {64: 93, 128: 81, 256: 88}, 120: {128: 120, 256: 112}, 256: {128: 174, 256: 175}},
    (64, 8, 2048, 768): {42: {64: 137, 128: 131, 256: 138}},
    (16, 2, 5120, 1536): {36: {64: 160, 128: 159, 256: 183}, 48: {64: 176, 256: 198}, 256: {128: 316, 256: 300}},
    (40, 4, 1536, 1024): {36: {64: 77, 128: 82, 256: 88}, 106: {128: 106, 256: 115}},
    (32, 4, 4096, 512): {36: {64: 103, 256: 116}, 120: {128: 127, 256: 152}},
    (8, 2, 4096, 1536): {256: {128: 123, 256: 147}}}


@pytest.mark.parametrize("sizes", sorted(UNEQUAL))
def test_tiles_where_experts_are_unequal(sizes):
    experts, top, hidden, ff = sizes
    for mean, times in UNEQUAL[sizes].items():
        taken = times.get(product_rows_for(mean * experts // top, top, experts, hidden, ff))
        assert taken is not None and taken <= 1.02 * min(times.values()), mean


@pytest.mark.parametrize("sizes,mean,rows", [
    ((32, 4, 2048, 1024), 15, 16), ((32, 4, 2048, 1024), 20, 32), ((32, 4, 2048, 1024), 24, 128), ((32, 4, 2048, 1024), 84, 128), ((32, 4, 2048, 1024), 256, 256), ((64, 8, 2048, 768), 48, 128),
    ((16, 4, 5120, 1536), 16, 32), ((128, 8, 1024, 512), 40, 64), ((8, 2, 4096, 1536), 128, 64), ((8, 2, 1024, 512), 96, 64),
    ((32, 4, 2048, 1000), 96, 128), ((32, 4, 2056, 1024), 96, 128)])
def test_tiles_by_their_rows_where_experts_fill_a_round(sizes, mean, rows):
    experts, top, hidden, ff = sizes
    if rows not in (128, 256):
        rows = tile_rows_for(mean * experts // top, top, experts, hidden, ff)
        assert rows != 256
    assert product_rows_for(mean * experts // top, top, experts, hidden, ff) == rows
    assert product_rows_for(2 ** 31 // (top * hidden), top, experts, hidden, ff) <= 128          # past what 32-bit offsets reach
