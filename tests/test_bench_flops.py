"""What the benchmark says its launch multiplies beyond the algorithmic count, against the placements the kernel has."""
import bench


def test_tiles_of_few_rows_are_counted_as_they_are_multiplied():
    per_row_tile = {c: bench.executed_flops([c]) for c in (1, 32, 33, 64, 65, 128, 129, 256)}
    assert per_row_tile[1] == per_row_tile[32] and per_row_tile[33] == per_row_tile[64] == 2 * per_row_tile[32]   # one or two fragments of rows
    tiles = -(-bench.I // 128) * 2 * 128 * bench.H + -(-bench.H // 256) * 256 * bench.I   # weight rows x contraction, whole column tiles
    assert per_row_tile[64] == 2.0 * 64 * tiles
    assert per_row_tile[65] == per_row_tile[128] < per_row_tile[129] == per_row_tile[256]
    assert bench.executed_flops([256 + 7, 0, 64]) == per_row_tile[256] + per_row_tile[32] + per_row_tile[64]
