"""Where quarters of down tiles fill the second turn that a launch's whole tiles take anyway: the rule at its edges (CPU), the
forward of such launches (GPU)."""
import subprocess

import pytest

from test_mok_narrow import SCHEDULE, _compile, test_forward_of_few_rows_matches_the_oracle as forward_matches


@pytest.mark.parametrize("gu,dn,experts,parts", [
    (19, 2, 16, (1, 4)),     # 304 + 32 whole, 304 + 128 with quarters: two turns either way, above the line of 299 tasks
    (20, 3, 16, (1, 4)),     # 512 tasks with quarters: the second turn is full
    (23, 3, 16, (1, 1)),     # 560: a third turn
    (15, 4, 13, (1, 1)),     # 247 whole, one turn; 403 with quarters is above the line of 243
    (15, 5, 12, (1, 1)),     # 240 whole; 420
    (24, 12, 7, (1, 1)),     # 84 down tiles: not all their quarters run at once
])
def test_quarters_within_two_turns(tmp_path, gu, dn, experts, parts):
    out = subprocess.run([_compile(tmp_path, SCHEDULE), "0", str(gu), str(dn)] + ["1"] * experts, check=True, capture_output=True, text=True).stdout.split()
    assert tuple(map(int, out[:2])) == parts


# contractions of one to four slots (64 columns and more; what the rule knows is that a column tile's columns are at least begun)
@pytest.mark.parametrize("gu,dn,counts,parts", [
    (1, 1, [4, 0, 0, 0], (1, 1)), (1, 1, [2, 1], (1, 1)), (1, 1, [13, 11, 12], (1, 1)),                # 64 x 64, 128 x 128: 11.1 us whole, 12.4 cut
    (2, 1, [16], (1, 1)), (2, 1, [1, 0, 3, 0], (1, 1)), (2, 1, [1, 1, 1, 2], (1, 1)), (2, 1, [9, 9, 9], (1, 1)),   # 256 x 256
    (4, 1, [1], (1, 4)),                                                                              # 256 x 512: seven slots of down contraction
    (2, 2, [1], (4, 4)),                                                                              # 512 x 256: 15.9 us whole, 14.0
    (2, 2, [1] * 3, (1, 1)),
])
def test_the_shortest_contractions_are_not_cut(tmp_path, gu, dn, counts, parts):
    out = subprocess.run([_compile(tmp_path, SCHEDULE), "0", str(gu), str(dn), *map(str, counts)], check=True, capture_output=True, text=True).stdout.split()
    assert tuple(map(int, out[:2])) == parts


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,counts", [(320, 2432, [3, 1, 32, 9] * 4), (704, 2560, [1, 5] * 8)])
def test_forward_of_launches_of_two_turns(H, I, counts):
    forward_matches(H, I, counts)
