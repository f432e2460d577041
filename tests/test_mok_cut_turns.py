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


@pytest.mark.gpu
@pytest.mark.parametrize("H,I,counts", [(320, 2432, [3, 1, 32, 9] * 4), (704, 2560, [1, 5] * 8)])
def test_forward_of_launches_of_two_turns(H, I, counts):
    forward_matches(H, I, counts)
