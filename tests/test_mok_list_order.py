"""The order of a list's down tiles in a launch of both GEMMs: the expert in whose middle the list begins comes last."""
import pytest

from test_mok_schedule import BOTH, DOWN, enumerate_schedule  # noqa: F401 (fixture)


@pytest.mark.parametrize("gu,dn,counts", [(23, 12, [3, 0, 1, 40, 2, 2, 0, 1, 1, 1, 1, 1, 5]), (23, 12, [1037, 980, 1, 0, 256, 257, 255, 512, 3000]),
                                          (23, 12, [128] * 32), (3, 2, [300, 20]), (2, 5, [7] * 19)])
@pytest.mark.parametrize("op", [BOTH, DOWN])
def test_a_list_runs_the_rest_of_a_divided_expert_last(enumerate_schedule, op, gu, dn, counts):  # noqa: F811
    tiles, _, items = enumerate_schedule(op, gu, dn, counts)
    order = []   # the down tiles, numbered expert by expert, column tile by column tile, row tiles innermost
    for e, c in enumerate(counts):
        order += [(e, row, col) for col in range(dn) for row in range(-(-c // 256))]
    start = [sum(counts[:e]) for e in range(len(counts))]
    for q in range(8):
        first, end = q * len(order) // 8, (q + 1) * len(order) // 8
        want = order[first:end]
        if op == BOTH and first and end > first and order[first - 1][0] == order[first][0]:
            rest = [t for t in want if t[0] == want[0][0]]
            want = want[len(rest):] + rest if len(rest) < len(want) else want
        got = [(e, (row - start[e]) // 256, col // 256) for l, _, top, e, row, _, col, _, _ in items if l == q and top == DOWN]
        assert got == want
