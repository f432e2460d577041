"""Tiles of at most 64 routed rows: the ring of seven slots around every length a contraction can have against it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _forward_matches(H, I, counts):
    from oracle import moe_ffn
    from pipelink_amd.host import mok_inputs
    from pipelink_amd.host.mok import MoKSession, code_pitch
    from pipelink_amd.stages.mok import build as mok_build
    from test_gpu_moe import TOL, _oracle, _run

    paths = mok_build.images()
    inp = mok_inputs.generate(max(counts) + 3, H, I, len(counts), 1, seed=H + I, counts=counts)
    ref = _oracle(inp)
    ys = []
    for image in ("linked", "one_unit"):
        with MoKSession(paths[image].read_bytes(), str(paths["link_json"])) as sess:
            for launches in (1, 2):
                sess.launches(launches)
                y = _run(sess, inp, H, I, pitch_i=code_pitch(I))[2].float().numpy()
                assert sess.status() == 0 and not np.isnan(y).any() and moe_ffn.rel_frobenius(y, ref["y"]) <= TOL
                ys.append(y)
    assert all(np.array_equal(ys[0], other) for other in ys[1:])


# one fragment of routed rows (up to 32) at every length around the ring (6, 7, 8, 13, 14 and 15 slots among them), and beside two
# fragments and full tiles; averages an expert that neither cut nor divide a column tile
@pytest.mark.parametrize("H,I", [(64, 128), (192, 320), (384, 448), (512, 576), (832, 896), (960, 1024), (448, 960), (2880, 64)])
@pytest.mark.parametrize("counts,want", [([32, 1, 17], {"rows32"}), ([31, 20, 0, 32], {"rows32"}), ([40, 300, 1] + [0] * 4, {"rows32", "rows64", "wide"}),
                                         ([33, 16, 64], {"rows32", "rows64"})])
def test_forward_of_one_and_two_fragments_of_rows_matches_the_oracle(H, I, counts, want):
    from mok_route import kinds

    assert {{"full": "wide", "cols": "wide"}.get(k, k) for k in kinds(H, I, counts)} == want
    _forward_matches(H, I, counts)


# (rows 40, 300 and 1 of three experts are parts of 64 columns where parts_for says so)
# slots of the two contractions: one, less than a ring, a ring, one more, two rings and around them, odd and even; rows 33, 64 and
# beside an expert of few, of none and of more than a tile
@pytest.mark.parametrize("H,I", [(64, 128), (192, 320), (384, 448), (512, 576), (832, 896), (960, 1024), (2880, 64)])
@pytest.mark.parametrize("counts", [[33, 0, 64], [40, 300, 1]])
def test_forward_of_tiles_of_few_rows_matches_the_oracle(H, I, counts):
    _forward_matches(H, I, counts)
