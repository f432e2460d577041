"""Tiles of 33 to 64 routed rows: the ring of seven slots around every length a contraction can have against it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# slots of the two contractions: one, less than a ring, a ring, one more, two rings and around them, odd and even; rows 33, 64 and
# beside an expert of few, of none and of more than a tile
@pytest.mark.parametrize("H,I", [(64, 128), (192, 320), (384, 448), (512, 576), (832, 896), (960, 1024), (2880, 64)])
@pytest.mark.parametrize("counts", [[33, 0, 64], [40, 300, 1]])
def test_forward_of_tiles_of_few_rows_matches_the_oracle(H, I, counts):
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
