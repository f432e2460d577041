"""Attention launches small enough for half tiles (64 queries a workgroup, a wave per half of each key block)."""
import numpy as np
import pytest
import torch

from test_attention import _bits

pytestmark = pytest.mark.gpu


# one and two query tiles; one block of keys and an odd number; windows that leave one half of the first block's keys
# invisible to some queries, that are one key, that are longer than the sequence; more tiles than a launch by itself would
# run as half tiles
@pytest.mark.parametrize("b,hq,hkv,s,window", [(1, 1, 1, 128, None), (2, 4, 2, 128, 1), (1, 4, 4, 256, 33), (1, 8, 2, 384, 97), (1, 4, 1, 640, None),
                                               (1, 2, 2, 512, 5000), (3, 32, 4, 512, None), (5, 7, 1, 1408, 200)])
def test_half_tiles_match_attention_in_64_bits(b, hq, hkv, s, window):
    from pipelink_amd.host.attention import open_session
    from pipelink_amd.stages.attention import build as fa_build

    g = torch.Generator().manual_seed(s + b)
    q, k, v = (torch.randn(b, h, s, 128, generator=g).to(torch.bfloat16) for h in (hq, hkv, hkv))
    link_json = fa_build.images()["window_half_linked" if window else "half_linked"].parent / "link.json"
    sess = open_session(link_json, _bits(q), _bits(k), _bits(v), window=window)
    sess.write("o", np.full((b, s, hq * 128), 0x7FC0, dtype=np.uint16))
    sess.launch()
    sess.synchronize()
    got = torch.from_numpy(sess.read("o").view(np.int16).copy()).view(torch.bfloat16).double().view(b, s, hq, 128)
    sess.close()
    pos = torch.arange(s)
    seen = pos[None, :] <= pos[:, None]
    if window:
        seen &= pos[None, :] > pos[:, None] - window
    for head in sorted({0, hq // 2, hq - 1}):
        kv = head // (hq // hkv)
        for n in sorted({0, b - 1}):
            score = (q[n, head].double() @ k[n, kv].double().T / 128 ** 0.5).masked_fill(~seen, -torch.inf)
            want = score.softmax(-1) @ v[n, kv].double()
            # probabilities and result in bf16 (2^-9 each, relative): the bar the other attention tests use
            assert (got[n, :, head] - want).norm() / want.norm() <= 5e-3


def test_an_image_of_the_other_tile_size_covers_the_whole_output():
    """An image beside a link (a session's second one, or one the caller names) has the link's grid, not its own."""
    from pathlib import Path

    from pipelink_amd.host.attention import open_session
    from pipelink_amd.stages.attention import build as fa_build

    images = fa_build.images()
    g = torch.Generator().manual_seed(7)
    q, k, v = (_bits(torch.randn(2, h, 640, 128, generator=g).to(torch.bfloat16)) for h in (4, 2, 2))

    def run(sess):
        sess.write("o", np.full((2, 640, 512), 0x7FC0, dtype=np.uint16))
        sess.launch()
        sess.synchronize()
        return sess.read("o")

    sess = open_session(images["link_json"], q, k, v)                                   # 40 tiles: half tiles
    half = run(sess)
    whole = run(sess.with_image(images["linked"]))
    sess.close()
    sess = open_session(images["link_json"], q, k, v, image=images["linked"])
    assert np.array_equal(run(sess), whole) and np.array_equal(run(sess.with_image(images["half_linked"])), half)
    sess.close()
    for link, image in ((images["link_json"], images["half_linked"]), (Path(images["half_linked"]).parent / "link.json", None)):
        sess = open_session(link, q, k, v, image=image)
        assert np.array_equal(run(sess), half)
        sess.close()
    assert not np.array_equal(whole, half) and not (half == 0x7FC0).any() and not (whole == 0x7FC0).any()
