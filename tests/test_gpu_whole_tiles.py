"""Whole column tiles, also where a session's launch would run parts of 64 columns: through the owners' host-ABI providers, which
offer none.  Full tiles, their stores and their activation, with column tails, odd contractions and several row tiles an expert."""
import json

import numpy as np
import pytest
import torch

from mok_route import kinds, tiles
from oracle import moe_ffn, mxfp8
from test_gpu_moe import CASES, TOL, _oracle, _random_cases, _run, cell  # noqa: F401 (fixture)

pytestmark = pytest.mark.gpu


def _owners(image: bytes, link: dict, inp, H, I, pitch, passes, limit=7.0):
    """hidden_q, hidden_sc, y of launches by the providers: both GEMMs in one (passes (0,)) or one after the other."""
    from pipelink_amd.host import broker
    from pipelink_amd.host.backend import HipBackend
    from pipelink_amd.host.mok import scale_pitch, weight_codes_to_k64_tiled, weight_scales_to_slot_major

    dev = torch.device("cuda:0")
    t = {n: v.to(dev) for n, v in inp.__dict__.items()}
    for name, k in (("w_gate", H), ("w_up", H), ("w_down", I)):
        t[name + "_q"], t[name + "_sc"] = weight_codes_to_k64_tiled(t[name + "_q"], k), weight_scales_to_slot_major(t[name + "_sc"], k)
    rows, experts = int(inp.tokens_per_expert.sum()), len(inp.tokens_per_expert)
    words = 32 + (rows + 255) // 256 + experts
    t["hidden_q"] = torch.full((rows, pitch), 0xFF, dtype=torch.uint8, device=dev)
    t["hidden_sc"] = torch.full((rows, scale_pitch(I)), 0xFF, dtype=torch.uint8, device=dev)
    t["y"] = torch.full((rows, H), float("nan"), dtype=torch.bfloat16, device=dev)
    t["workspace"] = torch.zeros(words, dtype=torch.int32, device=dev)
    res = lambda n: broker.Resource(t[n].data_ptr(), t[n].numel() * t[n].element_size())
    resources = {"mok.framework": {n: res(n) for n in ("tokens_per_expert", "workspace")},
                 "mok.gemm": {n: res(n) for n in ("x_q", "x_sc", "w_gate_q", "w_gate_sc", "w_up_q", "w_up_sc", "w_down_q", "w_down_sc",
                                                  "hidden_q", "hidden_sc", "y", "row_token")},
                 "mok.act": {n: res(n) for n in ("hidden_q", "hidden_sc")}}
    scalars = {"mok.num_local_tokens": inp.x_q.shape[0], "mok.hidden": H, "mok.intermediate": I, "mok.num_local_experts": experts,
               "mok.swiglu_limit": limit, "mok.precision": 1, "mok.routed_rows": rows, "mok.ld_q_h": H, "mok.ld_q_i": pitch,
               "mok.ld_sc_h": scale_pitch(H), "mok.ld_sc_i": scale_pitch(I), "mok.workspace_words": words}
    be = HipBackend(0, torch.cuda.current_stream().cuda_stream)
    for pass_ in passes:
        with broker.open_host(link, image, resources, dict(scalars, **{"mok.pass": pass_}), be) as s:
            s.launch()
            be.synchronize()
    assert not t["workspace"].cpu().any()
    return t["hidden_q"][:, :I].cpu().numpy(), t["hidden_sc"].cpu().numpy()[:, :I // 32], t["y"].cpu()


def _same(a, b) -> bool:
    return np.array_equal(a[0], b[0]) and np.array_equal(a[1], b[1]) and torch.equal(a[2].view(torch.int16), b[2].view(torch.int16))


def _check(cell, inp, H, I):  # noqa: F811
    """Whole tiles in one launch and in two against the oracle, and against the session, whatever tiles that chooses."""
    from pipelink_amd.host.mok import code_pitch
    from pipelink_amd.stages.mok import build as mok_build

    counts = inp.tokens_per_expert.tolist()
    whole = tiles(H, I, counts, parts=False)
    assert not {"part"} & kinds(H, I, counts, parts=False)
    # what this test is for: full tiles where there are rows and columns for them
    assert ("gate_up_full" in whole) == (I > 64 and max(counts) > 64) and ("down_full" in whole) == (H > 64 and max(counts) > 64)
    paths = mok_build.images()
    link, ref = json.loads(paths["link_json"].read_text()), _oracle(inp)
    first = None
    for image in ("linked", "one_unit"):
        for pitch, passes in ((code_pitch(I), (0,)), (I, (1, 2))):
            hq, hsc, y = got = _owners(paths[image].read_bytes(), link, inp, H, I, pitch, passes)
            assert torch.isfinite(y.float()).all() and moe_ffn.rel_frobenius(y.float().numpy(), ref["y"]) <= TOL
            padded = np.zeros((hq.shape[0], -(-(I // 32) // 16) * 16), np.uint8)
            padded[:, :I // 32] = hsc
            assert moe_ffn.rel_frobenius(mxfp8.mx_dequantize(hq, padded), mxfp8.mx_dequantize(ref["hidden_q"], ref["hidden_sc"])) <= TOL
            assert first is None or _same(got, first)
            first = first or got
    hq, hsc, y = _run(cell[0], inp, H, I, pitch_i=code_pitch(I))
    assert _same((hq, hsc[:, :I // 32], y), first)   # parts: the same sums in the same order
    return kinds(H, I, counts)


@pytest.mark.parametrize("T,H,I,E,k,seed,conc", CASES + _random_cases(16, 7))
def test_whole_tiles_match_the_oracle_and_the_session(cell, T, H, I, E, k, seed, conc):  # noqa: F811
    from pipelink_amd.host import mok_inputs

    print(f"case T={T} H={H} I={I} E={E} k={k} seed={seed} conc={conc}", flush=True)
    _check(cell, mok_inputs.generate(T, H, I, E, k, seed=seed, concentrate=conc), H, I)


# row tiles of an expert that end in 1 and in 56 rows beside full ones, a single full one, none; both GEMMs with a column tail and an
# odd contraction; down tiles on other XCDs' lists than the gate/up tiles they wait for
@pytest.mark.parametrize("H,I,counts", [(256, 384, [257, 1025, 0, 1080, 256]), (320, 448, [300, 0, 513]), (512, 640, [512] * 8)])
def test_whole_tiles_of_several_row_tiles_an_expert(cell, H, I, counts):  # noqa: F811
    from pipelink_amd.host import mok_inputs

    assert "part" in _check(cell, mok_inputs.generate(max(counts), H, I, len(counts), 1, seed=H, counts=counts), H, I)   # (in the session)


def test_whole_tiles_of_the_unclamped_image_match_the_unclamped_oracle():
    from pipelink_amd.host import mok_inputs
    from pipelink_amd.stages.mok import build as mok_build

    link_dir = mok_build.HERE / "build_unclamped" / "link"
    inp = mok_inputs.generate(200, 256, 192, 3, 2, seed=9)
    inp.w_gate_sc, inp.w_up_sc = ((s.to(torch.int16) + 3).to(torch.uint8) for s in (inp.w_gate_sc, inp.w_up_sc))   # weights x 8: beyond the limit
    assert "gate_up_full" in tiles(256, 192, inp.tokens_per_expert.tolist(), parts=False)
    link = json.loads((link_dir / "link.json").read_text())
    free, clamped = _oracle(inp, limit=None), _oracle(inp, limit=1.0)
    for pitch, passes in ((256, (0,)), (192, (1, 2))):
        y = _owners((link_dir / "pipeline.hsaco").read_bytes(), link, inp, 256, 192, pitch, passes, limit=1.0)[2].float().numpy()
        assert moe_ffn.rel_frobenius(y, free["y"]) <= TOL < moe_ffn.rel_frobenius(clamped["y"], free["y"]) / 10
