"""The device quantiser and the weight layout conversions at the edges of their kernels' pieces, against the oracle (bit
for bit) and numpy's transpositions."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import mxfp8

pytestmark = pytest.mark.gpu


# a row of 4 pieces and up; rows that end inside a workgroup's 1024 pieces, at its end and one behind; a piece's row more
# than one row on; pitches that are no multiple of 8, and pads longer than a row has pieces
@pytest.mark.parametrize("rows,k,pad", [(1, 32, 0), (3, 32, 4), (256, 32, 96), (257, 32, 60), (1025, 64, 0), (7, 2848, 20),
                                        (64, 128, 0), (65, 128, 128), (129, 2880, 64), (2, 32768, 0)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_quantiser_at_the_edges_of_its_pieces(rows, k, pad, dtype):
    from pipelink_amd.host.mok import mxfp8_quantize_device, scale_pitch

    g = torch.Generator().manual_seed(rows + k)
    x = torch.randn(rows, k, generator=g) * torch.exp2(torch.randint(-130, 120, (rows, 1), generator=g).float())
    x[0, 0], x[-1, -1], x[-1, 0] = float("nan"), -float("inf"), -0.0
    x[rows // 2, k - 32:] = 0
    # the values start 8 bytes (bf16) or 16 bytes (fp32) into their allocation
    room = torch.empty(rows * k + 4, dtype=dtype, device="cuda")
    src = room[4:].view(rows, k)
    src.copy_(x.to(dtype))
    q, sc = mxfp8_quantize_device(src, pitch=k + pad)
    oq, osc = mxfp8.mx_quantize(x.to(dtype).float().numpy())
    assert q.shape == (rows, k + pad) and sc.shape == (rows, scale_pitch(k))
    assert np.array_equal(q[:, :k].cpu().numpy(), oq) and not q[:, k:].any()
    assert np.array_equal(sc[:, :k // 32].cpu().numpy(), osc[:, :k // 32]) and not sc[:, k // 32:].any()


# one row to one behind a workgroup's; one column, an odd number, a pair of them and one more; a scale row that is no
# multiple of four bytes, one that holds one dword more than it needs, more slots than a workgroup's
@pytest.mark.parametrize("e,n,k,ld,ld_sc", [(1, 1, 64, 64, 2), (3, 127, 192, 208, 6), (2, 129, 128, 128, 4), (5, 64, 320, 336, 11),
                                            (2, 65, 2880, 2880, 96), (33, 31, 4224, 4224, 136)])
def test_weight_layouts_at_the_edges_of_their_tiles(e, n, k, ld, ld_sc):
    from pipelink_amd.host.mok import weight_codes_to_k64_tiled, weight_scales_to_slot_major

    g = torch.Generator().manual_seed(n)
    q = torch.randint(0, 256, (e, n, ld), dtype=torch.uint8, generator=g)
    sc = torch.randint(0, 256, (e, n, ld_sc), dtype=torch.uint8, generator=g)
    tiled = weight_codes_to_k64_tiled(q.cuda(), k).cpu().numpy()
    assert np.array_equal(tiled, q.numpy()[:, :, :k].reshape(e, n, k // 64, 64).transpose(0, 2, 1, 3))
    slots = (k + 127) // 128
    want = np.zeros((e, n, 4 * slots), np.uint8)
    want[:, :, :k // 32] = sc.numpy()[:, :, :k // 32]
    want = want.reshape(e, n, slots, 4).transpose(0, 2, 1, 3)
    assert np.array_equal(weight_scales_to_slot_major(sc.cuda(), k).cpu().numpy(), want)
    # scale bytes that do not start on a dword
    room = torch.empty(e * n * ld_sc + 1, dtype=torch.uint8, device="cuda")
    room[1:].copy_(sc.flatten())
    assert np.array_equal(weight_scales_to_slot_major(room[1:].view(e, n, ld_sc), k).cpu().numpy(), want)


def test_quantiser_of_the_plain_entry_leaves_the_pad_alone():
    from pipelink_amd.host.backend import check, load_library

    lib = load_library()
    x = torch.randn(9, 96, device="cuda")
    q = torch.full((9, 128), 0xA5, dtype=torch.uint8, device="cuda")
    sc = torch.empty((9, 3), dtype=torch.uint8, device="cuda")   # a scale pitch without padding
    check(lib, lib.plk_mxfp8_quantize(x.data_ptr(), 0, 9, 96, q.data_ptr(), 128, sc.data_ptr(), 3,
                                      ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))
    oq, osc = mxfp8.mx_quantize(x.cpu().numpy())
    assert np.array_equal(q[:, :96].cpu().numpy(), oq) and bool((q[:, 96:] == 0xA5).all())
    assert np.array_equal(sc.cpu().numpy(), osc[:, :3])


def test_scale_layout_of_more_rows_than_one_launch_has_threads_for():
    """2^30 rows and a few: four threads a row are 2^32 (1 GB of scale bytes, 4 GB of dwords)."""
    from pipelink_amd.host.mok import weight_scales_to_slot_major

    n = (1 << 30) + 65
    sc = torch.randint(0, 256, (1, n, 1), dtype=torch.uint8, device="cuda")
    got = weight_scales_to_slot_major(sc, 32).view(n, 4)
    for first in range(0, n, 1 << 28):
        assert torch.equal(got[first:first + (1 << 28), 0], sc[0, first:first + (1 << 28), 0]) and not got[first:first + (1 << 28), 1:].any()
