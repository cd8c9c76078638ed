"""The forward-only kernel (the loss under no_grad, lncc_map) where its tiles can go wrong: widths
around 48- and 64-column tiles and their overlaps, rows around 28 and 32, columns that a lane of
three or four straddles, chunk seams, more pieces than workgroups, empty tiles of padding."""
import numpy as np
import pytest
import torch

import oracle as O
import workloads as wl
from checks import RATIO
from fused_lncc import ext, fused_lncc_loss, lncc_map

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [
    (1, 2, 5, 27, 40), (1, 1, 7, 28, 47), (1, 1, 6, 29, 48), (1, 2, 5, 32, 49), (1, 1, 9, 33, 63), (1, 1, 4, 31, 64),
    (1, 1, 5, 56, 65), (1, 1, 3, 65, 90), (1, 1, 2, 20, 131), (1, 1, 1, 17, 1), (1, 1, 40, 3, 17), (2, 1, 18, 1, 200),
]


def check(p, t, k, dtype=torch.float32, dr=1e-5):
    """Loss and map against the float64 oracle, bounded by RATIO times the error of the reference's own
    float32 arithmetic on the same values (the loss is their mean: at most its largest error), or by
    float32's rounding of the result."""
    pd, td = p.to(dtype).to(DEV), t.to(dtype).to(DEV)
    pn, tn = pd.float().cpu().numpy(), td.float().cpu().numpy()
    with torch.no_grad():
        loss = fused_lncc_loss(pd, td, k, dr).item()
    m = lncc_map(pd, td, k, dr).double().cpu().numpy()
    l64, _, maps = O.lncc(pn, tn, k, dr, grad=True, maps=True)
    l32, _, m32 = O.lncc_ref32(pn, tn, k, dr, grad=True, ncc_map=True)
    err32 = np.abs(m32.astype(np.float64) - maps["ncc"])
    assert np.abs(m - maps["ncc"]).max() <= max(RATIO * err32.max(), 1e-5)
    bound = max(RATIO * max(abs(l32 - l64), err32.mean()), 2e-7)
    assert abs(loss - l64) <= bound
    return l64, bound


@pytest.mark.parametrize("k", [3, 5, 7, 9])
@pytest.mark.parametrize("shape", SHAPES)
def test_tile_edges(shape, k):
    check(*wl.randn_pair(shape, 100 * k + shape[4]), k)


@pytest.mark.parametrize("k", [3, 5, 7, 9])
@pytest.mark.parametrize("width", [49, 50, 51, 52, 93, 94, 95, 96, 97, 121, 122, 123, 124, 125, 193])
def test_last_tile_starts_early(width, k):
    """Every remainder of a row's last tile by the lane's three or four columns, two to five tiles a row:
    no column of the map left out or taken from the wrong tile, none counted twice in the loss."""
    check(*wl.randn_pair((1, 2, 4, 9, width), 10 * width + k), k)


@pytest.mark.parametrize("k", [3, 5, 7, 9])
def test_bf16_odd_rows(k):
    check(*wl.randn_pair((1, 2, 6, 30, 51), k), k, torch.bfloat16)


@pytest.mark.parametrize("k", [3, 7, 9])
@pytest.mark.parametrize("dchunk", [1, 4, 7])
def test_chunk_seams(k, dchunk, force_dchunk):
    force_dchunk(dchunk)
    check(*wl.randn_pair((1, 2, 23, 30, 50), k + dchunk), k)


@pytest.mark.parametrize("k", [5, 9])
def test_more_pieces_than_workgroups(k):
    """700 volumes: a workgroup takes several pieces in turn, each with its own march."""
    check(*wl.randn_pair((700, 1, 3, 18, 9), k), k)


def test_partial_sums_past_the_grid_are_zero():
    """The reduction reads the gradient plan's partials; the forward launch, with fewer workgroups,
    leaves none of an earlier call's there."""
    p, t = wl.randn_pair((1, 3, 40, 65, 33), 5)
    pd, td = p.to(DEV), t.to(DEV)
    pf, tf = pd.reshape(3, 40, 65, 33), td.reshape(3, 40, 65, 33)
    loss = ext.loss_grad(pf, tf, 3, 1e-5, False)[0]
    lib = ext._lib.load()
    ws = torch.full((ext.workspace_bytes(pf.shape, 3) // 8,), float("nan"), dtype=torch.float64, device=DEV)
    again = torch.empty((), device=DEV)
    ext._lib.check(lib.fl_lncc_loss_grad(pf.data_ptr(), tf.data_ptr(), 0, *pf.shape, 3, 1e-5, again.data_ptr(), None,
                                         ws.data_ptr(), ws.numel() * 8, torch.cuda.current_stream().cuda_stream))
    assert again.item() == loss.item()


@pytest.mark.parametrize("where", [(0, 0, 0), (2, 31, 44), (4, 60, 95)])
def test_nan_reaches_the_loss(where):
    p, t = wl.randn_pair((1, 1, 5, 61, 96), 3)
    p[(0, 0) + where] = float("nan")
    with torch.no_grad():
        assert torch.isnan(fused_lncc_loss(p.to(DEV), t.to(DEV), 7)).item()


@pytest.mark.parametrize("dr", [0.0, 1e-20])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("k", [3, 5, 7, 9])
@pytest.mark.parametrize("shape", [(1, 2, 9, 75, 40), (1, 1, 17, 32, 32), (1, 1, 5, 96, 96)])
def test_windows_past_the_volume_do_not_reach_the_loss(shape, k, dtype, dr):
    """Tiles reach past the volume by more than h rows or columns, where a window is all zeros: at a
    smooth_dr of 0 (or one whose square has no float32 reciprocal) its ncc is 0 * inf, which counts in
    no loss. With and without a gradient the loss is the oracle's."""
    p, t = wl.randn_pair(shape, 7 * k + shape[3])
    l64, bound = check(p, t, k, dtype, dr)
    with_grad = fused_lncc_loss(p.to(dtype).to(DEV).requires_grad_(True), t.to(dtype).to(DEV), k, dr).item()
    assert abs(with_grad - l64) <= bound
