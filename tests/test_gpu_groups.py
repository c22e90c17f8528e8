"""Slices taken together by one workgroup, and launches on small tiles: bit
for bit the slices of the one-slice kernel on 64x64 tiles, which the parity
tests hold against the oracle. The same additions in the same order leave no
room for a tolerance."""
import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu


def _sinos(torch, S, N, w, contrast, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    x = torch.rand((S, N, w), generator=g, device="cuda")
    return 0.2 + 0.8 * x if contrast == ca.ABS else x - 0.4


def _both(torch, w, N, centers, contrast, arc, store, seed=1):
    """Slices by the handle's own choice of launches and by the one-slice
    kernel, each also from the kept filtered sinograms."""
    S = len(centers)
    sino = _sinos(torch, S, N, w, contrast, seed)
    out = []
    for kind in (ca.TILE_AUTO, ca.TILE_64x64):
        rec = ca.CTrec(w, N, contrast, "HANN", anarc=arc, store=store)
        rec.set_tiles(kind, 0)
        a = torch.full((S, w, w), np.nan, device="cuda")
        b = torch.full((S, w, w), np.nan, device="cuda")
        rec.reconstruct_dev(sino, a, centers)
        rec.backproject_dev(b, centers)
        torch.cuda.synchronize()
        out += [a, b]
    return out


# 1400 px: 484 tiles a slice (242 mirrored), so four slices make a group from
# one float32 or two 16-bit groups on, and two from one float32 or three
# 16-bit pairs; centres repeat out of order and leave single slices.
@pytest.mark.parametrize("store,contrast,centers", [
    (ca.STORE_FP32, ca.ABS, [1.5, -2.25, 1.5, 1.5, -2.25, 1.5, 1.5, 0.0, 1.5, 1.5]),
    (ca.STORE_FP32, ca.PHS, [-7.0] * 4),
    (ca.STORE_FP32, ca.REF, [3.37] * 2),
    (ca.STORE_FP16, ca.ABS, [1.5, -2.25] * 5),
    (ca.STORE_FP16, ca.FLT, [3.0, 3.0, -4.5, 6.25, -4.5, 6.25]),
    (ca.STORE_BF16, ca.ABS, [0.75] * 9),
    (ca.STORE_BF16, ca.PHS, [-3.37] * 8),
    (ca.STORE_BF16, ca.PHS, [2.0, 2.0, -4.5, 6.25, -4.5, 6.25, 1.0]),
])
@pytest.mark.parametrize("N,arc", [(37, 180.0), (50, 360.0)])
def test_groups_equal_single_slices(torch_cuda, store, contrast, centers, N, arc):
    torch = torch_cuda
    auto, auto_kept, single, single_kept = _both(torch, 1400, N, centers, contrast, arc, store)
    assert torch.equal(single, single_kept)
    assert torch.equal(auto, single) and torch.equal(auto_kept, single)


def test_groups_in_graph_replays(torch_cuda):
    """The captured launches follow the data of each replay."""
    torch = torch_cuda
    w, N, centers = 1400, 40, [2.5] * 6
    rec = ca.CTrec(w, N, ca.ABS, "RAMP")
    one = rec.clone()
    one.set_tiles(ca.TILE_64x64, 0)
    sino = _sinos(torch, 6, N, w, ca.ABS, 0)
    out, want = (torch.empty((6, w, w), device="cuda") for _ in range(2))
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    rec.graph_capture(sino, out, centers, stream)
    for k in range(3):
        sino.copy_(_sinos(torch, 6, N, w, ca.ABS, k))
        one.reconstruct_dev(sino, want, centers)
        torch.cuda.synchronize()
        rec.graph_launch(stream)
        torch.cuda.synchronize()
        assert torch.equal(out, want)


# widths around the tiles' edges, the largest launch on 16x32 tiles (64 tiles
# of 64x64) and launches on 32x32 tiles; angle counts around a pass of 64
@pytest.mark.parametrize("w,S", [(2, 1), (15, 1), (16, 2), (17, 1), (33, 3), (64, 1), (65, 1), (512, 1), (513, 1),
                                 (700, 2), (1439, 1)])
@pytest.mark.parametrize("N,arc,c", [(1, 180.0, 0.0), (63, 180.0, 0.5), (64, 360.0, -0.25), (65, 150.0, 0.75)])
def test_small_tiles_equal_64x64(torch_cuda, w, S, N, arc, c):
    torch = torch_cuda
    auto, auto_kept, single, _ = _both(torch, w, N, [c + 0.01 * k for k in range(S)], ca.PHS, arc, ca.STORE_FP32)
    assert torch.equal(auto, single) and torch.equal(auto_kept, single)


@pytest.mark.parametrize("S", [7, 8, 9, 19])
@pytest.mark.parametrize("interp,store", [(ca.INTERP_LINEAR, ca.STORE_FP32), (ca.INTERP_CTAS, ca.STORE_FP16)])
@pytest.mark.parametrize("w", [200, 330])
def test_every_tile_of_many_slices_once(torch_cuda, S, interp, store, w):
    """Whole slices per XCD, and the rows of those left over: each slice as
    if it were alone."""
    torch = torch_cuda
    sino = _sinos(torch, S, 24, w, ca.ABS, S)
    rec = ca.CTrec(w, 24, ca.ABS, "HANN", store=store, interp=interp)
    rec.set_tiles(ca.TILE_64x64, 0)
    got = torch.full((S, w, w), np.nan, device="cuda")
    want = torch.empty((w, w), device="cuda")
    rec.reconstruct_dev(sino, got, [1.25] * S)
    for s in range(S):
        rec.reconstruct_dev(sino[s:s + 1], want.view(1, w, w), [1.25])
        torch.cuda.synchronize()
        assert torch.equal(got[s], want), s


# Mirrored launches of few tile pairs: widths at the edges of the quarter
# tiles, odd ones, a table with angles that have no partner, and both sides of
# the tile count where the whole ones take over (448 and 512 at 256 CUs).
@pytest.mark.parametrize("interp,store", [(ca.INTERP_LINEAR, ca.STORE_FP32), (ca.INTERP_LINEAR, ca.STORE_FP16),
                                          (ca.INTERP_LINEAR, ca.STORE_BF16), (ca.INTERP_CTAS, ca.STORE_FP16),
                                          (ca.INTERP_CTAS, ca.STORE_BF16)])
@pytest.mark.parametrize("S,w,N,c", [(1, 31, 40, 0.0), (1, 33, 37, 1.5), (2, 64, 50, -2.0), (1, 127, 91, 5.5),
                                     (3, 130, 36, -4.25), (1, 513, 180, 3.37), (3, 1024, 20, 1.0), (4, 1024, 20, 1.0)])
@pytest.mark.parametrize("contrast,arc", [(ca.ABS, 180.0), (ca.PHS, 360.0)])
def test_quarter_tiles_equal_whole_ones(torch_cuda, interp, store, S, w, N, c, contrast, arc):
    torch = torch_cuda
    sino = _sinos(torch, S, N, w, contrast, w)
    got = []
    for kind in (ca.TILE_AUTO, ca.TILE_64x64):
        rec = ca.CTrec(w, N, contrast, "HANN", anarc=arc, store=store, interp=interp)
        rec.set_tiles(kind, 0)
        out = torch.full((S, w, w), np.nan, device="cuda")
        rec.reconstruct_dev(sino, out, [c + 0.5 * s for s in range(S)])
        torch.cuda.synchronize()
        got.append(out)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("interp,store", [(ca.INTERP_LINEAR, ca.STORE_FP32), (ca.INTERP_CTAS, ca.STORE_BF16)])
@pytest.mark.parametrize("S", [5, 6, 7, 8])
def test_quarter_tiles_where_whole_ones_take_over(torch_cuda, interp, store, S):
    """720, 864, 1008 and 1152 tile pairs: the last counts on quarters are 720
    of 16-bit storage and 1008 LINEAR at 256 CUs."""
    test_quarter_tiles_equal_whole_ones(torch_cuda, interp, store, S, 1024, 20, 1.0, ca.ABS, 180.0)
