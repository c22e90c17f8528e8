"""NaN and infinite samples in the registration and in the axis scores have the
oracle's outcome, and a pass length of the caller's changes no bit of the
slices."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("where", [(0, 0), (3, 40), (15, 299)])
def test_registration(bad, where):
    rng = np.random.default_rng(1)
    p = rng.uniform(0.5, 1.0, (16, 300)).astype(np.float32)
    q = np.ascontiguousarray(p[:, ::-1])
    p[where] = bad
    with pytest.raises(ValueError):
        oracle.raxis_pair(p, q, 0.25)
    with pytest.raises(ca.CtasError):
        ca.raxis_pair(p, q, 0.25)


@pytest.mark.parametrize("N,w", [(9, 16), (90, 70)])
def test_scores(N, w):
    """A filtered row of NaN: the oracle's score, NaN or (where no pixel counts)
    zero."""
    rng = np.random.default_rng(N)
    P = rng.uniform(0.2, 1.0, (N, w)).astype(np.float32)
    P[N // 2, w // 2] = np.nan
    step = 180.0 / (N - 1)
    rec = ca.CTrec(w, N, ca.ABS, "RAMP", anarc=step)
    rec.sino(P.copy())
    axes = np.array([0.5 * (w - 1), 0.5 * (w - 1) + 1.25], np.float32)
    got = rec.axis_scores(axes)
    Pf = oracle.prepare(P, oracle.filter_window(1, 0.0, w, ca.ABS), ca.ABS)
    sigma = np.float32(oracle.angO(step, N) * np.float32(w) / np.pi)
    ref = np.array([oracle.ag_score(Pf, oracle.angles(N, step), float(sigma), float(a)) for a in axes])
    assert np.allclose(got, ref, rtol=2e-4, atol=0.0, equal_nan=True), (got, ref)


@pytest.mark.parametrize("store", [ca.STORE_FP32, ca.STORE_FP16])
@pytest.mark.parametrize("interp", [ca.INTERP_CTAS, ca.INTERP_LINEAR])
@pytest.mark.parametrize("S,w", [(1, 130), (6, 700)])
@pytest.mark.parametrize("ac", [16, 32])
def test_pass_length(torch_cuda, store, interp, S, w, ac):
    torch = torch_cuda
    sino = 0.2 + 0.8 * torch.rand((S, 50, w), generator=torch.Generator("cuda").manual_seed(w), device="cuda")
    out = [torch.empty((S, w, w), device="cuda") for _ in range(2)]
    for o, length in zip(out, (0, ac)):
        rec = ca.CTrec(w, 50, ca.ABS, "HANN", store=store, interp=interp)
        rec.set_tiles(ca.TILE_AUTO, length)
        assert rec.tiles()[1] == (length or rec.tiles()[1])
        rec.reconstruct_dev(sino, o, [1.5] * S)
        torch.cuda.synchronize()
    assert torch.equal(out[0], out[1])
