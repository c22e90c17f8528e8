"""The score kernel at the edges of its tiles (32 x 64 derivatives), with few
taps and with as many as it takes, on slices smaller than its border: the
oracle's score to the 2e-4 of the parity tests (the filtered rows' rounding;
both sample the same bins)."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,w", [(4, 5), (9, 16), (33, 33), (90, 34), (200, 64), (60, 65), (40, 66), (67, 67), (12, 97),
                                 (6, 130), (140, 131)])
def test_scores_match_oracle(torch_cuda, N, w):
    rng = np.random.default_rng(N * w)
    P = rng.uniform(0.2, 1.0, (N, w)).astype(np.float32)
    step = 180.0 / (N - 1)
    rec = ca.CTrec(w, N, ca.ABS, "RAMP", anarc=step)
    rec.sino(P)
    axes = np.array([0.5 * (w - 1) + d for d in (-0.2 * w, -0.75, 0.0, 1.25, 0.15 * w)], np.float32)
    got = rec.axis_scores(axes)
    Pf = oracle.prepare(P, oracle.filter_window(1, 0.0, w, ca.ABS), ca.ABS)
    sigma = np.float32(oracle.angO(step, N) * np.float32(w) / np.pi)
    ref = np.array([oracle.ag_score(Pf, oracle.angles(N, step), float(sigma), float(a)) for a in axes])
    assert np.allclose(got, ref, rtol=2e-4), (got, ref)
