"""raxis_pair against the oracle at the row and column counts where its
kernels' blocks end: rows below, at and past a block of rows and the 1024-row
stage of the edge sums, columns past a wave, trials past a chunk of eight,
and shifts outside the sweep, which the walk finds. Both search the same
trials from the same seed, whose rounding (a quotient of sums near 1e6 in
float, 1e-7 of the width) bounds the difference."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle

pytestmark = pytest.mark.gpu


def _pair(rows, w, shift, seed):
    rng = np.random.default_rng(seed)
    x, y = np.linspace(-1, 1, w)[None, :], np.linspace(-1, 1, rows)[:, None] if rows > 1 else np.zeros((1, 1))
    p = np.zeros((rows, w))
    for _ in range(4):
        cx, cy, r, m = rng.uniform(-0.3, 0.3), rng.uniform(-0.5, 0.5), rng.uniform(0.2, 0.5), rng.uniform(0.2, 0.8)
        p += m * np.sqrt(np.maximum(0.0, 1 - ((x - cx) / r) ** 2 - (0.5 * (y - cy)) ** 2))
    q = np.roll(p[:, ::-1], shift, axis=1)
    noise = 2e-3 * rng.standard_normal((2, rows, w))
    return (np.exp(-p) + noise[0]).astype(np.float32), (np.exp(-q) + noise[1]).astype(np.float32)


@pytest.mark.parametrize("rows", [1, 3, 255, 1023, 1030])
@pytest.mark.parametrize("w,shift,max_dev", [(256, 5, 0.25), (321, -31, 0.25), (1000, 40, 0.25), (700, 60, 0.05),
                                             (700, -90, 0.05)])
def test_registration_matches_oracle(rows, w, shift, max_dev):
    p0, p180 = _pair(rows, w, shift, 1000 * rows + w + shift)
    try:
        want = oracle.raxis_pair(p0, p180, max_dev)
    except ValueError:
        with pytest.raises(ca.CtasError):
            ca.raxis_pair(p0, p180, max_dev)
        return
    assert abs(ca.raxis_pair(p0, p180, max_dev) - want) <= 1e-7 * w * 10
