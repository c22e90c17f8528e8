"""raxis with a sweep of one or two trials (max_dev w below 4 and 8 px), whose
walk starts beside the sweep: the oracle's search and the device's agree to its
last bisection step, as in test_random_raxis."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle
from tests.test_gpu_random import _dots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,N", [(96, 200), (151, 190)])
@pytest.mark.parametrize("c0", [0.0, 1.5, -6.0, 11.0])
@pytest.mark.parametrize("trials", [1, 2])
def test_few_trials_match_oracle(w, N, c0, trials):
    rng = np.random.default_rng(w + N + int(4 * c0))
    P = np.exp(-oracle.phantom_sino(N, w, c0, _dots(w, 8, rng), 0.0, 0)).astype(np.float32)
    step, max_dev = 180.0 / (N - 1), (2.0 if trials == 1 else 6.0) / w
    try:
        ref = oracle.raxis(P, step, max_dev, 1)
    except ValueError:
        with pytest.raises(ca.CtasError):
            ca.raxis(P, step, max_dev, 1)
        return
    assert abs(ca.raxis(P, step, max_dev, 1) - ref) <= 0.25
