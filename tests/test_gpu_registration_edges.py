"""raxis_pair with a sweep of one or two trials (max_dev w below 8 and 16 px):
the walk's bracket then starts beside the sweep. Against the oracle, to the
rounding of the seed as in test_gpu_registration."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle
from tests.test_gpu_registration import _pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 64])
@pytest.mark.parametrize("w,shift", [(64, 1), (256, 5), (321, -31), (700, 60), (700, -9), (1000, 0)])
@pytest.mark.parametrize("trials", [1, 2])
def test_few_trials_match_oracle(rows, w, shift, trials):
    max_dev = (2.0 if trials == 1 else 10.0) / w
    p0, p180 = _pair(rows, w, shift, rows + w + shift)
    try:
        want = oracle.raxis_pair(p0, p180, max_dev)
    except ValueError:
        with pytest.raises(ca.CtasError):
            ca.raxis_pair(p0, p180, max_dev)
        return
    assert abs(ca.raxis_pair(p0, p180, max_dev) - want) <= 1e-7 * w * 10
