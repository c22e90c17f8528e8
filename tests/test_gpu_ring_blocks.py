"""The ring filter at the edges of its blocks (64 rows a step, 64 columns a
workgroup, chunks of rows in the update): bit for bit the oracle's sums."""
import numpy as np
import pytest

import ctas_amd as ca
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 3, 63, 64, 65, 127, 129, 400])
@pytest.mark.parametrize("w,box", [(2, 1), (63, 62), (64, 1), (65, 15), (257, 40), (300, 299)])
def test_ring_blocks_match_oracle(torch_cuda, N, w, box):
    torch = torch_cuda
    rng = np.random.default_rng(N * 1000 + w)
    P = rng.uniform(0.1, 1.0, (2, N, w)).astype(np.float32)
    d = torch.from_numpy(P).cuda()
    ca.ring_filter_dev(d, box)
    got = d.cpu().numpy()
    for k in range(2):
        assert np.array_equal(got[k], oracle.ring_filter(P[k], box))
