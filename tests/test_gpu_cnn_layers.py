"""The network's layer kernels at batch sizes where they end early: one
sample (a single split of the pixels, 22 steps in the last layer), counts
whose splits stop within the loads in flight, and odd ones. Bars as for the
batches of test_gpu_cnn: the bf16 roundings that flip between float32 and
float64 sums."""
import numpy as np
import pytest

import ctas_amd as ca
from oracle import cnn_oracle as co
from tests.conftest import rel_rms

pytestmark = pytest.mark.gpu


def _batch(torch, B, seed):
    x = torch.empty((B, 2, 180, 256), dtype=torch.int16, device="cuda")
    t = torch.empty((B, 2), dtype=torch.float32, device="cuda")
    ca.cnn_make_batch(seed, 0, x, t)
    return x, t


@pytest.mark.parametrize("B", [1, 2, 5])
def test_gradients_of_small_batches(torch_cuda, B):
    torch = torch_cuda
    x, t = _batch(torch, B, 41 + B)
    net = ca.AxisCNN(seed=3)
    loss = net.gradients_dev(x, t)
    xin = co.from_bf16_bits(x.cpu().numpy().view(np.uint16))
    lref, gref, _ = co.loss_and_grads(net.params().astype(np.float64), xin, t.cpu().numpy().astype(np.float64), True)
    assert loss == pytest.approx(lref, rel=1e-2)
    starts = np.cumsum([0] + co.SIZES)
    got = net.grads()
    for k, n in enumerate(co.SIZES):
        a, b = got[starts[k]:starts[k] + n], gref[starts[k]:starts[k] + n]
        assert rel_rms(a, b) < 3e-2, k


@pytest.mark.parametrize("B", [6, 23])
def test_gradients_across_the_widths_of_the_sums(torch_cuda, B):
    """Split counts on either side of where a sum takes more threads: 270 and
    67 in the first two layers, 1035 and 258, and bias sums of 17 or more."""
    test_gradients_of_small_batches(torch_cuda, B)


@pytest.mark.parametrize("N,w", [(1, 2), (7, 255), (180, 256), (181, 257), (360, 1024), (900, 4096), (365, 4097)])
def test_features_at_cell_edges(torch_cuda, N, w):
    """Cells of one sample, of uneven sizes and across the staged columns:
    within a bf16 rounding of the oracle's maps."""
    torch = torch_cuda
    rng = np.random.default_rng(N + w)
    P = rng.uniform(0.0, 1.0, (N, w)).astype(np.float32)
    d_x = torch.zeros((2, 180, 256), dtype=torch.int16, device="cuda")
    ca.cnn_features_dev(torch.from_numpy(P).cuda(), d_x)
    got = co.from_bf16_bits(d_x.cpu().numpy().view(np.uint16))
    ref = co.features(P)
    # one rounding of values up to 10 in magnitude, and one more flipped by the float32 sums
    assert np.abs(got - ref).max() <= 2 * 2.0 ** -8 * np.abs(ref).max()
