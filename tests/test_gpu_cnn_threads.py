"""Parameters read (or saved) by one thread while another predicts with the
same network: reading leaves the network's own buffers alone."""
import threading

import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu


def test_parameters_read_beside_predictions(torch_cuda, tmp_path):
    torch = torch_cuda
    net = ca.AxisCNN(seed=5)
    params = net.params()
    sino = 0.2 + 0.8 * torch.rand((360, 512), generator=torch.Generator("cuda").manual_seed(2), device="cuda")
    torch.cuda.synchronize()
    want = net.predict_dev(sino)
    got, failed, stop = [], [], threading.Event()

    def read():
        while not stop.is_set():
            net.save(str(tmp_path / "net.bin"))
            got.append(np.array_equal(net.params(), params))

    t = threading.Thread(target=read)
    t.start()
    try:
        for _ in range(200):
            if net.predict_dev(sino) != want:
                failed.append(1)
    finally:
        stop.set()
        t.join()
    assert not failed and got and all(got)
