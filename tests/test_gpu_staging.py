"""Host-array calls whose copies go through pinned blocks: sizes around a
block (512 KiB), around the eight of a set and past the largest staged copy
(8 MiB) give what the device-array call gives, bit for bit; so do more threads
at once than there are sets, and a rejected sinogram leaves the caller's arrays
alone."""
import threading

import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu


def _sino(S, N, w, seed=0):
    return np.random.default_rng(seed).uniform(0.2, 1.0, (S, N, w)).astype(np.float32)


@pytest.mark.parametrize("S,N,w", [(1, 1, 2), (1, 3, 33), (1, 255, 512), (1, 256, 512), (1, 257, 512), (9, 128, 1023),
                                   (1, 1024, 2048), (1, 1025, 2048)])
@pytest.mark.parametrize("store", [ca.STORE_FP32, ca.STORE_FP16])
def test_host_arrays_equal_device_arrays(torch_cuda, S, N, w, store):
    torch = torch_cuda
    P, c = _sino(S, N, w, N), [0.25] * S
    rec = ca.CTrec(w, N, ca.ABS, "HANN", store=store)
    filt, out = rec.reconstruct(P, c)
    assert np.array_equal(rec.prepare(P), filt)
    assert np.array_equal(rec.repeat([0.25])[0], out[0])
    d_out = torch.empty((S, w, w), device="cuda")
    ca.CTrec(w, N, ca.ABS, "HANN", store=store).reconstruct_dev(torch.from_numpy(P).cuda(), d_out, c)
    assert np.array_equal(d_out.cpu().numpy(), out)


def test_more_threads_than_sets(torch_cuda):
    N, w, T = 300, 700, 7
    P = [_sino(1, N, w, k) for k in range(T)]
    want = [ca.CTrec(w, N, ca.ABS, "RAMP").reconstruct(p, 1.0) for p in P]
    got = [None] * T

    def work(k):
        rec = ca.CTrec(w, N, ca.ABS, "RAMP")
        for _ in range(5):
            got[k] = rec.reconstruct(P[k], 1.0)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(T)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for (a, b), (c, d) in zip(got, want):
        assert np.array_equal(a, c) and np.array_equal(b, d)


def test_rejected_sinogram_is_left_alone(torch_cuda):
    N, w = 64, 600
    rec = ca.CTrec(w, N, ca.ABS, "RAMP")
    s = np.full((1, N, w), -1.0, np.float32)  # deAbs: the maximum is not positive
    out = np.full((1, w, w), 7.0, np.float32)
    c = np.zeros(1, np.float32)
    rc = ca.lib().ctas_fbp_reconstruct(rec._h, ca._f32p(s), ca._f32p(out), ca._f32p(c), 1)
    assert rc == ca.CTAS_E_DATA
    assert (s == -1.0).all() and (out == 7.0).all()
