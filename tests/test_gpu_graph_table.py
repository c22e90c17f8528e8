"""A captured graph replays its own call whatever the handle does in between:
calls with other centres (which other slices may share a workgroup), more
slices (the handle's buffers are replaced), fewer, the filter alone or the
autotuner. Bit for bit the slices of a handle that does nothing else."""
import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu

W, N, S = 1400, 24, 6


def _sino(torch, S, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return 0.2 + 0.8 * torch.rand((S, N, W), generator=g, device="cuda")


def _between(torch, rec, what):
    if what == "centres":
        out = torch.empty((S, W, W), device="cuda")
        rec.reconstruct_dev(_sino(torch, S, 7), out, [0.5 * k - 1.0 for k in range(S)])
    elif what == "more":
        out = torch.empty((3 * S, W, W), device="cuda")
        rec.reconstruct_dev(_sino(torch, 3 * S, 8), out, [4.0] * (3 * S))
    elif what == "fewer":
        out = torch.empty((1, W, W), device="cuda")
        rec.reconstruct_dev(_sino(torch, 1, 9), out, [-2.0])
    elif what == "prepare":
        rec.prepare_dev(_sino(torch, 2, 10))
    elif what == "autotune":
        rec.autotune(2)
    torch.cuda.synchronize()


@pytest.mark.parametrize("store", [ca.STORE_FP32, ca.STORE_FP16])
@pytest.mark.parametrize("between", [["centres"], ["more"], ["fewer", "more"], ["prepare"], ["autotune"],
                                     ["more", "centres"]])
def test_replay_after_other_calls(torch_cuda, store, between):
    torch = torch_cuda
    centers = [2.5] * S
    rec = ca.CTrec(W, N, ca.ABS, "RAMP", store=store)
    one = ca.CTrec(W, N, ca.ABS, "RAMP", store=store)
    sino, out = _sino(torch, S, 0), torch.empty((S, W, W), device="cuda")
    want, again = torch.empty_like(out), torch.empty_like(out)
    rec.graph_capture(sino, out, centers)
    for k in range(3):
        _between(torch, rec, between[k % len(between)])
        sino.copy_(_sino(torch, S, 20 + k))
        if k == 1:
            sino[2] = -1.0  # this slice's status follows the replay
        one.reconstruct_dev(sino, want, centers)
        out.fill_(np.nan)
        torch.cuda.synchronize()
        rec.graph_launch()
        torch.cuda.synchronize()
        ok = [s for s in range(S) if not (k == 1 and s == 2)]
        assert torch.equal(out[ok], want[ok]), (k, between)
        assert (rec.status(S) == one.status(S)).all() and rec.status(S)[2] == (ca.CTAS_E_DATA if k == 1 else 0)
        if between != ["fewer", "more"] and between != ["prepare"]:  # as many filtered slices are kept
            rec.backproject_dev(again, centers)
            torch.cuda.synchronize()
            assert torch.equal(again[ok], want[ok]), (k, between)


@pytest.mark.parametrize("store", [ca.STORE_FP32, ca.STORE_FP16, ca.STORE_BF16])
@pytest.mark.parametrize("more", [False, True])
def test_replay_reads_the_handles_angles(torch_cuda, store, more):
    """A table of another number of mirrored pairs, set after the capture."""
    torch = torch_cuda
    centers = [2.5] * S
    theta = np.sort(np.random.default_rng(4).uniform(0.05, 1.5, N // 2)).astype(np.float32)
    half = np.stack([np.sin(theta), np.cos(theta)], 1).astype(np.float32)
    table = np.concatenate([half, half[::-1] * np.float32([1, -1])])
    rec = ca.CTrec(W, N, ca.ABS, "RAMP", store=store)
    one = rec.clone()
    one.set_angles(table)
    sino, out = _sino(torch, S, 1), torch.empty((S, W, W), device="cuda")
    want = torch.empty_like(out)
    rec.graph_capture(sino, out, centers)
    rec.set_angles(table)
    if more:
        _between(torch, rec, "more")
    one.reconstruct_dev(sino, want, centers)
    out.fill_(np.nan)
    torch.cuda.synchronize()
    for _ in range(2):
        rec.graph_launch()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
