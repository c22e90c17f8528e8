"""A call that needs more device memory than there is fails with
CTAS_E_NOMEM and leaves the handle usable: the filtered slices that went with
its buffer are gone for repeat, and the next call works."""
import ctypes as C

import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("store", [ca.STORE_FP32, ca.STORE_FP16])
def test_refused_batch(torch_cuda, store):
    torch = torch_cuda
    S, N, w = 2, 1000, 1000
    sino = 0.2 + 0.8 * torch.rand((S, N, w), generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    out, again = (torch.empty((S, w, w), device="cuda") for _ in range(2))
    rec = ca.CTrec(w, N, ca.ABS, "HANN", store=store)
    rec.reconstruct_dev(sino, out, [1.5] * S)
    torch.cuda.synchronize()
    # 4 TB of filtered slices: refused before any pointer is used
    rc = ca.lib().ctas_fbp_prepare_dev(rec._h, C.c_void_p(sino.data_ptr()), 2_000_000 if store else 1_000_000, None)
    assert rc == ca.CTAS_E_NOMEM
    with pytest.raises(ca.CtasError) as e:
        rec.repeat_dev(again[:1], [1.5])
    assert e.value.code == ca.CTAS_E_STATE
    rec.reconstruct_dev(sino, again, [1.5] * S)
    torch.cuda.synchronize()
    assert torch.equal(out, again) and (rec.status(S) == 0).all()
