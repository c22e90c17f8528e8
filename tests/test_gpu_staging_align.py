"""Host-array calls whose sample count is not a multiple of four: the filtered
rows of 16-bit storage come back from a float32 copy that starts on a 16-byte
boundary all the same (an odd start is refused by the copy). Bit for bit the
rows of one slice at a time, whose copy starts elsewhere."""
import numpy as np
import pytest

import ctas_amd as ca

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S,N,w", [(1, 1, 2), (1, 3, 33), (3, 5, 127), (2, 7, 513), (5, 181, 1437)])
@pytest.mark.parametrize("store", [ca.STORE_FP16, ca.STORE_BF16])
def test_filtered_rows_of_odd_counts(torch_cuda, S, N, w, store):
    P = np.random.default_rng(N + w).uniform(0.2, 1.0, (S, N, w)).astype(np.float32)
    filt, out = ca.CTrec(w, N, ca.ABS, "HANN", store=store).reconstruct(P, [0.25] * S)
    for s in range(S):
        one_filt, one_out = ca.CTrec(w, N, ca.ABS, "HANN", store=store).reconstruct(P[s:s + 1], [0.25])
        assert np.array_equal(filt[s], one_filt[0]) and np.array_equal(out[s], one_out[0])
