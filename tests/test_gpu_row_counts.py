"""Each active-row count of the four-row GEMVs has its own product loop: every row of a call with
two to four rows equals that row alone, bit for bit, for plain and .p12 weights.  The output rows
do not divide over the waves, so waves with several groups and without any take part."""
import numpy as np
import pytest
import torch

from oracle.bf16 import bits_np, roundbf_np
from plamo_hip import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(36, 1536), (5000, 1536), (36, 2048), (5000, 2048), (20, 6144), (5000, 6144)])
@pytest.mark.parametrize("packed", [False, True])
def test_rows_equal_single_rows(m, n, packed):
    print(f"  rows m={m} n={n} packed={packed}", flush=True)
    lib = native.load()
    rng = np.random.default_rng(m + n)
    w = bits_np(rng.standard_normal((m, n)).astype(np.float32) * 0.02)
    w[1, :128] = bits_np(np.full(128, 1e-30, np.float32))  # a raw .p12 block
    if packed:
        payload, table = native.pack_tensor(w)
        held = [torch.from_numpy(a).cuda() for a in (payload, table.view(np.int32))]
        addresses = [t.data_ptr() for t in held]
    else:
        held = [torch.from_numpy(w.view(np.int16)).cuda()]
        addresses = [held[0].data_ptr(), 0]
    x = torch.from_numpy(roundbf_np(rng.standard_normal((4, n)).astype(np.float32))).cuda()

    def linear(first, rows):
        y = torch.full((rows, m), -1.0, dtype=torch.float32, device="cuda")
        assert lib.plamo_kernel_linear(*addresses, x[first:].data_ptr(), y.data_ptr(), n, m, rows, 0, 0) == 0
        torch.cuda.synchronize()
        return y.cpu().numpy().view(np.uint32)

    single = np.concatenate([linear(q, 1) for q in range(4)])
    for rows in (2, 3, 4):
        assert np.array_equal(linear(0, rows), single[:rows]), rows
