"""Global prefill attention at the edges between one key tile, two (calls of up to two have a kernel of
their own) and three, and at the smallest ring that the direct kernel takes and the largest that it
leaves to the staged one; and at the edge between blocks of one part and of two, from where a call uses
the shared workspace: bit for bit the CPU restatement."""
import numpy as np
import pytest
import torch

from oracle import exact_prefill as xp
from oracle.bf16 import bits_np
from plamo_hip import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p0,tokens,cap", [
    (0, 1, 64), (0, 63, 64), (3, 61, 64), (63, 1, 64),     # one tile, a partial one and a full one
    (3, 62, 65), (64, 1, 65), (60, 9, 80),                 # blocks of one tile and of two in one call
    (0, 128, 128), (120, 8, 128),                          # two full tiles: the last call of the short kernel
    (127, 2, 200), (0, 129, 129),                          # three: the first of the other
    (10, 53, 63),                                          # a ring below one tile
    (696, 8, 704), (697, 8, 705), (696, 9, 705),           # one part, two, and both in one call
])
def test_short_global_calls_bit_exact(p0, tokens, cap):
    print(f"  flash p0={p0} tokens={tokens} cap={cap}", flush=True)
    rng = np.random.default_rng(31 * p0 + tokens)
    q = bits_np(rng.standard_normal((tokens, 16, 128)).astype(np.float32))
    keys = bits_np(rng.standard_normal((cap, 128)).astype(np.float32))
    values = bits_np(rng.standard_normal((cap, 128)).astype(np.float32))
    out = torch.full((tokens, 2048), -1, dtype=torch.int16, device="cuda")
    qd, kd, vd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (q, keys, values))
    assert native.load().plamo_kernel_attention_prefill(qd.data_ptr(), kd.data_ptr(), vd.data_ptr(), cap, p0, tokens, 1,
                                                        0, out.data_ptr(), 0) == 0
    torch.cuda.synchronize()
    table = np.zeros((2064, 64), np.uint16)  # global keys are stored rotated: not read
    want = xp.flash(q, keys, values, table, table, cap, p0, True)
    assert np.array_equal(out.cpu().numpy().view(np.uint16), want)
