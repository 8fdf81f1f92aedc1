"""The prefill GEMM's tiles (`matrix`, Kernels.metal:149-200; `swiglu`, Kernels.metal:202-210): one
size per tile of the dispatch, with ragged token and row counts, depths of 128 mod 256, rows that
are no multiple of four and outputs that are not aligned for four, each bit for bit against the
order-exact restatement (oracle/exact_prefill.py).  Token rows repeat 29 distinct ones, so the
restatement runs 29 rows whatever the token count."""
import numpy as np
import pytest
import torch

from oracle import exact, exact_prefill as xp
from oracle.bf16 import bits_np, roundbf_np
from plamo_hip import native

pytestmark = pytest.mark.gpu


def _case(m, n, tokens):
    rng = np.random.default_rng(m + n + tokens)
    w = bits_np(rng.standard_normal((m, n)).astype(np.float32) * 0.02)
    rows = bits_np(rng.standard_normal((min(29, tokens), n)).astype(np.float32))
    of = rng.integers(0, len(rows), tokens)
    return w, rows, of


def _run(w, x, mode, cols, element, skip):
    """`skip`: elements before y in its (over-long) buffer, whose ends must stay untouched."""
    lib = native.load()
    tokens, n = x.shape
    wd, xd = (torch.from_numpy(a.view(np.int16)).cuda() for a in (w, np.ascontiguousarray(x)))
    y = torch.full((tokens * cols + 16,), 77, dtype=torch.float32 if element == 4 else torch.int16, device="cuda")
    assert lib.plamo_kernel_gemm(wd.data_ptr(), 0, xd.data_ptr(), y.data_ptr() + skip * element, n, w.shape[0], tokens,
                                 mode, 0) == 0
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    end = skip + tokens * cols
    assert (y[:skip] == 77).all() and (y[end:] == 77).all()
    return y[skip:end].reshape(tokens, cols)


@pytest.mark.parametrize("m,n,tokens,skip", [
    (100, 256, 5, 0),      # 16 x 16, 256-deep stages, one ragged block
    (98, 384, 33, 0),      # 16 x 16, 128-deep stages, rows no multiple of four
    (1536, 6144, 16, 1),   # 16 x 16 at the down projection, y one element past alignment
    (2304, 256, 31, 0),    # 32 x 16
    (2304, 384, 40, 2),    # 16 x 32
    (1536, 2048, 129, 0),  # 32 x 32
    (1540, 128, 257, 3),   # 64 x 32
    (1530, 128, 449, 0),   # 64 x 48, rows no multiple of four
    (2304, 128, 401, 0),   # 64 x 64
    (640, 1536, 1700, 0),  # 96 x 64, the QSA indexer's rows
    (1536, 128, 700, 0),   # 96 x 64
    (2304, 128, 700, 0),   # 128 x 64
    (1536, 128, 1024, 0),  # 64 x 96
    (1536, 128, 1431, 1),  # 96 x 96
    (1536, 128, 2047, 0),  # 128 x 96
    (2304, 128, 1501, 0),  # 128 x 128
    (2304, 128, 2045, 0),  # 128 x 192
    (12304, 128, 700, 0),  # several rounds, rows past the last whole tile
])
def test_gemm_tiles_bit_exact(m, n, tokens, skip):
    print(f"  gemm {m}x{n} tokens={tokens}", flush=True)
    w, rows, of = _case(m, n, tokens)
    want = xp.mfma_gemm(w, rows)
    assert np.array_equal(_run(w, rows[of], 2, m, 4, skip).view(np.uint32), want.view(np.uint32)[of])
    assert np.array_equal(_run(w, rows[of], 1, m, 2, skip).view(np.uint16), bits_np(want)[of])
    assert np.array_equal(_run(w, rows[of], 0, m, 4, skip), roundbf_np(want)[of])


@pytest.mark.parametrize("tokens,skip", [(3, 0), (17, 0), (33, 1), (65, 0), (129, 0), (257, 0), (385, 0), (700, 2),
                                         (1281, 0), (1537, 0)])
def test_swiglu_tiles_bit_exact(tokens, skip):
    """16 x 64, 32 x 64, 64 x 64, 64 x 96, 128 x 128, 192 x 128, 128 x 192, 256 x 192, 192 x 128 in
    three rounds, 256 x 128."""
    print(f"  swiglu tokens={tokens}", flush=True)
    w, rows, of = _case(12288, 1536, tokens)
    want = xp.mfma_gemm(w, rows)
    g, u = roundbf_np(want[:, :6144]), roundbf_np(want[:, 6144:])
    act = bits_np(roundbf_np(g / (np.float32(1) + exact.exp_det(-g))) * u)
    assert np.array_equal(_run(w, rows[of], 3, 6144, 2, skip).view(np.uint16), act[of])
