"""plamo_kernel_attention_decode takes its positions as arguments and its tickets from one of 64
sets in turn: more calls than sets, of rows merged in the attention kernel (2 to 8 partitions) and by
the merge kernel, local and global, give the first call's bits every time."""
import numpy as np
import pytest
import torch

from plamo_hip import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("full,positions", [(0, [343, 130]), (0, [2500, 700, 64]), (1, [511]), (1, [900, 63, 2000, 300])])
def test_calls_in_turn_repeat(full, positions):
    print(f"  positions {positions} full {full}", flush=True)
    g = torch.Generator("cuda").manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    rows, cap = len(positions), 4096
    qkv, gain = rnd(rows, 2304).float(), rnd(2, 128)
    keys, values = rnd(rows, cap, 128), rnd(rows, cap, 128)
    rope = torch.zeros(cap, 64, dtype=torch.int32, device="cuda")
    rope += torch.tensor(np.uint32(0x3F80).view(np.int32), device="cuda")  # cos 1, sin 0
    pos, first = native.i32(positions), None
    for _ in range(70):
        out = torch.zeros(rows, 2048, dtype=torch.int16, device="cuda")
        assert native.load().plamo_kernel_attention_decode(
            qkv.data_ptr(), gain[0].data_ptr(), gain[1].data_ptr(), keys.data_ptr(), values.data_ptr(), cap, pos, rows,
            full, rope.data_ptr(), rope.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream) == 0
        first = out if first is None else first
        assert torch.equal(out, first) and bool((out != 0).any())
