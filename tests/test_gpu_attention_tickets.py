"""plamo_kernel_attention_decode takes its positions as arguments, and its tickets under a number of
its own: calls in a row, of rows merged in the attention kernel (2 to 8 partitions) and by the merge
kernel, local and global, give the first call's bits every time; a count that another call left in a
ticket (calls that overlapped, against the header's rule) changes nothing, neither for calls that run
at once nor for replays of a recorded one."""
import ctypes

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


def _leave_counts():
    """What overlapping calls may leave in the static scratch's tickets: call 1's number and a count."""
    lib = native.load()
    scratch, fill = lib._ZN5plamo19static_attn_scratchEv, lib._ZN5plamo15launch_fill_u32EPjjmP12ihipStream_t
    scratch.restype = ctypes.c_void_p
    fill.argtypes = [ctypes.c_void_p, ctypes.c_uint32, ctypes.c_size_t, ctypes.c_void_p]
    base = scratch()
    for i in range(32):  # 256 bytes: both sets
        fill(base + 8 * i, (1 << 8) + 1 + i % 3, 1, None)
    torch.cuda.synchronize()


def _static_call(seed, rows, positions, full):
    """Inputs of one call of the static entry point -> a function that makes the call into `out`."""
    g = torch.Generator("cuda").manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)
    cap = 1024
    qkv, gain, keys, values = rnd(rows, 2304).float(), rnd(2, 128), rnd(rows, cap, 128), rnd(rows, cap, 128)
    rope = torch.zeros(2064, 64, dtype=torch.int32, device="cuda")
    rope += torch.tensor(np.uint32(0x3F80).view(np.int32), device="cuda")
    out, pos = torch.zeros(rows, 2048, dtype=torch.int16, device="cuda"), native.i32(positions)
    keep = (qkv, gain, keys, values, rope)

    def call():
        err = ctypes.create_string_buffer(256)
        assert native.load().plamo_kernel_attention_decode_static(
            qkv.data_ptr(), gain[0].data_ptr(), gain[1].data_ptr(), keys.data_ptr(), values.data_ptr(), cap, pos, rows,
            full, rope.data_ptr(), rope.data_ptr(), out.data_ptr(), torch.cuda.current_stream().cuda_stream, err,
            256) == 0, err.value
        return keep and out
    return call


@pytest.mark.parametrize("full", [0, 1])
def test_counts_left_in_tickets_change_nothing(full):
    call = _static_call(5, 4, [511, 64, 300, 130], full)
    want = call().clone()
    assert bool((want != 0).any(1).all())
    for _ in range(66):
        _leave_counts()
        out = call()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
        out.zero_()


@pytest.mark.parametrize("full", [0, 1])
@pytest.mark.parametrize("positions", [[513, 476, 130, 127], [511, 512], [1023, 64, 3]])
def test_rows_together_equal_rows_alone(full, positions):
    """Which kernel merges a row depends on the rows beside it; its bits do not."""
    print(f"  positions {positions} full {full}", flush=True)
    together = _static_call(8, len(positions), positions, full)().clone()
    for row, pos in enumerate(positions):
        alone = _static_call(8, len(positions), [pos if q == row else 0 for q in range(len(positions))], full)()
        torch.cuda.synchronize()
        assert torch.equal(alone[row], together[row]), row


def test_replays_between_calls():
    recorded, other = _static_call(6, 2, [450, 200], 0), _static_call(7, 3, [64, 500, 129], 1)
    want, want_other = recorded().clone(), other().clone()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        out = recorded()
    for i in range(6):
        out.zero_()
        if i % 2:
            _leave_counts()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), i
        got = other()
        torch.cuda.synchronize()
        assert torch.equal(got, want_other), i
        got.zero_()
