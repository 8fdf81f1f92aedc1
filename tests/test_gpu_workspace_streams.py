"""Kernel-level attention whose shared workspace has just grown, called on a stream of its own while
the default stream has work queued: the tickets are cleared on the calling stream, so rows and query
blocks of several parts are right without any wait between the streams."""
import numpy as np
import pytest
import torch

from plamo_hip import native

pytestmark = pytest.mark.gpu


def _inputs(*shapes):
    g = torch.Generator("cuda").manual_seed(9)
    return [torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16) for s in shapes]


def _rope(rows):
    one = torch.tensor(np.uint32(0x3F80).view(np.int32), device="cuda")  # cos 1, sin 0
    return torch.zeros(rows, 64, dtype=torch.int32, device="cuda") + one


def _on_own_stream(call):
    """`call(out, stream)` on a stream of its own behind a busy default stream -> (out, then again alone)."""
    busy = torch.randn(4096, 4096, device="cuda")
    outs = [torch.zeros_like(call.out) for _ in range(2)]
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    for _ in range(20):
        busy = torch.tanh(busy @ busy)
    call(outs[0], stream.cuda_stream)
    stream.synchronize()
    torch.cuda.synchronize()
    call(outs[1], 0)
    torch.cuda.synchronize()
    return outs


@pytest.mark.parametrize("full", [0, 1])
def test_flash_prefill(full):
    tokens, p0 = 2330 + 200 * full, 900  # more tokens than any other test's call
    cap = p0 + tokens
    q, k, v = _inputs((tokens, 16, 128), (cap, 128), (cap, 128))
    rope = _rope(2064)

    def call(out, stream):
        print(f"  flash tokens {tokens} p0 {p0} full {full} stream {stream != 0}", flush=True)
        assert native.load().plamo_kernel_attention_prefill(q.data_ptr(), k.data_ptr(), v.data_ptr(), cap, p0, tokens,
                                                            full, rope.data_ptr(), out.data_ptr(), stream) == 0
    call.out = torch.empty(tokens, 2048, dtype=torch.int16, device="cuda")
    first, alone = _on_own_stream(call)
    assert torch.equal(first, alone) and bool((first != 0).any(1).all())


def test_attention_decode():
    rows, cap, positions = 4, 32768, native.i32([511, 130, 64, 32767])
    qkv, gain, k, v = _inputs((rows, 2304), (2, 128), (rows, cap, 128), (rows, cap, 128))
    qkv, rope = qkv.float(), _rope(cap)

    def call(out, stream):
        print(f"  decode stream {stream != 0}", flush=True)
        assert native.load().plamo_kernel_attention_decode(
            qkv.data_ptr(), gain[0].data_ptr(), gain[1].data_ptr(), k.data_ptr(), v.data_ptr(), cap, positions, rows, 1,
            rope.data_ptr(), rope.data_ptr(), out.data_ptr(), stream) == 0
    call.out = torch.empty(rows, 2048, dtype=torch.int16, device="cuda")
    first, alone = _on_own_stream(call)
    assert torch.equal(first, alone) and bool((first != 0).any(1).all())
