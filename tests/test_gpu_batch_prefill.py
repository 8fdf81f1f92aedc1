"""Batch.prefill (Batch.swift:80-107) with prompts that share passes over the weights: every lane's
prediction, logits, hidden row, keys and values equal Runtime.prefill of its prompt bit for bit,
whatever the lengths share a pass (odd ones, partial query blocks, a single token beside them, more
rows than one pass holds), and so do the steps after."""
import numpy as np
import pytest

import plamo_hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("context,packed,lengths", [
    (96, False, [17, 2, 1, 33]),       # a single token beside three shared prompts
    (96, True, [90, 90, 90, 90]),      # a pass of four full prompts (lanes x chunk rows)
    (700, True, [601, 8, 129, 64]),    # whole and partial query blocks, two flash parts
    (2100, False, [700, 1500, 9, 2048]),  # more rows than one pass: 700 | 1500 + 9 | 2048
])
def test_shared_pass_equals_scalar(model_dir, context, packed, lengths):
    print(f"  batch prefill {lengths} context {context} packed {packed}", flush=True)
    d, sha = model_dir
    prompts = [np.random.default_rng(7 + i).integers(1024, 107520, n).tolist() for i, n in enumerate(lengths)]
    rt = plamo_hip.Runtime(d, context, packed=packed, source_sha256=sha)
    b = plamo_hip.Batch(rt)
    for _ in range(2):  # the second on the state the first left
        first = b.prefill(prompts)
        for lane, p in enumerate(prompts):
            rt.reset()
            assert rt.prefill(p) == first[lane], lane
            assert np.array_equal(b.logit_bits(lane), rt.logit_bits()), lane
            assert np.array_equal(b.hidden(lane).view(np.uint32), rt.hidden().view(np.uint32)), lane
            for layer in (0, 7, 11, 15):
                for got, want in zip(b.kv(lane, layer), rt.kv(layer)):
                    assert np.array_equal(got[:len(p)], want[:len(p)]), (lane, layer)
    second = b.step(first)
    for lane, p in enumerate(prompts):
        rt.reset()
        rt.prefill(p)
        assert rt.forward([first[lane]]) == second[lane], lane
        assert np.array_equal(b.logit_bits(lane), rt.logit_bits()), lane
    b.close()
    rt.close()
