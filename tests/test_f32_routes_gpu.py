"""A request's logits on the 32-bit path do not depend on which kernels its step's size takes: bit for bit the same alone, among 16
single tokens (the fused few-row products), among 17 (the kernels one by one) and beside a prompt's portion."""

from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


def _logits(model, others, portion, steps=5):
    """Of request 0, after a prompt of 37 tokens and ``steps`` single ones; beside it so many others, or a prompt in portions."""
    from dli_amd.engine.core import build_core
    from dli_amd.trace import TraceSession

    session = TraceSession(build_core(model, num_pages=160, page_size=16, max_seqs=20, enable_prefix_caching=False, watermark=0.0))
    vocab = model.spec.vocab_size
    token = lambda i, t: (31 * i + 17 * t + 5) % vocab
    prompts = {i: [token(i, t) for t in range(37 if i == 0 else 3 + 5 * i % 40)] for i in range(1 + others)}
    outs = [session.step([{"id": i, "tokens": p, "want": [len(p) - 1] if i == 0 else []} for i, p in prompts.items()]).clone()]
    for s in range(steps):
        step = [{"id": i, "tokens": [token(i, 50 + s)], "want": [0] if i == 0 else []} for i in prompts]
        if portion:
            step.append({"id": "portion", "tokens": [token(99, 20 * s + t) for t in range(20)], "want": []})
        outs.append(session.step(step).clone())
    return outs


# heads of 16, of 32 with the scaled rotation, of 48 with biases everywhere, of 128
@pytest.mark.parametrize("config", ["A", "B", "C", "H"])
def test_a_request_is_the_same_by_every_route(config):
    import torch

    from dli_amd.weights import load_model
    from tiny_configs import model_folder

    model = load_model(model_folder(config), dtype="float32")
    fused, inner = [], model._forward_stream
    model._forward_stream = lambda *a: fused.append(1) or inner(*a)
    want = _logits(model, 0, False)
    assert len(fused) == 5
    for others, portion, runs in ((15, False, 5), (16, False, 0), (0, True, 0), (3, True, 0)):
        fused.clear()
        got = _logits(model, others, portion)
        assert len(fused) == runs
        assert all(torch.equal(g, w) for g, w in zip(got, want)), (others, portion)
