"""A decode step of one row in one launch: against the plain implementation, and against the same steps block by block."""

import tempfile
from pathlib import Path

import pytest
import torch

import plain_llama as P

pytestmark = pytest.mark.gpu


def _config(layers, hidden, heads, kv, dim, inner):
    return {"architectures": ["LlamaForCausalLM"], "model_type": "llama", "vocab_size": 256, "hidden_size": hidden, "intermediate_size": inner,
            "num_hidden_layers": layers, "num_attention_heads": heads, "num_key_value_heads": kv, "head_dim": dim, "rms_norm_eps": 1e-5,
            "max_position_embeddings": 16384, "rope_theta": 10000.0, "tie_word_embeddings": True, "hidden_act": "silu"}


# the 135M and 360M sizes; the most it takes; one head, widths that are no whole blocks of 128 (a part of one, and two and a part) and that
# divide into few rows a workgroup; heads of 128 of another width than the stream; sixteen heads on one
SIZES = [(3, 576, 9, 3, 64, 1536), (2, 960, 15, 5, 64, 2560), (2, 1024, 16, 8, 64, 3072), (1, 96, 1, 1, 64, 32), (2, 288, 2, 2, 64, 160),
         (2, 384, 6, 2, 128, 640), (1, 256, 16, 1, 64, 512)]
# keys in the pages before the first decode step: none, around a pair of tiles, around a run of a workgroup's waves (eight pairs with the
# new token's), around the most runs, where waves get a second pair
CONTEXTS = [0, 1, 31, 223, 255, 479]


@pytest.mark.parametrize("graphs", [False, True])
@pytest.mark.parametrize("sizes", SIZES)
def test_steps_of_one_row(sizes, graphs):
    _compare(sizes, CONTEXTS, 16, 4, graphs)


@pytest.mark.parametrize("sizes,page,context", [(SIZES[3], 48, 700), (SIZES[3], 16, 4063), (SIZES[5], 64, 4100), (SIZES[3], 256, 8150)])
def test_long_contexts_and_pages(sizes, page, context):
    _compare(sizes, [context], page, 3, True)


def _compare(sizes, contexts, page, steps, graphs):
    """The error of each route is the roundings of its activations to bfloat16, about as many on either, so the one may be no further from
    exact logits than the other but for chance (a quarter, over all steps), nor a row by more than three times the other's mean."""
    from dli_amd.engine.core import build_core
    from dli_amd.kernels import ops
    from dli_amd.trace import TraceSession
    from dli_amd.weights import load_model, write_random_model

    assert ops.decode_flow_bytes(*sizes) > 0
    with tempfile.TemporaryDirectory() as tmp:
        folder = write_random_model(Path(tmp) / "m", _config(*sizes), seed=sum(sizes), std=0.5 / sizes[1] ** 0.5, norm_jitter=0.1)
        cfg, weights = P.load_folder(folder)
        model = load_model(folder, dtype="bfloat16")
    gen = torch.Generator().manual_seed(len(contexts) + sizes[1])
    longest = max(contexts) + steps
    tokens = torch.randint(0, 256, (longest,), generator=gen).tolist()
    exact = P.forward_logits(weights, cfg, tokens)
    errors = {}
    for flow in (True, False):
        model.native_steps = flow
        core = build_core(model, num_pages=len(contexts) * (-(-longest // page) + 1), page_size=page, max_seqs=8, enable_prefix_caching=False,
                          watermark=0.0)
        if graphs:
            core.step.enable_decode_graphs(1, longest)
        session, off = TraceSession(core), []
        for i, context in enumerate(contexts):
            if context:
                session.step([{"id": f"r{i}", "tokens": tokens[:context]}])
            for at in range(context, context + steps):
                got = session.step([{"id": f"r{i}", "tokens": [tokens[at]], "want": [0]}]).double().cpu()
                off.append(((got[0] - exact[at]).norm() / exact[at].norm()).item())
        errors[flow] = torch.tensor(off)
        assert bool(core.step.caches.flow) == flow
    assert errors[True].mean() <= 1.25 * errors[False].mean() + 1e-4, errors
    assert errors[True].max() <= 3 * errors[False].mean() + 1e-4, errors


def test_what_it_does_not_take():
    from dli_amd.kernels import ops

    refused = [(2, 1032, 16, 8, 64, 3072), (2, 1024, 17, 17, 64, 3072), (2, 1024, 16, 8, 64, 3080), (2, 576, 9, 3, 48, 1536), (0, 576, 9, 3, 64, 1536),
               (2, 576, 9, 2, 64, 1536), (1, 256, 17, 1, 64, 512), (1, 60, 1, 1, 64, 64), (1, 64, 1, 1, 64, 20)]
    assert not any(ops.decode_flow_bytes(*s) for s in refused)


class _Launches:
    """Launches of the kernel by itself, over weights and pages of its own: one request of 20 keys, in the order of a page table."""

    def __init__(self, sizes, seed):
        from dli_amd.kernels import ops

        layers, hidden, heads, kv, dim, inner = self.sizes = sizes
        gen = torch.Generator(device="cuda").manual_seed(seed)
        draw = lambda *s: torch.randn(*s, device="cuda", generator=gen)
        matrix = lambda *s: draw(*s).mul_(s[1] ** -0.5).bfloat16()
        self.held = [[1 + 0.1 * draw(hidden), 1 + 0.1 * draw(hidden), matrix((heads + 2 * kv) * dim, hidden), matrix(hidden, heads * dim),
                      matrix(2 * inner, hidden), matrix(hidden, inner), draw(3, kv, 16, dim).bfloat16(), draw(3, kv, dim, 16).bfloat16()]
                     for _ in range(layers)]
        self.table = torch.tensor([[t.data_ptr() for t in row] for row in self.held], dtype=torch.int64).cuda()
        self.xs = draw(6, hidden).bfloat16()
        turn = 19 * 10000.0 ** (-torch.arange(dim // 2, device="cuda") / (dim // 2))
        self.angles = torch.stack([turn.cos(), turn.sin()])[None].float().contiguous()
        on = lambda *v: torch.tensor(v, dtype=torch.int32, device="cuda")
        self.slot, self.keys, self.pages = on(2 * 16 + 3), on(20), on(1, 2)[None].contiguous()
        self.words_of = lambda: torch.zeros(ops.decode_flow_bytes(*sizes) // 4, dtype=torch.int32, device="cuda")
        self.ssq = torch.empty(ops.decode_flow_parts(*sizes), 1, device="cuda")

    def run(self, words, launch, x, **more):
        """The stream behind a launch that is the ``launch``-th of these words (from 0 on), on a row."""
        from dli_amd.kernels import ops

        dim, stream = self.sizes[4], x[None].clone()
        ops.decode_flow(self.table, words, torch.tensor([launch << 32], dtype=torch.int64, device="cuda"), stream, self.ssq, self.angles,
                        self.slot, self.keys, self.pages, self.sizes, 16, 1e-5, dim ** -0.5, **more)
        return stream[0]


def test_numbers_of_launches_go_round():
    """A word's tag is 16 bits of the launch's number: on both sides of 65,536 launches the results are those of the first ones."""
    at = _Launches(SIZES[1], 5)
    early, late = at.words_of(), at.words_of()
    for i, x in enumerate(at.xs):
        first, then = at.run(early, i, x), at.run(late, 65533 + i, x)
        assert first.isfinite().all() and torch.equal(first, then)


@pytest.mark.parametrize("sizes", [SIZES[3], (1, 576, 9, 3, 64, 1536), (1, 384, 6, 2, 128, 640)])
def test_values_that_never_came_are_not_numbers(sizes):
    """Attention that gives up at its first look, where the query, the key and as many of a value's sixteen as a kv head has heads carry
    the launch's tag already and the others the one before's: the result is the right one (they came in time) or is not a number."""
    _, _, heads, kv, dim, _ = sizes
    at = _Launches(sizes, 6)
    words, of_second = at.words_of(), at.words_of()
    at.run(words, 0, at.xs[0])
    right = at.run(of_second, 1, at.xs[1])
    there = torch.arange((heads + 2 * kv) * dim, device="cuda")
    there = there[(there < (heads + kv) * dim) | (there % 16 < heads // kv)]
    words[there] = of_second[there]
    got = at.run(words, 1, at.xs[1], impatient=True)
    assert right.isfinite().all() and (torch.equal(got, right) or got.isnan().all())


@pytest.mark.parametrize("recorded", [False, True])
def test_reloaded_weights_are_used(recorded):
    """Steps recorded on other weights are forgotten with them, and the route's own memory is made anew."""
    from dli_amd.engine.core import build_core
    from dli_amd.trace import TraceSession
    from dli_amd.weights import load_model, write_random_model

    with tempfile.TemporaryDirectory() as tmp:
        folder = write_random_model(Path(tmp) / "m", _config(*SIZES[3]), seed=3, std=0.1)
        _, weights = P.load_folder(folder)
        model = load_model(folder, dtype="bfloat16")
    core = build_core(model, num_pages=8, page_size=16, max_seqs=4, enable_prefix_caching=False, watermark=0.0)
    if recorded:
        core.step.enable_decode_graphs(1, 32)
    session = TraceSession(core)
    step = lambda name: session.step([{"id": name, "tokens": [7], "want": [0]}]).clone()
    first, again = step("a"), step("b")
    assert torch.equal(first, again)
    before = core.step.caches.flow
    kinds = {"matrix": torch.bfloat16, "float32": torch.float32}
    model.load_weights({n: (weights[n].float() * 0.5).to("cuda", kinds[s.role]) for n, s in model.weight_specs().items()})
    second = step("c")
    assert core.step.caches.flow is not before and not torch.equal(first, second)
    core.step.graphs, model.native_steps = None, False
    by_blocks = step("d")
    assert (second - by_blocks).norm() <= 0.02 * by_blocks.norm()
