"""Parts of one's own that derive from built-in ones: where they change what their parent computes, the fused forms that
they inherit step aside, in both runtimes."""

from __future__ import annotations

import contextlib
import dataclasses
from types import SimpleNamespace

import pytest
import torch

from dli_amd.parts import PartSpec, register_part, unregister_part
from dli_amd.parts.attention import GQAttention
from dli_amd.parts.base import Runtime, fused_form, takes_stream
from dli_amd.parts.block import NormPair, ParallelNormsBlock, PreNormBlock
from dli_amd.parts.embedding import TokenEmbedding
from dli_amd.parts.experts import RoutedExperts
from dli_amd.parts.feed_forward import GatedMLP
from dli_amd.parts.head import LinearHead
from dli_amd.parts.norm import RMSNorm

gpu = pytest.mark.gpu
ROLES = {"mixer": GQAttention, "feed_forward": GatedMLP, "mixer_norm": RMSNorm, "feed_forward_norm": RMSNorm}


def _halved(parent):
    class Halved(parent):
        calls = 0

        def forward(self, *args, **kw):
            type(self).calls += 1
            return super().forward(*args, **kw) * 0.5
    return Halved


def test_the_form_and_the_method_that_it_stands_for():
    class Plain:
        rt = SimpleNamespace(is_bf16=False)

        def forward(self): ...

    class Fused(Plain):
        streams_32_bit = True

        def forward_stream(self): ...

    class Changed(Fused):
        def forward(self): ...

    class Both(Changed):
        def forward_stream(self): ...

    class Mixin:
        def forward(self): ...

    class Mixed(Mixin, Fused): ...

    class Same(Fused):
        def other(self): ...

    assert [fused_form(c(), "forward_stream") is not None for c in (Plain, Fused, Changed, Both, Mixed, Same)] == \
        [False, True, False, True, False, True]
    assert fused_form(Changed(), "forward_stream", "other") is not None and fused_form(Same(), "forward_stream", "other") is None
    own = Fused()
    own.forward = lambda: None
    assert fused_form(own, "forward_stream") is None
    # a 32-bit stream goes only to a form whose class, or one below, takes it
    assert takes_stream(Fused()) and takes_stream(Same()) and not takes_stream(Both())
    Plain.rt.is_bf16 = True
    assert takes_stream(Both()) and not takes_stream(Changed())


def _pre_norm(classes):
    rt = Runtime(torch.device("cpu"), torch.float32)
    parts = {"mixer": classes["mixer"](rt, hidden_size=64, num_heads=4, num_kv_heads=2, head_dim=16,
                                       position=PartSpec("rotary", {"dim": 16, "theta": 1e4})),
             "feed_forward": classes["feed_forward"](rt, hidden_size=64, intermediate_size=96)}
    for role in ("mixer_norm", "feed_forward_norm"):
        parts[role] = classes[role](rt, width=64, eps=1e-5)
        parts[role].weight = torch.ones(64)
    parts["mixer"].w_qkv, parts["feed_forward"].w_gate_up = torch.zeros(128, 64), torch.zeros(192, 64)
    parts["mixer"].finalize()
    parts["mixer"].position.finalize()
    return PreNormBlock(rt), parts


@pytest.mark.parametrize("changed", [None, *ROLES])
def test_a_pre_norm_block_asks_for_the_parts_own_arithmetic(changed):
    ctx = SimpleNamespace(num_tokens=2, num_decode=2, num_entries=2, page_size=16)
    block, parts = _pre_norm({role: _halved(cls) if role == changed else cls for role, cls in ROLES.items()})
    assert block.streams(ctx, parts) == (changed is None)


@pytest.mark.parametrize("role", ["mixer", "feed_forward"])
def test_a_32_bit_step_is_fused_where_that_is_ahead(role):
    block, parts = _pre_norm(ROLES)
    matrix = {"mixer": "w_qkv", "feed_forward": "w_gate_up"}[role]
    setattr(parts[role], matrix, torch.zeros(8256, 64))   # more columns than three rows and more are normalised for again
    ctx = lambda n: SimpleNamespace(num_tokens=n, num_decode=n, num_entries=n, page_size=16)
    assert block.streams(ctx(2), parts) and not block.streams(ctx(3), parts)


@pytest.mark.parametrize("changed", [False, True])
def test_a_parallel_block_adds_what_its_feed_forward_computes(changed, monkeypatch):
    """On the CPU, with plain additions in the kernels' place: ones from the experts, halved by a class of one's own."""
    from dli_amd.kernels import ops

    class Ones(RoutedExperts):
        def __init__(self): ...

        def forward(self, x, ctx):
            return torch.ones_like(x)

        def forward_into_stream(self, x, ctx, stream, other, following):
            stream += other + 1.0

    monkeypatch.setattr(ops, "add_pair_into_stream", lambda x, a, b: x.add_(a + b))
    ff = (_halved(Ones) if changed else Ones)()
    norm = SimpleNamespace(forward=lambda x: x)
    x = torch.zeros(2, 4)
    ParallelNormsBlock(Runtime(torch.device("cpu"), torch.float32)).forward(
        x, None, None, None, {"mixer_norm": norm, "mixer": SimpleNamespace(forward=lambda h, ctx, cache: torch.zeros_like(h)),
                              "feed_forward_norm": norm, "feed_forward": ff})
    assert torch.equal(x, torch.full((2, 4), 0.5 if changed else 1.0))


def test_norms_of_ones_own_are_no_pair():
    rt = Runtime(torch.device("cpu"), torch.float32)
    plain, halved = RMSNorm(rt, width=8, eps=1e-5), _halved(RMSNorm)(rt, width=8, eps=1e-5)
    assert NormPair.of(plain, plain) is not None and NormPair.of(plain, halved) is None and NormPair.of(halved, plain) is None


# ------------------------------------------------------------------ whole models

@contextlib.contextmanager
def _registered(family, cls):
    register_part(family, "toy_halved")(cls)
    try:
        yield
    finally:
        unregister_part(family, "toy_halved")


def _renamed(spec):
    return dataclasses.replace(spec, kind="toy_halved")


def _decoded(model, prompts, steps):
    from dli_amd.engine.core import build_core
    from dli_amd.trace import TraceSession

    session = TraceSession(build_core(model, num_pages=16, page_size=16, max_seqs=4, enable_prefix_caching=False, watermark=0.0))
    outs = [session.step([{"id": i, "tokens": p, "want": [len(p) - 1]} for i, p in enumerate(prompts)]).clone()]
    for s in range(steps):
        outs.append(session.step([{"id": i, "tokens": [7 + 3 * i + s], "want": [0]} for i in range(len(prompts))]).clone())
    return outs


@gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("role", [None, *ROLES, "embedding", "final_norm", "head"])
def test_decode_steps_of_a_model_with_a_part_of_ones_own(role, dtype):
    from dli_amd.architectures.llama import build_llama_spec
    from dli_amd.config import LlamaConfig, register_architecture
    from dli_amd.weights import load_model
    from tiny_configs import model_folder

    top = {"embedding": TokenEmbedding, "final_norm": RMSNorm, "head": LinearHead}
    family = "norm" if role and role.endswith("norm") else role
    cls = _halved({**ROLES, **top}[role]) if role else None

    def build(cfg):
        spec = build_llama_spec(cfg)
        if role in top:
            return dataclasses.replace(spec, **{role: _renamed(getattr(spec, role))})
        layers = [dataclasses.replace(ls, parts={**ls.parts, role: (ls.parts[role][0], _renamed(ls.parts[role][1]))}) if role else ls
                  for ls in spec.layers]
        return dataclasses.replace(spec, layers=tuple(layers))

    register_architecture("LlamaForCausalLM", LlamaConfig.from_hf_dict, build, model_types=("llama",), replace=True)
    try:
        with _registered(family, cls) if role else contextlib.nullcontext():
            models = [load_model(model_folder("D"), dtype=dtype) for _ in range(2)]
    finally:
        register_architecture("LlamaForCausalLM", LlamaConfig.from_hf_dict, build_llama_spec, model_types=("llama",), replace=True)
    models[1].STREAM_ROWS = 0   # part by part
    fused, inner = [], models[0]._forward_stream
    models[0]._forward_stream = lambda *a: fused.append(1) or inner(*a)
    got, want = (_decoded(m, [list(range(3, 40)), list(range(50, 61))], 3) for m in models)
    assert len(fused) == (0 if role else 3)
    if role:
        assert cls.calls > 0 and all(torch.equal(g, w) for g, w in zip(got, want))
    else:   # the same sums in another order
        bound = 1e-4 if dtype == "float32" else 0.05
        assert all((g - w).abs().max() <= bound * w.abs().max() for g, w in zip(got, want))


@gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_experts_of_ones_own_beside_a_mixer(dtype, tmp_path, monkeypatch):
    import plain_betepel as T
    from dli_amd.parts import registry
    from dli_amd.weights import load_model

    mlp = {"kind": "moe", "expert": {"ff": 40}, "router": {"experts": 5, "top": 2}, "shared": {"ff": 24}}
    mixer = {"heads": 4, "kv_heads": 2, "dim": 16, "vdim": 24, "scale": 0.25, "diff": 0.4, "mask": {"size": 6, "keep_first": 2},
             "rot": {"dims": 8, "base": 1000.0, "scaling": {"factor": 4.0, "low": 1.0, "high": 4.0, "original": 32}}}
    cfg = {"architecture": "Betepel", "vocab": 120, "width": 64, "norm": {"eps": 1e-5}, "logit_scale": 0.5,
           "layers": [{"type": "attention", "mixer": mixer, "mlp": mlp}] * 2}
    folder = T.write_folder(tmp_path / "betepel", cfg, T.random_weights(cfg, seed=5))
    halved = _halved(RoutedExperts)
    plain = _decoded(load_model(folder, dtype=dtype), [list(range(3, 40)), list(range(50, 61))], 3)
    monkeypatch.setitem(registry._REGISTRY["feed_forward"], "routed_experts", halved)
    got = _decoded(load_model(folder, dtype=dtype), [list(range(3, 40)), list(range(50, 61))], 3)
    assert halved.calls == 2 * 4
    monkeypatch.delattr(RoutedExperts, "forward_into_stream")
    want = _decoded(load_model(folder, dtype=dtype), [list(range(3, 40)), list(range(50, 61))], 3)
    assert all(torch.equal(g, w) for g, w in zip(got, want))
    assert not any(torch.allclose(g, p, atol=1e-3) for g, p in zip(got, plain))


def test_a_block_of_ones_own_is_told_of_norms_only():
    """A block that takes ``following`` may apply whatever it is handed: a norm, or nothing where the next block meets the stream with
    two; that pair goes to the blocks that know it."""
    from dli_amd.parts.base import Norm
    from dli_amd.parts.model import BuiltLayer, Model

    rt = Runtime(torch.device("cpu"), torch.float32)
    norms = {"mixer_norm": RMSNorm(rt, width=8, eps=1e-5), "feed_forward_norm": RMSNorm(rt, width=8, eps=1e-5)}
    for n in norms.values():
        n.weight = torch.ones(8)
    both = BuiltLayer(ParallelNormsBlock(rt), {**norms, "mixer": None, "feed_forward": None})
    alone = BuiltLayer(ParallelNormsBlock(rt), {"mixer_norm": norms["mixer_norm"], "mixer": None})
    changed = BuiltLayer(_halved(ParallelNormsBlock)(rt), both.parts)
    assert Model._met_with(both, "first_norm") is None and isinstance(Model._met_with(both, "meets"), NormPair)
    assert isinstance(Model._met_with(alone, "first_norm"), Norm) and Model._met_with(alone, "meets") is None
    assert Model._met_with(changed, "first_norm") is None and Model._met_with(changed, "meets") is None


@pytest.mark.parametrize("role", [None, "mixer", "feed_forward", "mixer_norm", "feed_forward_norm"])
def test_one_launch_steps_aside_for_an_object_with_a_form_of_its_own(role):
    """A block or part whose object, not its class, has another ``forward_stream`` or ``fused_params`` is asked for it in steps of one
    row too: all layers in one launch would pass it by."""
    from dli_amd.parts.model import BoundCaches, Model
    from dli_amd.weights.loader import build_model
    from tiny_configs import TINY_B

    model, _ = build_model(TINY_B, Runtime(torch.device("cpu"), torch.bfloat16))
    caches, flow = BoundCaches(), object()
    caches.flow, caches.flow_for = flow, model.weights_version
    assert isinstance(model, Model) and model._decode_flow(caches) is flow
    layer = model.layers[-1]
    part = layer.block if role is None else layer.parts[role]
    form = "fused_params" if "norm" in (role or "") else "forward_stream"
    own = getattr(part, form)
    setattr(part, form, lambda *a, **kw: own(*a, **kw))
    assert model._decode_flow(caches) is None
    delattr(part, form)
    assert model._decode_flow(caches) is flow
