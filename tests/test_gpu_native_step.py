"""lyra_decode_step (all layers of a decode step in one call) against the Python loop over the same launches: logits and every
byte of the caches."""
import sys
from dataclasses import replace

import pytest
import torch

from tests import gpu_util as U

pytestmark = pytest.mark.gpu


def _cfg(name):
    from lyra_amd.model import MODEL_VARIANTS, apply_inference_overrides, interleaved_moe

    small = replace(MODEL_VARIANTS["lyra-small"], n_layers=3, mlp_map=interleaved_moe(3, first=2, every=2), vocab_size=3000, padded_vocab_size=3072)
    gpt = replace(MODEL_VARIANTS["gpt-oss-20b"], n_layers=3, mlp_map=("moe", "dense", "moe"), n_embd=320, n_attn_heads=4, n_kv_heads=2, seq_len=512,
                  n_routed_experts=6, n_active_experts=2, vocab_size=1000, padded_vocab_size=1024)
    return {
        "dev": MODEL_VARIANTS["dev"],
        "small-bf16": small,
        "small-serve": apply_inference_overrides(small, fp8=True),
        "small-fp8": apply_inference_overrides(small, fp8=True, fp8_attn=True, per_channel=True),
        "small-e5m2": replace(apply_inference_overrides(small, fp8=True, fp8_attn=True), gemm_dtype=torch.float8_e5m2),
        "biases": gpt,
        "dense-only": replace(small, mlp_map=("dense",) * 3, use_sdpa_output_gate=False),
        "wide-gate": replace(small, n_attn_heads=32, head_dim=64),
    }[name]


def _logits(model, cache, tokens, cfg, native):
    import lyra_amd.model as M

    kept, M._NATIVE_STEP = M._NATIVE_STEP, native
    try:
        return M.model_apply(tokens, model, cache, cfg, advance=False)[0]
    finally:
        M._NATIVE_STEP = kept


def _cache_bytes(cache):
    from lyra_amd.nn.quant import QArray

    for layer in cache.layers:
        for t in (layer.k, layer.v):
            yield from ((t.qval.view(torch.uint8), t.scale) if isinstance(t, QArray) else (t,))


@pytest.mark.parametrize("name,B", [("dev", 1), ("dev", 33), ("small-bf16", 1), ("small-bf16", 8), ("small-serve", 9), ("small-serve", 3),
                                    ("small-fp8", 65), ("small-e5m2", 5), ("biases", 2), ("biases", 20), ("dense-only", 4), ("wide-gate", 4)])
def test_one_call_equals_the_launches_one_by_one(name, B, monkeypatch):
    import lyra_amd.model as M

    print(f"native step {name} B={B}", file=sys.stderr, flush=True)
    cfg, dev, S = _cfg(name), U.dev(), 300
    model = M.init_weights(cfg, dev, seed=B)
    tokens = torch.arange(B, dtype=torch.int32, device=dev) * 7 % cfg.vocab_size
    taken = []
    inner = M._layers_native
    monkeypatch.setattr(M, "_layers_native", lambda *a: taken.append(inner(*a)) or taken[-1])
    results = []
    for native in (False, True):
        gen = torch.Generator(device=dev).manual_seed(3)
        cache = M.init_cache(cfg, B, S, dev)
        for t in _cache_bytes(cache):
            if t.dtype == torch.uint8:
                t.random_(0, 0x60, generator=gen)  # (finite codes of both formats)
            elif t.dtype == torch.float32:
                t.uniform_(0.001, 0.003, generator=gen)
            else:
                t.normal_(generator=gen)
        cache.pos.fill_(257)
        results.append([_logits(model, cache, tokens, cfg, native)] + [t.clone() for t in _cache_bytes(cache)])
        results[-1].append(_logits(model, cache, tokens, cfg, native))  # (a second pass on the same caches)
    torch.cuda.synchronize()
    assert len(taken) == 2 and all(t is not None for t in taken), "the one-call path was not taken"
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_layers_that_share_a_parameters_memory():
    """One copy of a converted parameter is kept per address: the copies that two layers make of the same memory through tensors of
    their own have to outlive the results allocated after them."""
    import lyra_amd.model as M

    cfg, dev = _cfg("small-bf16"), U.dev()
    model = M.init_weights(cfg, dev, seed=4)
    first, last = model.layers[0].attn, model.layers[2].attn
    last.sdpa_gate = first.sdpa_gate.view(first.sdpa_gate.shape)
    tokens = torch.arange(8, dtype=torch.int32, device=dev)
    want = _logits(model, M.init_cache(cfg, 8, 64, dev), tokens, cfg, False)
    for _ in range(3):
        assert torch.equal(_logits(model, M.init_cache(cfg, 8, 64, dev), tokens, cfg, True), want)


def test_steps_that_the_call_does_not_cover_run_from_python(monkeypatch):
    import lyra_amd.model as M

    cfg, dev = _cfg("dev"), U.dev()
    model = M.init_weights(cfg, dev, seed=2)
    tokens = torch.arange(4, dtype=torch.int32, device=dev)
    fresh = lambda: M.init_cache(cfg, 4, 64, dev)  # noqa: E731
    want = _logits(model, fresh(), tokens, cfg, False)
    # 64-bit token ids; a position per row
    assert torch.equal(_logits(model, fresh(), tokens.long(), cfg, True), want)
    cache = fresh()
    cache.pos = torch.zeros(4, dtype=torch.int32, device=dev)
    U.assert_close(U.to_np(_logits(model, cache, tokens, cfg, True))[:, : cfg.vocab_size], U.to_np(want)[:, : cfg.vocab_size])
    # what a launch refuses: remembered, and the step is the Python loop's
    monkeypatch.setattr(M, "_NATIVE_REFUSED", set())
    monkeypatch.setattr(M._lib.lib, "lyra_decode_step", lambda *a: M._lib.E_UNSUPPORTED)
    assert torch.equal(_logits(model, fresh(), tokens, cfg, True), want) and len(M._NATIVE_REFUSED) == 1
    monkeypatch.setattr(M._lib.lib, "lyra_decode_step", lambda *a: pytest.fail("asked again"))
    assert torch.equal(_logits(model, fresh(), tokens, cfg, True), want)


@pytest.mark.parametrize("refused", ["lyra_decode_step", "lyra_decode_step_scratch"])
def test_a_refusal_is_remembered_for_its_formats_and_cache_length_only(refused, monkeypatch):
    import lyra_amd.model as M

    dev, tokens = U.dev(), torch.arange(4, dtype=torch.int32, device=U.dev())
    step = lambda m, cfg, S: _logits(m, M.init_cache(cfg, 4, S, dev), tokens, cfg, True)  # noqa: E731
    bf16, block, channel = _cfg("small-bf16"), _cfg("small-serve"), _cfg("small-fp8")  # (the same widths)
    models = [M.init_weights(cfg, dev, seed=2) for cfg in (bf16, block, channel)]
    monkeypatch.setattr(M, "_NATIVE_REFUSED", set())
    asked, inner = [], getattr(M._lib.lib, refused)
    answer = {"lyra_decode_step": M._lib.E_UNSUPPORTED, "lyra_decode_step_scratch": 0}[refused]
    monkeypatch.setattr(M._lib.lib, refused, lambda *a: asked.append(a) or (answer if len(asked) == 1 else inner(*a)))
    step(models[1], block, 64)
    step(models[1], block, 64)
    assert len(asked) == 1 and len(M._NATIVE_REFUSED) == 1
    step(models[0], bf16, 64)
    step(models[2], channel, 64)
    step(models[1], block, 96)
    assert len(asked) == 4 and len(M._NATIVE_REFUSED) == 1


def test_fewer_caches_than_layers_are_an_error():
    import lyra_amd.model as M

    cfg, dev = _cfg("dev"), U.dev()
    model, tokens = M.init_weights(cfg, dev, seed=2), torch.arange(4, dtype=torch.int32, device=dev)
    for native in (True, False):
        cache = M.init_cache(cfg, 4, 64, dev)
        cache.layers.pop()
        with pytest.raises(IndexError):
            _logits(model, cache, tokens, cfg, native)


def test_arguments_and_scratch_are_checked_before_any_launch():
    import ctypes

    import lyra_amd.model as M
    from lyra_amd import _lib

    L = _lib.lib
    assert L.lyra_decode_step(None, None) == -1 and L.lyra_decode_step_scratch(None) == 0
    layer = ctypes.create_string_buffer(b"\0" * M._LAYER.size)
    bad = M._STEP.pack(ctypes.addressof(layer), *([256] * 13), 1, 4, 256, 2, 1, 64, 0, 10, 10, 384, 0, 0, 0, 0, 1e-5, 1.0, 1.0, 1.0, 1.0, 1.0)
    assert L.lyra_decode_step(bad, None) == -1 and L.lyra_decode_step_scratch(bad) == 0  # no weights
    ptrs = lambda n: [256] * n  # noqa: E731
    good = M._LAYER.pack(256, *([256, 0, 0, 0, 0, 0] * 2), *ptrs(10), 64, 0, 256, *([256, 0, 0, 0, 0, 0] * 2), 0, 0, 0, 0)
    layer = ctypes.create_string_buffer(good, len(good))
    tail = (1, 4, 256, 2, 1, 64, 0, 10, 10, 384, 0, 0, 0, 0, 1e-5, 1.0, 1.0, 1.0, 1.0, 1.0)
    need = L.lyra_decode_step_scratch(M._STEP.pack(ctypes.addressof(layer), *ptrs(13), *tail))
    assert need > 0
    # the first result already does not fit: refused before the first launch (none of these addresses is ever used)
    small = M._STEP.pack(ctypes.addressof(layer), *ptrs(12), 512, *tail)
    assert L.lyra_decode_step(small, None) == -3
