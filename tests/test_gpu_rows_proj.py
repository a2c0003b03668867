"""The down projection of a few rows that forms its own input (SwiGLU of an up projection left in slices), against the launches
it stands for."""
import sys

import pytest
import torch

from tests import gpu_util as U

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


# one row and the most rows, one slice of the up projection and more than are requested at once (6), slices of 128, 256, 384 and
# 512 rows, a last span that the columns do not fill; scales per column, one block along all of K, and blocks along K that hold a
# wavefront's rows (128 and 256) or change within them (32 and 64)
@pytest.mark.parametrize("M,K,N,kind,splits,with_bias", [
    (1, 256, 512, "bf16", 2, False), (16, 3072, 2048, "channel", 4, False), (5, 2048, 6144, "block", 6, True), (9, 512, 136, "bf16", 13, True),
    (3, 2880, 5120, "channel", 7, False), (8, 1024, 2048, "e5m2", 1, False), (16, 768, 4096, "block", 3, True),
    (4, 1024, 2048, "b32", 3, False), (7, 2048, 6144, "b64", 2, True), (13, 2048, 6144, "b32", 4, False), (6, 2048, 2048, "column", 4, False),
    (10, 3456, 3584, "b128", 3, False), (2, 2880, 2816, "bf16", 4, True)])
@pytest.mark.parametrize("packed", [False, True])
def test_swiglu_inside_the_down_projection(M, K, N, kind, splits, with_bias, packed):
    from lyra_amd import _lib
    from lyra_amd.kernels import decode_fused as F
    from lyra_amd.nn.quant import quantize

    print(f"rows_proj_swiglu M={M} K={K} N={N} {kind} splits={splits} packed={packed}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(M * 5 + K + N)
    rand = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    w = (rand(1, K, N) * 0.05).to(torch.bfloat16)
    w_abs = w[0].abs().double()
    if kind != "bf16":
        block = {"block": (256, 256), "b32": (32, 32), "b64": (64, 64), "b128": (128, 128), "column": (K, 128)}.get(kind, (K, 1))
        w = quantize(w, torch.float8_e5m2 if kind == "e5m2" else FP8, block)
        s = w.scale[0].double().repeat_interleave(w.block[0], 0).repeat_interleave(w.block[1], 1)
        w_abs = (w.qval[0].float().double() * s).abs()
    sums = 3 * rand(splits, M, 2 * K)
    bias = rand(2 * K).to(torch.bfloat16).float() if with_bias else None
    got = F.rows_proj_swiglu(F.Unsummed(sums), F.pack_weights(w) if packed else w, 1.702, 7.0, bias=bias)
    # the operand: slices added in slice order, bias, SwiGLU, one rounding to bf16
    total = torch.zeros(M, 2 * K, device=dev)
    for part in sums:
        total = total + part
    if bias is not None:
        total = total + bias
    g, lin = total.double().split(K, 1)
    g, lin = g.clamp(max=7.0), lin.clamp(-7.0, 7.0)
    o = (lin + 1) * g * torch.sigmoid(1.702 * g)
    want = F.gemm_unsummed(o.to(torch.bfloat16), w, _lib.row_count(M, dev))
    torch.cuda.synchronize()
    assert got.partials.shape == want.partials.shape
    # float32 SwiGLU with a 1-ulp reciprocal and exponential against float64: an operand may round to the other neighbour in bf16
    # (2^-8 of it) where it lies next to a tie, a thousandth of them; and the order of float32 sums
    err = (got.partials.double().sum(0) - want.partials.double().sum(0)).abs()
    bound = (o.abs() * 2.0**-8) @ w_abs * 0.05 + (o.abs() * 2.0**-18 + 1e-4 * 2.0**-8) @ w_abs
    assert (err <= bound).all(), (err / bound).max()


@pytest.mark.parametrize("M,kind", [(1, "bf16"), (8, "channel"), (16, "block")])
def test_mlp_of_a_few_rows_is_the_same_with_the_launch_in_between(M, kind, monkeypatch):
    """The whole dense MLP of a layer with and without the launch: the slices that go on to the next norm, bit for bit."""
    from dataclasses import replace

    import lyra_amd.model as model
    from lyra_amd.kernels import decode_fused as F

    cfg = replace(model.MODEL_VARIANTS["lyra-small"], n_layers=1, mlp_map=("dense",), vocab_size=100, padded_vocab_size=128)
    if kind != "bf16":
        cfg = model.apply_inference_overrides(cfg, fp8=True, per_channel=kind == "channel")
    w = model.init_weights(cfg, U.dev(), seed=4).layers[0].mlp
    x = torch.randn(M, cfg.n_embd, device=U.dev(), generator=torch.Generator(device=U.dev()).manual_seed(M)).to(torch.bfloat16)
    outs = []
    for on in (True, False):
        monkeypatch.setattr(model, "_ROWS_PROJ", on)
        outs.append(model.dense_mlp_apply_fused(x, w, cfg))
    assert all(isinstance(o, F.Unsummed) for o in outs)
    assert torch.equal(outs[0].partials, outs[1].partials) and torch.equal(outs[0].residual, outs[1].residual)


def test_more_rows_and_other_weights_are_left_to_the_launch_in_between():
    from lyra_amd.kernels import decode_fused as F

    w = torch.zeros(1, 512, 512, dtype=torch.bfloat16, device=U.dev())
    up = lambda M: F.Unsummed(torch.zeros(2, M, 1024, device=U.dev()))  # noqa: E731
    assert F.rows_proj_swiglu(up(17), w, 1.702, 7.0) is None and not F.rows_proj_swiglu_exists(17, w)
    assert F.rows_proj_swiglu(up(4), w.expand(2, -1, -1).contiguous(), 1.702, 7.0) is None
    assert F.rows_proj_swiglu(up(16), w, 1.702, 7.0) is not None
