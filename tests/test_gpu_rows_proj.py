"""The projections of a few rows that finish their own input (residual update + RMS norm, or SwiGLU) and the attention launch
behind them, each against a float64 restatement or the launches they stand for."""
import sys

import pytest
import torch

from tests import gpu_util as U

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


def _weights(gen, kind, K, N):
    from lyra_amd.nn.quant import quantize

    w = torch.randn(1, K, N, device=U.dev(), generator=gen).mul_(0.05).to(torch.bfloat16)
    if kind == "bf16":
        return w, w[0].double(), w[0].abs().double()
    q = quantize(w, torch.float8_e5m2 if kind == "e5m2" else FP8, (K, 1) if kind != "block" else (256, 256))
    # (the scales are applied to the float32 products: the reference operand is not rounded to bf16)
    s = q.scale[0].double().repeat_interleave(q.block[0], 0).repeat_interleave(q.block[1], 1)
    d = q.qval[0].to(torch.float32).double() * s
    return q, d, d.abs()


# one row and the most rows, one slice set and more slices than are requested at once (12 / 6), slices of 256 and 512 rows, a last
# slice that ends inside 256 columns (2880), a last span that the columns do not fill, every scale layout, 0, 1 and 16 gates
SHAPES = [(1, 256, 512, "bf16", 2, 0, False), (8, 2048, 3072, "channel", 12, 16, False), (5, 2048, 6144, "block", 8, 0, True),
          (8, 512, 136, "bf16", 13, 3, True), (3, 2880, 5120, "channel", 7, 1, False), (7, 1024, 2048, "e5m2", 1, 16, False)]


@pytest.mark.parametrize("M,K,N,kind,splits,gates,with_bias", SHAPES)
@pytest.mark.parametrize("packed", [False, True])
def test_norm_inside_the_projection(M, K, N, kind, splits, gates, with_bias, packed):
    from lyra_amd.kernels import decode_fused as F

    print(f"rows_proj_norm M={M} K={K} N={N} {kind} splits={splits} gates={gates} packed={packed}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(M * 7 + K + N)
    rand = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    rhs, w, w_abs = _weights(gen, kind, K, N)
    x = F.Unsummed(rand(splits, M, K), rand(M, K).to(torch.bfloat16), 0.177,
                   rand(K).to(torch.bfloat16).float() if with_bias else None)
    norm = 1 + 0.1 * rand(K)
    gate = rand(K, gates) if gates else None
    eps = 1e-5
    got, x_out = F.rows_proj_norm(x, norm, eps, F.pack_weights(rhs) if packed else rhs, gate=gate)
    want_x = F.rmsnorm_proj(x, norm, eps)[2]
    torch.cuda.synchronize()
    assert torch.equal(x_out.view(torch.int16), want_x.view(torch.int16))
    sq = want_x.double().pow(2).sum(1)
    torch.testing.assert_close(got.factor.sq.double().sum(0), sq, rtol=1e-5, atol=0)  # (float32 sums of 64-term groups)
    a = (want_x.float() * norm).to(torch.bfloat16).double()
    # the products of bf16 operands are exact in float32: what is left are the roundings of K / 32 + splits sums
    err = (got.partials.double().sum(0) - a @ w).abs()
    assert (err <= 2.0**-18 * (a.abs() @ w_abs) + 1e-30).all(), err.max()
    if gates:
        err = (got.factor.gate.double().sum(0) - a @ gate.double()).abs()
        assert (err <= 2.0**-18 * (a.abs() @ gate.double().abs())).all(), err.max()
    else:
        assert got.factor.gate is None
    assert (got.factor.width, got.factor.eps) == (K, eps)


@pytest.mark.parametrize("M,K,N,kind,splits,gates,with_bias", SHAPES)
def test_swiglu_inside_the_projection(M, K, N, kind, splits, gates, with_bias):
    from lyra_amd.kernels import decode_fused as F

    print(f"rows_proj_swiglu M={M} K={K} N={N} {kind} splits={splits}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(M * 5 + K + N)
    rand = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    rhs, w, w_abs = _weights(gen, kind, K, N)
    sums, sq, width, eps, beta, limit = 3 * rand(splits, M, 2 * K), rand(9, M).abs() * 200, 1800, 1e-5, 1.702, 7.0
    bias = rand(2 * K).to(torch.bfloat16).float() if with_bias else None
    got = F.rows_proj_swiglu(F.Unsummed(sums, factor=F.RowFactor(sq, width, eps, None)), rhs, beta, limit, bias=bias)
    torch.cuda.synchronize()
    t = sums.double().sum(0) * torch.rsqrt(sq.double().sum(0) / width + eps)[:, None]
    if bias is not None:
        t = t + bias.double()
    g, lin = t[:, :K].clamp(max=limit), t[:, K:].clamp(-limit, limit)
    o = (lin + 1) * g * torch.sigmoid(beta * g)
    # the operand is rounded to bf16 (2^-9 of it), behind float32 arithmetic whose errors are of the order of 1e-6
    bound = (o.abs() * 2.0**-9 + 1e-4) @ w_abs + 2.0**-18 * (o.abs() @ w_abs)
    err = (got.partials.double().sum(0) - o @ w).abs()
    assert (err <= bound).all(), (err / bound).max()


@pytest.mark.parametrize("B,N,K,S,H,fp8,sw,splits", [(1, 16, 4, 700, 128, False, 0, 8), (8, 16, 4, 300, 128, True, 0, 12),
                                                     (8, 16, 4, 300, 128, True, 128, 8), (3, 2, 1, 90, 64, False, 0, 2)])
def test_attention_behind_rows_that_lack_their_factor(B, N, K, S, H, fp8, sw, splits):
    """Factors that are powers of two and gates of exactly 0, 1 and 2, so that the launch has to agree with the one on complete
    slices bit for bit, the caches included."""
    from lyra_amd.kernels import decode_fused as F
    from lyra_amd.nn.quant import quantize

    print(f"attention rows B={B} N={N} K={K} S={S} H={H} fp8={fp8} sw={sw} splits={splits}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(B + S)
    rand = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    part = rand(splits, B, (N + 2 * K) * H)
    width, parts = 512, 5
    factor = 2.0 ** torch.arange(-2, B - 2, device=dev).float()  # rsqrt(4^-e) = 2^e
    sq = torch.zeros(parts, B, device=dev)
    sq[B % parts] = width * factor.pow(-2)
    gates = torch.tensor([0.0, 1e4, -1e4, 0.0], device=dev)[torch.arange(B * N, device=dev) % 4].reshape(B, N)
    gate_part = torch.zeros(splits, B, N, device=dev)
    gate_part[splits - 1] = gates
    cos, sin = rand(S, H // 2).cos(), rand(S, H // 2).sin()
    qn, kn, sinks = 1 + 0.1 * rand(H), 1 + 0.1 * rand(H), rand(N)
    hist = [rand(B, K, S, H).to(torch.bfloat16) for _ in range(2)]
    cache = lambda: [quantize(h, FP8, (1, H)) if fp8 else h.clone() for h in hist]  # noqa: E731
    pos = torch.tensor(S - 2, dtype=torch.int32, device=dev)
    (ka, va), (kb, vb) = cache(), cache()
    got = F.attention_qkv(F.Unsummed(part, factor=F.RowFactor(sq, width, 0.0, gate_part)), qn, kn, cos, sin, pos, ka, va, sinks,
                          H**-0.5, sw, N, K, H, 1e-5)
    gate = (2 * torch.sigmoid(gates * factor[:, None])).to(torch.bfloat16)
    want = F.attention_qkv(F.Unsummed(part * factor[:, None]), qn, kn, cos, sin, pos, kb, vb, sinks, H**-0.5, sw, N, K, H, 1e-5, gate=gate)
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    for a, b in ((ka, kb), (va, vb)):
        if fp8:
            assert torch.equal(a.qval.view(torch.uint8), b.qval.view(torch.uint8)) and torch.equal(a.scale, b.scale)
        else:
            assert torch.equal(a, b)


def test_more_rows_and_other_inputs_are_left_to_the_launches_in_between():
    from lyra_amd.kernels import decode_fused as F

    dev = U.dev()
    w = torch.zeros(1, 512, 512, dtype=torch.bfloat16, device=dev)
    rows = lambda M: F.Unsummed(torch.zeros(2, M, 512, device=dev), torch.zeros(M, 512, dtype=torch.bfloat16, device=dev))  # noqa: E731
    norm = torch.ones(512, device=dev)
    assert F.rows_proj_norm(rows(9), norm, 1e-5, w) is None and not F.rows_proj_swiglu_exists(9, w)
    assert F.rows_proj_norm(rows(4), norm, 1e-5, w, gate=torch.zeros(512, 17, device=dev)) is None
    assert F.rows_proj_norm(rows(4), norm, 1e-5, w.expand(2, -1, -1).contiguous()) is None
    assert F.rows_proj_norm(rows(8), norm, 1e-5, w) is not None and F.rows_proj_swiglu_exists(8, w)
