"""Dense projections of a few rows whose K slices are summed inside the launch: against the same slices summed outside."""
import sys

import pytest
import torch

from tests import gpu_util as U

pytestmark = pytest.mark.gpu


def _slices_in_order(part):
    t = torch.zeros_like(part[0])
    for s in part:
        t = t + s
    return t


# rows at both ends of the rule (8 and 9 with SwiGLU or more than 8 slices, 16 and 17 without), one slice, more than 8 slices,
# a width that leaves a last span partly empty, fp8 scales per column and per block
@pytest.mark.parametrize("M", [1, 5, 8, 9, 16, 17])
@pytest.mark.parametrize("K,N,kind", [(2048, 3072, "bf16"), (3072, 2048, "channel"), (128, 512, "bf16"), (2880, 328, "channel"),
                                      (512, 1024, "block")])
def test_slices_summed_in_the_launch(M, K, N, kind):
    from lyra_amd import _lib
    from lyra_amd.kernels import decode_fused as F
    from lyra_amd.nn.quant import QArray, quantize

    print(f"dense finish M={M} K={K} N={N} {kind}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(M + K + N)
    rand = lambda *s: torch.randn(*s, device=dev, generator=gen)  # noqa: E731
    w = (rand(1, K, N) * 0.05).to(torch.bfloat16)
    if kind != "bf16":
        w = quantize(w, torch.float8_e5m2 if kind == "e5m2" else torch.float8_e4m3fn, (256, 256) if kind == "block" else (K, 1))
    x, bias, res = rand(M, K).to(torch.bfloat16), rand(1, N).to(torch.bfloat16).float(), rand(M, N).to(torch.bfloat16)
    one = _lib.row_count(M, dev)
    sums = _slices_in_order(F.gemm_unsummed(x, w, one).partials)
    r16 = lambda t: t.to(torch.bfloat16).float()  # noqa: E731
    for _ in range(3):  # (the arrival counters are zero again after every call)
        assert torch.equal(F.gemm(x, w, one, out_f32=True), sums)
        assert torch.equal(F.gemm(x, w, one), sums.to(torch.bfloat16))
        assert torch.equal(F.gemm(x, w, one, bias=bias), (sums + bias).to(torch.bfloat16))
        got = F.gemm(x, w, one, bias=bias, bias_after_cast=True, residual=res, out_scale=0.25)
        assert torch.equal(got, (res.float() + r16(r16(r16(sums) + bias) * 0.25)).to(torch.bfloat16))
    if N % 16 == 0:
        g, lin = (sums + bias).double().split(N // 2, 1)
        g, lin = g.clamp(max=7.0), lin.clamp(-7.0, 7.0)
        want = (lin + 1) * g * torch.sigmoid(1.702 * g)
        for tiled in ([False, True] if N // 2 % 32 == 0 else [False]):
            got = F.gemm(x, w, one, bias=bias, fused_swiglu=True, out_tiled=tiled)
            got = got.untiled() if tiled else got
            # (one rounding to bf16 behind float32 arithmetic with a 1-ulp reciprocal and exponential)
            assert ((got.double() - want).abs() <= want.abs() * 2.0**-8 + 1e-5).all()
    # a row count below M: the rows behind it are products of nothing, whatever the weights hold
    bad = w.clone() if kind == "bf16" else QArray(w.qval.clone(), w.scale.clone(), w.block)
    if kind == "bf16":
        bad[0, 0, 0] = float("inf")
    else:
        bad.scale.view(-1)[0] = float("inf")
    few = _lib.row_count(M // 2, dev)
    got = F.gemm(x, bad, few, out_f32=True)
    assert (got[M // 2 :] == 0).all() and torch.isfinite(got[M // 2 :]).all()
    ws = [v for k, v in _lib._WORKSPACES.items() if k[0] == "gemm"]
    torch.cuda.synchronize()
    assert all(int(b[:65536].view(torch.int32).abs().sum()) == 0 for b in ws)


# slices longer than a wavefront's register sets hold at once (1024, 2048 and 768 rows: the middle variant's projections), the sum
# inside the launch up to 8 rows, with more than 8 only without SwiGLU
@pytest.mark.parametrize("M", [1, 8, 9, 16])
@pytest.mark.parametrize("K,N,kind", [(4096, 6144, "bf16"), (4096, 6144, "block"), (4096, 12288, "channel"), (6144, 4096, "channel"),
                                      (6144, 4096, "e5m2")])
def test_long_slices_summed_in_the_launch(M, K, N, kind):
    from lyra_amd import _lib

    assert K / _lib.gemm_splits(M, K, N, 0 if kind == "bf16" else (256 if kind == "block" else K)) > 512
    test_slices_summed_in_the_launch(M, K, N, kind)


# slices of at most 2048 rows, also where that makes a second round of workgroups: longer ones add up more terms in a row
@pytest.mark.parametrize("M,K,N,kind,splits", [(128, 4096, 12288, "channel", 2), (192, 6144, 4096, "channel", 3), (256, 2880, 5120, "bf16", 2),
                                               (97, 4096, 12288, "block", 2), (96, 4096, 12288, "channel", 2), (129, 6144, 4096, "channel", 3),
                                               (256, 4096, 12288, "channel", 2)])
def test_slices_of_at_most_2048_rows(M, K, N, kind, splits):
    from lyra_amd import _lib
    from lyra_amd.kernels import decode_fused as F
    from lyra_amd.nn.quant import quantize

    print(f"dense plan M={M} K={K} N={N} {kind}", file=sys.stderr, flush=True)
    dev, gen = U.dev(), torch.Generator(device=U.dev()).manual_seed(M + K)
    w = (torch.randn(1, K, N, device=dev, generator=gen) * 0.05).to(torch.bfloat16)
    x = torch.randn(M, K, device=dev, generator=gen).to(torch.bfloat16)
    if kind == "bf16":
        ref = w[0].double()
    else:
        w = quantize(w, torch.float8_e4m3fn, (K, 1) if kind == "channel" else (256, 256))
        s = w.scale[0].double().repeat_interleave(w.block[0], 0).repeat_interleave(w.block[1], 1)
        ref = w.qval[0].float().double() * s
    got = F.gemm_unsummed(x, w, _lib.row_count(M, dev)).partials
    assert got.shape == (splits, M, N)
    err = (got.double().sum(0) - x.double() @ ref).abs()
    # exact products of bf16 operands, float32 sums of K / 128 matrix instructions per wavefront and of 4 wavefronts
    assert (err <= 2.0**-18 * (x.double().abs() @ ref.abs())).all()
