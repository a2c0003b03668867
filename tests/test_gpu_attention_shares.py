"""The attention launch whose (row, kv head) pairs do not make whole rounds over the compute units: whole pairs and a chunked
remainder in one launch, against the oracle and against the plan it replaces."""
import sys

import numpy as np
import pytest
import torch

from oracle import clib
from oracle import lyra_oracle as O
from tests import gpu_util as U
from tests.test_gpu_attention import test_learned_exclusive_self_attention_in_the_epilogue as exclusive_self_attention
from tests.test_gpu_fused import test_attention_with_the_front_step_equals_the_two_launches as front_step

pytestmark = pytest.mark.gpu


def _call(case, B, N, K, S, H, pos, ws):
    from lyra_amd import _lib

    q, k, v, sinks = U.attention_torch_inputs(case)
    fp8 = case["fp8"]
    ptr = lambda t: t.data_ptr()  # noqa: E731
    kv = (ptr(k.qval), ptr(v.qval), ptr(k.scale), ptr(v.scale)) if fp8 else (ptr(k), ptr(v), None, None)
    out = torch.full((B, N, 1, H), float("nan"), dtype=torch.float32, device=U.dev())
    p = torch.tensor(pos, dtype=torch.int32, device=U.dev())
    rc = _lib.lib.lyra_decode_attention(ptr(q), *kv, ptr(sinks), ptr(p), 0 if p.dim() == 0 else 1, None, ptr(out),
                                        None if ws is None else ptr(ws), 0 if ws is None else ws.numel(), B, N, K, S, H, H**-0.5, 0,
                                        _lib.DTYPE_E4M3FN if fp8 else _lib.DTYPE_BF16, _lib.DTYPE_F32,
                                        torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return rc, U.to_np(out)


# pairs = B * K: remainders of 1 (cut finest), 4, 8, 36 and 128 pairs (2 chunks) behind one and two rounds, one too large to cut,
# and fewer pairs than units (3 or 2 chunks instead of 4 or 3; whole instead of 2)
@pytest.mark.parametrize("B,K,N,S,H,fp8", [
    (257, 1, 4, 1300, 128, True), (65, 4, 16, 700, 128, True), (33, 8, 32, 1025, 64, True), (73, 4, 16, 300, 128, False),
    (129, 4, 8, 1000, 64, False), (96, 4, 16, 1200, 128, True), (100, 4, 16, 600, 128, True), (23, 4, 16, 1100, 128, True),
    (17, 4, 64, 900, 64, False), (50, 4, 16, 500, 128, True), (65, 4, 16, 1500, 128, True), (33, 8, 32, 2100, 64, True),
    (73, 4, 16, 1000, 128, False), (96, 4, 8, 1500, 128, False),
])
def test_whole_pairs_and_a_chunked_remainder(B, K, N, S, H, fp8):
    from lyra_amd import _lib

    print(f"attention shares B={B} N={N} K={K} S={S} H={H} fp8={fp8}", file=sys.stderr, flush=True)
    case = U.attention_case(B + S, B, N, K, S, H, fp8=fp8)
    need = _lib.lib.lyra_decode_attention_workspace(B, N, K, S, H, 0)
    ws = torch.zeros(need, dtype=torch.uint8, device=U.dev())
    rng = np.random.default_rng(S)
    for pos in (S - 1, S // 2, 0, -1, rng.integers(-1, S, B)):
        rc, got = _call(case, B, N, K, S, H, pos, ws)
        _lib.check(rc, "lyra_decode_attention")
        rc, again = _call(case, B, N, K, S, H, pos, ws)
        assert rc == 0 and np.array_equal(got, again)
        assert int(ws[: 64 * 1024].view(torch.int32).abs().sum()) == 0 or need == 256  # the counters are zero again
        if fp8:
            (kq, ks), (vq, vs) = case["k"], case["v"]
            full = np.broadcast_to(np.asarray(pos, np.int32), (B,)).copy()
            want = clib.decode_attention(O.bf16_bits(case["q"]), kq, vq, ks[..., 0], vs[..., 0], case["sinks"], full, None, H**-0.5, 0)
        else:
            want = O.decode_attention_reference(case["q"], case["k"], case["v"], case["sinks"], H**-0.5, 0, pos)
        U.assert_close(got, want, what=f"shares pos={pos}")
        if B * K > 256:  # without a workspace these ran unchunked, and still do: the same sums in another order
            rc, plain = _call(case, B, N, K, S, H, pos, None)
            assert rc == 0
            # (float32 outputs of probabilities rounded to bf16 against another running maximum: 2^-8 of sum p |v|, |v| < 6)
            np.testing.assert_allclose(got, plain, rtol=0, atol=6 * 2.0**-8)


@pytest.mark.parametrize("B,N,K,S", [(65, 16, 4, 600), (33, 32, 8, 1100), (23, 16, 4, 1100), (65, 16, 4, 1500)])
def test_front_step_in_a_launch_of_uneven_pairs(B, N, K, S):
    front_step(B, N, K, S, 128, True, True, 0, True, "full")


# a launch with a chunked remainder leaves it whole while the cache is filled too little for the merge to pay (104 KB of keys and
# values beyond the first chunk): the same bits as without a workspace below that, the sums in another order from there on
@pytest.mark.parametrize("B,K,N,S,H,fp8,chunk", [(65, 4, 16, 1500, 128, True, 128), (33, 8, 32, 2100, 64, True, 128), (73, 4, 16, 1000, 128, False, 256),
                                                 (96, 4, 8, 1500, 128, False, 768)])
def test_a_remainder_stays_whole_in_a_part_filled_cache(B, K, N, S, H, fp8, chunk):
    from lyra_amd import _lib

    case = U.attention_case(B + S, B, N, K, S, H, fp8=fp8)
    ws = torch.zeros(_lib.lib.lyra_decode_attention_workspace(B, N, K, S, H, 0), dtype=torch.uint8, device=U.dev())
    assert ws.numel() > 256
    first_cut = chunk + 104 * 1024 // (2 * H * (1 if fp8 else 2)) - 1
    for pos, cut in ((-1, False), (chunk, False), (first_cut - 1, False), (first_cut, True), (S - 1, True)):
        print(f"attention part-filled B={B} K={K} S={S} H={H} fp8={fp8} pos={pos}", file=sys.stderr, flush=True)
        rc, got = _call(case, B, N, K, S, H, pos, ws)
        rc2, whole = _call(case, B, N, K, S, H, pos, None)
        assert rc == rc2 == 0 and np.array_equal(got, whole) != cut
        np.testing.assert_allclose(got, whole, rtol=0, atol=6 * 2.0**-8)  # (the bound above)
        assert int(ws[: 64 * 1024].view(torch.int32).abs().sum()) == 0
    # with the front step in the same launch: the new key belongs to the first workgroup of a pair that stays whole
    for pos in (first_cut - 1, first_cut):
        front_step(B, N, K, S, H, fp8, True, 0, True, pos)


# whole pairs and a chunked remainder (65 x 4, 33 x 8 as lyra-medium's heads at 33 rows, 64-wide heads), chunks only (23 x 4)
@pytest.mark.parametrize("B,N,K,S,H", [(65, 16, 4, 1500, 128), (33, 32, 8, 1500, 128), (33, 64, 8, 2100, 64), (23, 16, 4, 1100, 128)])
def test_exclusive_self_attention_in_a_launch_of_uneven_pairs(B, N, K, S, H):
    exclusive_self_attention(B, N, K, S, H, 0, False)


@pytest.mark.parametrize("B,K,N,S,H", [(65, 4, 16, 1500, 128), (33, 8, 32, 2100, 64)])
def test_whole_pairs_and_a_chunked_remainder_in_e5m2(B, K, N, S, H):
    from lyra_amd.kernels.decode_attention import decode_attention

    print(f"attention shares e5m2 B={B} N={N} K={K} S={S} H={H}", file=sys.stderr, flush=True)
    case = U.attention_case(B + S, B, N, K, S, H, fp8=True, fmt=2)
    q, k, v, sinks = U.attention_torch_inputs(case)
    (kq, ks), (vq, vs) = case["k"], case["v"]
    for pos in (S - 1, S // 2):
        at = torch.tensor(pos, dtype=torch.int32, device=U.dev())
        got = decode_attention(q, k, v, sinks, H**-0.5, 0, at, dtype=torch.float32, implementation="pallas")
        want = clib.decode_attention(O.bf16_bits(case["q"]), kq, vq, ks[..., 0], vs[..., 0], case["sinks"], np.full(B, pos, np.int32), None,
                                     H**-0.5, 0, fp8_format=2)
        U.assert_close(U.to_np(got), want, what=f"e5m2 shares pos={pos}")


# windows that begin at every offset from a tile and from 16 bytes of scales, at the end of caches whose length is and is not a
# multiple of 4; windows that are and are not whole tiles, one chunked
@pytest.mark.parametrize("S,sw", [(520, 128), (517, 128), (520, 100), (519, 33), (520, 1), (904, 300)])
@pytest.mark.parametrize("fp8", [True, False])
def test_windows_at_every_offset(S, sw, fp8):
    from lyra_amd.kernels.decode_attention import decode_attention

    print(f"attention window S={S} sw={sw} fp8={fp8}", file=sys.stderr, flush=True)
    B, N, K, H = 40, 8, 2, 64
    case = U.attention_case(S + sw, B, N, K, S, H, fp8=fp8)
    q, k, v, sinks = U.attention_torch_inputs(case)
    first = np.concatenate([np.arange(S - 36, S), [0, 1, sw - 1, sw]]).astype(np.int32)
    got = decode_attention(q, k, v, sinks, H**-0.5, sw, torch.from_numpy(first).to(U.dev()), implementation="pallas")
    want = O.decode_attention_reference(case["q"], case["k"], case["v"], case["sinks"], H**-0.5, sw, first)
    U.assert_close(U.to_np(got), want, what="windows")
    for i in (0, 5, 34, 35):  # (one position for the batch: the same launch as a step's)
        one = decode_attention(q, k, v, sinks, H**-0.5, sw, torch.tensor(int(first[i]), dtype=torch.int32, device=U.dev()), implementation="pallas")
        assert torch.equal(one[i], got[i])


# a window's sums are those of a global layer over the keys from the last multiple of 32 before it, bit for bit: the order of its
# sums does not move with the position inside a tile
@pytest.mark.parametrize("pos", [127, 128, 140, 158, 159, 160, 299])
def test_window_adds_in_the_order_of_tiles_at_multiples_of_32(pos):
    from lyra_amd.kernels.decode_attention import decode_attention

    print(f"attention window tiles pos={pos}", file=sys.stderr, flush=True)
    B, N, K, S, H, sw = 64, 8, 4, 300, 64, 128
    gen = torch.Generator(device=U.dev()).manual_seed(pos)
    q, k, v = (torch.randn(*s, device=U.dev(), generator=gen).to(torch.bfloat16) for s in ((B, N, 1, H), (B, K, S, H), (B, K, S, H)))
    sinks = torch.randn(N, device=U.dev(), generator=gen)
    q[..., 0], k[..., 0] = 1.0, 0.0
    at = lambda p: torch.tensor(p, dtype=torch.int32, device=U.dev())  # noqa: E731
    got = decode_attention(q, k, v, sinks, H**-0.5, sw, at(pos), implementation="pallas")
    lo = max(0, pos - sw + 1)
    a = lo // 32 * 32
    kk, vv = k[:, :, a : pos + 1].contiguous(), v[:, :, a : pos + 1].contiguous()
    kk[:, :, : lo - a] = 0.0
    kk[:, :, : lo - a, 0] = -30000.0  # (exp2 of it is exactly zero: these keys add nothing, in their place)
    want = decode_attention(q, kk, vv, sinks, H**-0.5, 0, at(pos - a), implementation="pallas")
    assert torch.equal(got, want)


# up to 15 rows a short cache is cut into chunks whatever its format (from 16 rows on, one of FP8 this short stays whole): codes
# with unit scales and the same numbers in bf16 then give the same bits.  (Small whole numbers in q and k: exact in any order.)
@pytest.mark.parametrize("B,K,S", [(1, 4, 300), (2, 4, 300), (3, 4, 300), (3, 8, 300), (1, 1, 330), (4, 4, 300), (15, 4, 300)])
def test_few_rows_keep_their_chunks(B, K, S):
    from lyra_amd.kernels.decode_attention import decode_attention
    from lyra_amd.nn.quant import QArray

    print(f"attention few rows B={B} K={K} S={S}", file=sys.stderr, flush=True)
    H, gen = 128, torch.Generator(device=U.dev()).manual_seed(B + K)
    q = torch.randint(-3, 4, (B, 4 * K, 1, H), device=U.dev(), generator=gen).to(torch.bfloat16)
    k = torch.randint(-3, 4, (B, K, S, H), device=U.dev(), generator=gen).float().to(torch.float8_e4m3fn)
    v = torch.randn(B, K, S, H, device=U.dev(), generator=gen).to(torch.float8_e4m3fn)
    one = torch.ones(B, K, S, 1, device=U.dev())
    sinks = torch.randn(4 * K, device=U.dev(), generator=gen)
    for pos in (S - 1, S // 2):
        at = torch.tensor(pos, dtype=torch.int32, device=U.dev())
        codes = decode_attention(q, QArray(k, one, (1, H)), QArray(v, one, (1, H)), sinks, H**-0.5, 0, at, implementation="pallas")
        plain = decode_attention(q, k.to(torch.bfloat16), v.to(torch.bfloat16), sinks, H**-0.5, 0, at, implementation="pallas")
        assert torch.equal(codes, plain)
