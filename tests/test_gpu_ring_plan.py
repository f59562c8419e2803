"""The LDS-ring GEMM at the sizes where its plan changes: every tile shape with
whole and short last stages of k, ragged last tiles in both directions, the
smallest row counts that take it, K splits, and a workspace too small for the
splits. plan_cases.py has the shapes whose tile counts, held to the plan by
test_plan.py.

int8: bit-exact against the oracle. f16: the normalized error of one f16
rounding (2^-11 of the value) and of an f32 sum over K <= 11008 terms in any
order (2^-24 sqrt(K) of the rms, far below it): 2e-3, as in test_gpu_fp."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
import datagen as dg
import nnops_amd as na
from nnops_amd import ops
from gpu_util import dev, host, announce, norm_err, oracle_rows, pitched
import plan_cases as pc
from test_plan import i8_plan, f16_plan

pytestmark = pytest.mark.gpu

# (M, K, N). An odd width of a packed [K,N] weight is copied, not read in place.
SHAPES = [
    (17, 704, 68),          # gemm_i8_mfma
    (63, 8192, 132),        # 64 x 64, 16 K splits
    (65, 4096, 260),        # 64 x 64, 8 splits, one row past a tile
    (500, 256, 4000),       # 128 x 64
    (130, 4160, 1028),      # 64 x 64, 5 splits, the last stage half as deep
    (20, 32, 36),           # gemm_i8_mfma, one slice of k in all
    (65, 4128, 260),        # 32 k in the last stage, 8 splits
    (333, 1120, 1024),      # 96 k in the last stage
    (40, 8160, 257),        # 16 splits, N % 4 == 1
    (200, 288, 4003),       # N % 4 == 3
    (1000, 96, 16130),      # N % 4 == 2, 256 x 256, a short stage only
    (500, 256, 4100),       # 128 x 128, last tile 4 columns wide, f16 through partials
    (300, 2048, 1024),      # 64 x 64, partials in 3 splits
    (384, 256, 16000),      # 192 x 128
    (500, 128, 16100),      # 256 x 128, one stage, through partials
    (640, 128, 11776),      # 128 x 256, one stage
    (500, 128, 11004),      # 128 x 192, one stage, through partials
    (1000, 96, 11008),      # 256 x 192 (256 x 256 over a [K,N] B), a short stage only
    (1000, 128, 16132),     # 256 x 256, one stage, through partials
]


def run_i8(M, K, N, trans_b, out, rows):
    """One call against the oracle at the given rows (a row's result depends on
    that row only). s8: the fused requant; s8_tokens: with a scale per row,
    partials and the reduce; f16: the fused dequantizing output."""
    seed = M + K + N
    a = dg.act_s8(seed, (M, K))
    w = dg.ints(seed + 1, (N, K), -127, 127)
    sb = dg.uniform(seed + 2, (N,), 0.001, 0.01)
    kind, okind, dt = {"f16": (na.OUT_F16, oracle.OUT_F16, np.float16),
                       "s32": (na.OUT_S32, oracle.OUT_S32, np.int32)}.get(out, (na.OUT_S8, oracle.OUT_S8, np.int8))
    s_a = dg.uniform(seed + 3, (M,), 0.01, 0.03) if out == "s8_tokens" else 0.02
    bias = dg.ints(seed + 4, (N,), -5000, 5000, np.int32) if out != "f16" else None
    act = (na.ACT_RELU, oracle.ACT_RELU) if out == "s8" else (na.ACT_NONE, oracle.ACT_NONE)
    c = dev(np.zeros((M, N), dt))
    b = w if trans_b else np.ascontiguousarray(w.T)
    na.gemm_i8(dev(a), dev(b), c, trans_b=trans_b, out_kind=kind, bias=None if bias is None else dev(bias),
               s_a=dev(s_a) if out == "s8_tokens" else s_a, s_b=dev(sb), s_out=0.4, act=act[0])
    got = host(c)
    for r in rows:
        want = oracle.gemm_i8(a[r:r + 1], w, trans_b=True, bias=bias, out_kind=okind,
                              s_a=s_a[r:r + 1] if out == "s8_tokens" else s_a, s_b=sb, s_out=0.4, act=act[1])
        assert np.array_equal(got[r:r + 1].view(np.uint8), want.view(np.uint8)), r


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("out", ["s8", "s8_tokens", "f16"])
def test_i8_shapes(M, K, N, trans_b, out):
    announce(f"ring i8 {M}x{K}x{N} tb={trans_b} {out}")
    run_i8(M, K, N, trans_b, out,
           sorted({r for e in (0, 64, 128, 192, 256, 384, 512, M) for r in range(e - 2, e + 2) if 0 <= r < M}))


@pytest.mark.parametrize("M,K,N,nk,kn", pc.I8_TILES)
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("out", ["s8", "s8_tokens", "s32", "f16"])
def test_i8_tiles(M, K, N, nk, kn, trans_b, out):
    announce(f"ring i8 tile {M}x{K}x{N} tb={trans_b} {out}")
    p = i8_plan(M, K, N, trans_b=trans_b)
    assert (p.tile_m, p.tile_n) == (nk if trans_b else kn)
    run_i8(M, K, N, trans_b, out, pc.edge_rows(M, p.tile_m, 41))


# [K,N] weights of odd width at a 16-byte pitch: read in place, the last k
# row's last columns in a dword that N ends inside
@pytest.mark.parametrize("M,K,N,tile_m", pc.I8_IN_PLACE_ODD)
def test_i8_in_place_odd_columns(M, K, N, tile_m):
    announce(f"ring i8 in place {M}x{K}x{N}")
    plan = i8_plan(M, K, N, trans_b=False, ldb=(N + 15) // 16 * 16, ldc=N, out_kind=na.OUT_S32)
    assert plan.in_place and plan.tile_m == tile_m, plan.tile_m
    a = dg.act_s8(M, (M, K))
    w = dg.ints(N, (N, K), -127, 127)
    b = pitched(np.ascontiguousarray(w.T), (N + 15) // 16 * 16)
    c = dev(np.zeros((M, N), np.int32))
    na.gemm_i8(dev(a), b, c, trans_b=False)
    got = host(c)
    want = oracle_rows(lambda r0, r1: oracle.gemm_i8(a[r0:r1], w, trans_b=True), M)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("M,K,N", [(18, 224, 69), (70, 4128, 132), (300, 160, 1030)])
@pytest.mark.parametrize("trans_b", [True, False])
def test_u8_zero_points_short_stage(M, K, N, trans_b):
    """u8 A (flipped in registers, not in the padding) and zero points over a
    short last stage."""
    announce(f"ring u8 {M}x{K}x{N} tb={trans_b}")
    a = dg.ints(M, (M, K), 0, 255, np.uint8)
    w = dg.ints(N, (N, K), -127, 127)
    sb = dg.uniform(3, (N,), 0.001, 0.01)
    zb = dg.ints(4, (N,), -3, 3, np.int32)
    c = dev(np.zeros((M, N), np.int8))
    na.gemm_i8(dev(a), dev(w if trans_b else np.ascontiguousarray(w.T)), c, trans_b=trans_b, out_kind=na.OUT_S8,
               s_a=0.02, zp_a=117, s_b=dev(sb), zp_b=dev(zb), s_out=0.4, zp_out=3)
    want = oracle.gemm_i8(a, w, trans_b=True, out_kind=oracle.OUT_S8, s_a=0.02, zp_a=117, s_b=sb, zp_b=zb, s_out=0.4,
                          zp_out=3)
    assert np.array_equal(host(c), want)


@pytest.mark.parametrize("M,K,N", [(3, 512, 100), (4, 1792, 260), (8, 768, 1001), (20, 48, 33), (130, 1040, 1001), (40, 8208, 78), (3, 4096, 68), (16, 96, 40), (17, 1024, 132), (40, 11008, 260), (64, 4096, 1024),
                                   (500, 128, 4000), (500, 128, 4100), (384, 128, 16000), (500, 64, 11004),
                                   (1000, 48, 11000)])
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("out_f16", [True, False])
def test_f16_shapes(M, K, N, trans_b, out_f16):
    run_f16(M, K, N, trans_b, out_f16)


@pytest.mark.parametrize("M,K,N,want", pc.F16_TILES)
@pytest.mark.parametrize("trans_b", [True, False])
@pytest.mark.parametrize("out_f16", [True, False])
def test_f16_tiles(M, K, N, want, trans_b, out_f16):
    p = f16_plan(M, K, N, trans_b=trans_b)
    assert (p.tile_m, p.tile_n) == want
    run_f16(M, K, N, trans_b, out_f16)


def run_f16(M, K, N, trans_b, out_f16):
    import torch
    announce(f"ring f16 {M}x{K}x{N} tb={trans_b} f16={out_f16}")
    a = dg.normal(M + K, (M, K)).astype(np.float16)
    w = dg.normal(N + K, (N, K)).astype(np.float16)
    c = torch.zeros((M, N), dtype=torch.float16 if out_f16 else torch.float32, device="cuda")
    na.gemm_fp(dev(a), dev(w if trans_b else np.ascontiguousarray(w.T)), c, trans_b=trans_b, alpha=0.5)
    got = host(c).astype(np.float32)
    want = 0.5 * oracle.gemm_fp(a, w)
    if out_f16:
        want = want.astype(np.float16).astype(np.float32)
    assert norm_err(got, want) <= (2e-3 if out_f16 else 2e-5)


@pytest.mark.parametrize("M", [3, 24, 40])
def test_f16_without_workspace(M):
    """Calls of fewer than 64 rows need no workspace: without one they take
    the kernels that split nothing."""
    import torch
    announce(f"f16 no workspace M={M}")
    K, N = 4096, 256
    a = dg.normal(M, (M, K)).astype(np.float16)
    w = dg.normal(5, (N, K)).astype(np.float16)
    da, dw = dev(a), dev(w)
    c = torch.zeros((M, N), dtype=torch.float16, device="cuda")
    g = na.GemmFpArgs()
    g.a, g.b, g.c, g.m, g.n, g.k = da.data_ptr(), dw.data_ptr(), c.data_ptr(), M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b, g.in_f16, g.out_f16, g.alpha = K, K, N, 1, 1, 1, 1.0
    assert na.lib().nnops_hip_gemm_fp_workspace_size(C.byref(g)) > 0
    assert na.lib().nnops_hip_gemm_fp(C.byref(g), None, 0, ops._stream_ptr(None)) == na.OK
    want = oracle.gemm_fp(a, w).astype(np.float16).astype(np.float32)
    assert norm_err(host(c).astype(np.float32), want) <= 2e-3


def test_i8_least_workspace():
    """24 rows with the row and column sums' room alone (what the call took
    before its K was split): the unsplit kernel, the same bits."""
    import torch
    announce("i8 least workspace")
    M, K, N = 24, 8192, 512
    a, w = dg.act_s8(1, (M, K)), dg.ints(2, (N, K), -127, 127)
    c = dev(np.zeros((M, N), np.int32))
    da, dw = dev(a), dev(w)
    g = na.GemmI8Args()
    g.a, g.b, g.c, g.m, g.n, g.k = da.data_ptr(), dw.data_ptr(), c.data_ptr(), M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b, g.out_kind = K, K, N, 1, na.OUT_S32
    g.s_a_scalar = g.s_b_scalar = g.s_out = 1.0
    least = 256 + (N * 4 + 255) // 256 * 256
    assert na.lib().nnops_hip_gemm_i8_workspace_size(C.byref(g)) > least
    ws = torch.empty(least, dtype=torch.uint8, device="cuda")
    assert na.lib().nnops_hip_gemm_i8(C.byref(g), ws.data_ptr(), least, ops._stream_ptr(None)) == na.OK
    assert np.array_equal(host(c), oracle.gemm_i8(a, w, trans_b=True))


@pytest.mark.parametrize("s_out", [0.031, 0.0007, 1.3])
@pytest.mark.parametrize("even", [False, True])
@pytest.mark.parametrize("clip", [False, True])
def test_gelu_requant_dense(s_out, even, clip):
    """GELU on an s8 destination over a dense range of accumulators (a bias per
    column, 70 rows of different sums): bit for bit the oracle's, so every
    value near a rounding boundary took the exact evaluation."""
    announce(f"gelu dense s_out={s_out} even={even} clip={clip}")
    M, K, N = 70, 128, 40000
    a = np.zeros((M, K), np.int8)
    a[:, 0] = np.arange(M)
    w = dg.ints(1, (N, K), -127, 127)
    bias = (np.arange(N, dtype=np.int32) - N // 2) * 7
    sb = dg.uniform(2, (N,), 0.9, 1.1).astype(np.float32)
    kw = dict(s_a=4.0e-5 * max(1.0, s_out * 10), s_out=s_out, zp_out=-3, float_ep=True, round_even=even,
              min_clip=-1.5 if clip else -np.inf, max_clip=2.0 if clip else np.inf)
    c = dev(np.zeros((M, N), np.int8))
    na.gemm_i8(dev(a), dev(w), c, trans_b=True, out_kind=na.OUT_S8, bias=dev(bias), s_b=dev(sb), act=na.ACT_GELU, **kw)
    want = oracle.gemm_i8(a, w, trans_b=True, out_kind=oracle.OUT_S8, bias=bias, s_b=sb, act=oracle.ACT_GELU, **kw)
    assert np.array_equal(host(c), want)
