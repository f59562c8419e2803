"""The blocks-along-K Q4_1 ring at the sizes where its plan changes: every
tile shape with ragged edges, whole and split over K, with whole and short last
stages, K splits whose last one is longer, row counts just past the skinny
kernel, the output pass over the splits' partials (plain and gated), and calls
without a workspace. plan_cases.py has the shapes whose tile counts, held to the
plan by test_plan.py.

Bar: the Q4_1 tolerance (2e-3, normalized), against the oracle with weights
decoded to f16 (the decode's rounding, 2^-12 of a weight, is in both; an f32
sum of K <= 14336 terms in any order adds 2^-24 sqrt(K) of the rms and an f16
destination one rounding, 2^-11 of the value)."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
import datagen as dg
import nnops_amd as na
from nnops_amd import ops
import plan_cases as pc
from gpu_util import dev, host, announce, norm_err, oracle_rows
from test_plan import q41_plan, L

pytestmark = pytest.mark.gpu

TOL = 2e-3

# (M, K, N): the tile and the K splits that the plan takes
SHAPES = [
    (3, 320, 100),          # 32 x 128, fewer rows than a tile, K % 256 != 0
    (5, 32, 40),            # 32 x 128, one block of k in all
    (48, 1696, 1000),       # 32 x 128 in 6, half a stage last
    (300, 4128, 260),       # the same in 8
    (1000, 96, 14080),      # 256 x 256
    (17, 256, 130),         # 32 x 128, unsplit (4 stages of k)
    (31, 4160, 1025),       # 32 x 128, 65 stages over 16 splits
    (33, 4096, 260),        # 32 x 128 in 16, one row past a tile
    (77, 4096, 1024),       # 32 x 128 in 8
    (77, 4096, 4096),       # 96 x 128 in 8
    (97, 1088, 516),        # 32 x 128, 17 stages over 4 splits, four tiles of rows
    (128, 14336, 256),      # 32 x 128 in 16
    (130, 512, 8192),       # 64 x 128
    (300, 4096, 300),       # 32 x 128 in 8
    (260, 256, 28700),      # 96 x 128
]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("out_f16", [True, False])
def test_q4_1_ring_shapes(M, K, N, out_f16):
    import torch
    announce(f"q4_1 ring {M}x{K}x{N} f16={out_f16}")
    x = dg.normal(M + K, (M, K)).astype(np.float16)
    blk = dg.q4_1_blocks(N + K, N, K)
    c = torch.full((M, N + 8), 7.0, dtype=torch.float16 if out_f16 else torch.float32, device="cuda")
    na.gemm_q4_1(dev(x), dev(blk), c[:, :N], n=N, trans_b=True)
    got = host(c).astype(np.float32)
    assert (got[:, N:] == 7.0).all()
    want = oracle_rows(lambda r0, r1: oracle.gemm_q4_1(x, blk, N, trans_b=True, rows=(r0, r1),
                                                       w_round_f16=True)[r0:r1], M, band=4)
    assert norm_err(got[:, :N], want) <= TOL


# (the partials of a split do not depend on the destination's type)
@pytest.mark.parametrize("M,K,N,want,splits,out_f16",
                         [(*c, f16) for c in pc.Q41_TILES for f16 in ((True, False) if c[4] == 1 else (True,))])
def test_q4_1_ring_tiles(M, K, N, want, splits, out_f16):
    import torch
    announce(f"q4_1 ring tile {M}x{K}x{N} f16={out_f16}")
    p = q41_plan(M, K, N)
    assert (p.tile_m, p.tile_n) == want and p.splits == splits
    x = dg.normal(M + K, (M, K)).astype(np.float16)
    blk = dg.q4_1_blocks(N + K, N, K)
    c = torch.zeros((M, N), dtype=torch.float16 if out_f16 else torch.float32, device="cuda")
    na.gemm_q4_1(dev(x), dev(blk), c, n=N, trans_b=True)
    rows = pc.edge_rows(M, p.tile_m, 101)
    xr = np.ascontiguousarray(x[rows])
    want_rows = oracle_rows(lambda r0, r1: oracle.gemm_q4_1(xr, blk, N, trans_b=True, rows=(r0, r1),
                                                            w_round_f16=True)[r0:r1], len(rows), band=4)
    assert norm_err(host(c)[rows].astype(np.float32), want_rows) <= TOL


@pytest.mark.parametrize("M,K,N2", [(17, 4096, 520), (40, 4096, 2050), (128, 2048, 1032), (200, 4096, 516)])
@pytest.mark.parametrize("kw", [dict(gated=True), dict(gated=True, add_to=True), dict(act=na.EP_RELU),
                                dict(add_to=True, residual_pre_activation=True)])
@pytest.mark.parametrize("f16", [True, False])
def test_q4_1_ring_split_pass(M, K, N2, kw, f16):
    """Linear with a bias: the splits' partials through the output pass (an
    f32 X takes its own route to the same pass)."""
    import torch
    announce(f"q4_1 split pass {M}x{K}x{N2} {kw} f16={f16}")
    dt = np.float16 if f16 else np.float32
    gated = kw.get("gated", False)
    n = N2 // 2 if gated else N2
    x = dg.normal(M, (M, K)).astype(dt)
    blk = dg.q4_1_blocks(N2 + 3, N2, K)
    bias = (0.1 * dg.normal(N2, (N2,))).astype(dt)
    old = dg.normal(4, (M, n)).astype(dt)
    y = dev(old)
    op = na.Linear(gate_activation=na.EP_SILU, output_dtype=na.DT_F16 if f16 else na.DT_F32, **kw)
    rc = op.compute([na.tensor(y)], [na.tensor(dev(x)), na.tensor(dev(blk), dtype=na.DT_Q4_1, shape=[N2, K]),
                                     na.tensor(dev(bias))])
    assert rc == na.OK
    torch.cuda.synchronize()
    want = oracle_rows(lambda r0, r1: oracle.q4_1_linear(
        x, blk, N2, rows=(r0, r1), w_round_f16=f16 or M > 48, gated=gated, out_f16=f16, bias=bias,
        out=old if kw.get("add_to") else None, gate_act=oracle.ACT_SILU,
        act=oracle.ACT_RELU if kw.get("act") else oracle.ACT_NONE, add_to=kw.get("add_to", False),
        residual_pre=kw.get("residual_pre_activation", False)), M, band=4).astype(np.float32)
    assert norm_err(host(y).astype(np.float32), want) <= TOL


@pytest.mark.parametrize("M", [3, 24, 100])
def test_q4_1_ring_without_workspace(M):
    """No workspace (none was needed before K was split): the unsplit kernels."""
    import torch
    announce(f"q4_1 no workspace M={M}")
    K, N = 4096, 384
    x = dg.normal(M, (M, K)).astype(np.float16)
    blk = dg.q4_1_blocks(11, N, K)
    dx, db = dev(x), dev(blk)
    c = torch.zeros((M, N), dtype=torch.float16, device="cuda")
    g = na.GemmQ41Args()
    g.a, g.b, g.c, g.m, g.n, g.k = dx.data_ptr(), db.data_ptr(), c.data_ptr(), M, N, K
    g.lda, g.ldc, g.ldb_bytes, g.trans_b, g.a_f16, g.out_kind = K, N, db.stride(0), 1, 1, na.OUT_F16
    assert na.lib().nnops_hip_gemm_q4_1(C.byref(g), None, 0, ops._stream_ptr(None)) == na.OK
    want = oracle.gemm_q4_1(x, blk, N, trans_b=True, w_round_f16=True)
    assert norm_err(host(c).astype(np.float32), want) <= TOL


@pytest.mark.parametrize("M,K,n,want", pc.Q41_GATED)
@pytest.mark.parametrize("kw", [dict(), dict(gate_limit=1.5), dict(add_to=True)])
@pytest.mark.parametrize("f16", [True, False])
def test_q4_1_gated_tiles(M, K, n, want, kw, f16):
    """The fused gated form on its 128- and 256-row tiles (ragged rows and
    columns, the plain SwiGLU and the general combine), bit for bit the product
    and then the pass."""
    import torch
    announce(f"q4_1 gated {M}x{K}x{n} {kw} f16={f16}")
    plan = q41_plan(M, K, 2 * n, L.PLAN_GATED_PASS)
    assert (plan.tile_m, plan.tile_n) == want and plan.fused
    x, blk = dev(dg.normal(M, (M, K)).astype(np.float16)), dev(dg.q4_1_blocks(n, 2 * n, K))
    tdt = torch.float16 if f16 else torch.float32
    bias = (0.1 * torch.randn(2 * n, device="cuda")).to(tdt)
    old = torch.randn((M, n), device="cuda").to(tdt)
    prod = torch.zeros((M, 2 * n), dtype=torch.float32, device="cuda")
    lib, st = na.lib(), ops._stream_ptr(None)
    g = na.GemmQ41Args()
    g.a, g.b, g.c, g.m, g.n, g.k = x.data_ptr(), blk.data_ptr(), prod.data_ptr(), M, 2 * n, K
    g.lda, g.ldc, g.ldb_bytes, g.trans_b, g.a_f16, g.out_kind = K, 2 * n, blk.stride(0), 1, 1, na.OUT_F32
    outs = []
    for fused in (True, False):
        y = old.clone()
        p = na._lib.FpOutArgs()
        p.src, p.ld_src, p.out, p.ld_out, p.rows, p.n = prod.data_ptr(), 2 * n, y.data_ptr(), n, M, n
        p.out_f16, p.bias, p.gated, p.gate_act, p.gate_alpha = int(f16), bias.data_ptr(), 1, na.ACT_SILU, 1.0
        p.min_clip, p.max_clip, p.act_beta = -np.inf, np.inf, 1.0
        p.gate_limit, p.add_to = kw.get("gate_limit", np.inf), int(kw.get("add_to", False))
        if fused:
            assert lib.nnops_hip_gemm_q4_1_fused(C.byref(g), C.byref(p), st) == na.OK
        else:
            # unsplit (no workspace): the fused tiles sum K in the same order
            assert lib.nnops_hip_gemm_q4_1(C.byref(g), None, 0, st) == na.OK
            assert lib.nnops_hip_fp_output_pass(C.byref(p), st) == na.OK
        outs.append(host(y))
    assert np.array_equal(outs[0].view(np.uint8), outs[1].view(np.uint8))


@pytest.mark.parametrize("K", [4224, 8192, 8320, 11008, 16384])
@pytest.mark.parametrize("M,N", [(1, 37), (2, 130)])
@pytest.mark.parametrize("out_f16", [True, False])
def test_q4_1_gemv_long_rows(K, M, N, out_f16):
    """GEMV rows past 128 blocks, K over two or four waves: the shortest and
    longest rows of each, the last part shorter, ragged N. The pitch is wider
    than the row; the weights of the padding would show up as huge values."""
    import torch
    announce(f"q4_1 gemv parts {M}x{K}x{N} f16={out_f16}")
    x = dg.normal(M + K, (M, K)).astype(np.float16)
    blk = dg.q4_1_blocks(N + K, N, K)
    wide = np.full((N, blk.shape[1] + 48), 0x7b, np.uint8)
    wide[:, :blk.shape[1]] = blk
    c = torch.zeros((M, N), dtype=torch.float16 if out_f16 else torch.float32, device="cuda")
    na.gemm_q4_1(dev(x), dev(wide), c, n=N, trans_b=True)
    want = oracle.gemm_q4_1(x, blk, N, trans_b=True)
    assert norm_err(host(c).astype(np.float32), want) <= TOL


@pytest.mark.parametrize("M,K,N", [(3, 14336, 100), (16, 11008, 516), (7, 6144, 1000), (5, 3072, 32)])
@pytest.mark.parametrize("bias", [False, True])
def test_q4_1_skinny_splits(M, K, N, bias):
    """Up to 16 rows over a long K: the skinny kernel's K splits (one longer
    than the others), summed by the store pass or the bias pass."""
    import torch
    announce(f"q4_1 skinny split {M}x{K}x{N} bias={bias}")
    x = dg.normal(M + K, (M, K)).astype(np.float16)
    blk = dg.q4_1_blocks(N + K, N, K)
    b = dg.normal(1, (N,)).astype(np.float16)
    y = torch.zeros((M, N), dtype=torch.float16, device="cuda")
    ins = [na.tensor(dev(x)), na.tensor(dev(blk), dtype=na.DT_Q4_1, shape=[N, K])] + ([na.tensor(dev(b))] if bias else [])
    assert na.Linear(output_dtype=na.DT_F16).compute([na.tensor(y)], ins) == na.OK
    want = oracle.q4_1_linear(x, blk, N, w_round_f16=True, out_f16=True, bias=b if bias else None).astype(np.float32)
    assert norm_err(host(y).astype(np.float32), want) <= TOL


@pytest.mark.parametrize("lda", [8388608, 16777216])
@pytest.mark.parametrize("gated", [True, False])
def test_q4_1_wide_row_pitch(lda, gated):
    """Rows of A millions of elements apart (the last token of many sequences,
    as a slice): the same bits as from packed rows, which the same sums over K
    give on any unsplit tile. 256-row tiles would pass 2^31 here."""
    import torch
    M, K, N = 300, 512, 28672
    announce(f"q4_1 row pitch {lda} gated={gated}")
    x, blk = dev(dg.normal(M, (M, K)).astype(np.float16)), dev(dg.q4_1_blocks(N, N, K))
    wide = torch.empty(M * lda, dtype=torch.float16, device="cuda").view(M, lda)[:, :K]
    wide.copy_(x)
    outs = []
    for a in (x, wide):
        y = torch.zeros((M, N // 2 if gated else N), dtype=torch.float16, device="cuda")
        op = na.Linear(output_dtype=na.DT_F16, gated=gated, gate_activation=na.EP_SILU if gated else na.EP_NONE)
        assert op.compute([na.tensor(y)], [na.tensor(a), na.tensor(blk, dtype=na.DT_Q4_1, shape=[N, K])]) == na.OK
        outs.append(host(y))
    assert np.abs(outs[0][-1].astype(np.float32)).max() > 0
    assert np.array_equal(outs[0].view(np.uint8), outs[1].view(np.uint8))


@pytest.mark.parametrize("M,K,N", [(20, 96, 40), (20, 320, 40), (130, 4128, 260), (300, 416, 1000)])
@pytest.mark.parametrize("gated", [False, True])
def test_q4_1_weight_at_the_end_of_its_buffer(M, K, N, gated):
    """A weight that is the right part of a wider buffer: its last row ends
    where the allocation does, less than a stage's bytes past its last block.
    The same bits as from the packed weight."""
    import torch
    announce(f"q4_1 end of buffer {M}x{K}x{N} gated={gated}")
    x, blk = dev(dg.normal(M, (M, K)).astype(np.float16)), dev(dg.q4_1_blocks(N, N, K))
    wide = torch.full((N, 48 + blk.shape[1]), 0x7b, dtype=torch.uint8, device="cuda")[:, 48:]
    wide.copy_(blk)
    outs = []
    for w in (blk, wide):
        y = torch.zeros((M, N // 2 if gated else N), dtype=torch.float16, device="cuda")
        op = na.Linear(output_dtype=na.DT_F16, gated=gated, gate_activation=na.EP_SILU)
        assert op.compute([na.tensor(y)], [na.tensor(x), na.tensor(w, dtype=na.DT_Q4_1, shape=[N, K])]) == na.OK
        outs.append(host(y))
    assert np.abs(outs[0].astype(np.float32)).max() > 0
    assert np.array_equal(outs[0].view(np.uint8), outs[1].view(np.uint8))


@pytest.mark.parametrize("M,N", [(17, 4096), (512, 28672)])
def test_q4_1_gated_linear_timed(M, N):
    """Armed timing events reach the operator's first launch, on the route
    whose partials the pass sums (17 rows) and on the fused tiles."""
    import torch
    announce(f"q4_1 timed gated M={M}")
    K = 1024
    x, blk = dev(dg.normal(M, (M, K)).astype(np.float16)), dev(dg.q4_1_blocks(N, N, K))
    y = torch.zeros((M, N // 2), dtype=torch.float16, device="cuda")
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e1.record()          # in this order their own span is not positive
    e0.record()
    torch.cuda.synchronize()
    assert na.lib().nnops_hip_time_next_launch(C.c_void_p(e0.cuda_event), C.c_void_p(e1.cuda_event)) == na.OK
    op = na.Linear(output_dtype=na.DT_F16, gated=True, gate_activation=na.EP_SILU)
    assert op.compute([na.tensor(y)], [na.tensor(x), na.tensor(blk, dtype=na.DT_Q4_1, shape=[N, K])]) == na.OK
    torch.cuda.synchronize()
    assert e0.elapsed_time(e1) > 0.0
