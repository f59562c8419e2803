"""The kernel selection of the ring GEMMs (nnops_hip_gemm_*_plan), on the host:
no call here reaches a kernel launch."""
from __future__ import annotations

import ctypes as C

import pytest

import nnops_amd as na
from nnops_amd import _lib as L
import plan_cases as pc

ALL = 1 << 62       # a workspace with room for any plan


def q41_plan(M, K, N, pass_=L.PLAN_NO_PASS, ws=ALL, lda=None, ldb=None, a=0):
    g = na.GemmQ41Args()
    g.a, g.m, g.n, g.k = a, M, N, K
    g.lda, g.ldc, g.ldb_bytes = lda or K, N, ldb or (K + 31) // 32 * 20
    g.trans_b, g.a_f16, g.out_kind = 1, 1, na.OUT_F16
    p = L.GemmPlan()
    assert na.lib().nnops_hip_gemm_q4_1_plan(C.byref(g), pass_, ws, C.byref(p)) == na.OK
    return p


def i8_plan(M, K, N, ws=ALL, trans_b=True, ldb=None, ldc=None, b=0, **fields):
    g = na.GemmI8Args()
    g.b, g.m, g.n, g.k = b, M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b = K, ldb or (K if trans_b else N), ldc or N, int(trans_b)
    g.out_kind, g.s_a_scalar, g.s_b_scalar, g.s_out = na.OUT_S8, 1.0, 1.0, 1.0
    g.min_clip, g.max_clip = -float("inf"), float("inf")
    for k, v in fields.items():
        setattr(g, k, v)
    p = L.GemmPlan()
    assert na.lib().nnops_hip_gemm_i8_plan(C.byref(g), ws, C.byref(p)) == na.OK
    return p


def f16_plan(M, K, N, ws=ALL, trans_b=True, c=0):
    g = na.GemmFpArgs()
    g.c, g.m, g.n, g.k = c, M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b, g.in_f16, g.out_f16, g.alpha = K, K if trans_b else N, N, int(trans_b), 1, 1, 1.0
    p = L.GemmPlan()
    assert na.lib().nnops_hip_gemm_fp_plan(C.byref(g), ws, C.byref(p)) == na.OK
    return p


# pitches of the last token of M sequences, 4096 wide: up to 4096 tokens each
@pytest.mark.parametrize("lda", [4096, 4194304, 4227136, 8388608, 8454144, 16777216, 33554432, 134217728])
@pytest.mark.parametrize("M", [17, 130, 300, 512])
@pytest.mark.parametrize("N,pass_", [(4096, L.PLAN_NO_PASS), (28672, L.PLAN_PASS), (28672, L.PLAN_GATED_PASS)])
def test_q4_1_row_pitch(lda, M, N, pass_):
    """Every offset of the planned tile's rows of A stays below 2^31 (the
    kernel forms them in 32 bits): a wide pitch takes lower tiles, and past
    the lowest one another kernel."""
    p = q41_plan(M, 4096, N, pass_, lda=lda)
    if p.tile_m:
        assert (min(p.tile_m, M) - 1) * lda * 2 + 4096 * 2 < 2**31
    assert p.tile_m or lda > 16777216


def test_q4_1_row_pitch_keeps_the_tall_tile():
    """512 rows of a gated product: the 256-row tiles where their offsets fit,
    else the 128-row ones."""
    tiles = [q41_plan(512, 4096, 28672, L.PLAN_GATED_PASS, lda=lda) for lda in (4096, 4194304, 8388608)]
    assert [t.tile_m for t in tiles] == [256, 256, 128]
    assert all(t.fused for t in tiles)


@pytest.mark.parametrize("ldb", [2560, 8388608, 16777216, 134217728])
def test_q4_1_weight_pitch(ldb):
    p = q41_plan(300, 4096, 300, ldb=ldb)
    assert p.tile_m == 0 or (min(p.tile_n, 300) - 1) * ldb + 2560 < 2**31


NOALLOC = 64 << 20


@pytest.mark.parametrize("M", [77, 104, 128])
@pytest.mark.parametrize("fields", [dict(a_u8=1), dict(zp_a_scalar=3), dict(a_u8=1, out_kind=na.OUT_S32)])
def test_i8_splits_within_the_fixed_scratch(M, fields):
    """A transposed copy that nearly fills the library's own 64 MiB: K splits
    as far as the rest holds, where the full plan's partials do not fit."""
    full, p = (i8_plan(M, 14336, 4096, ws, trans_b=False, **fields) for ws in (ALL, NOALLOC))
    assert full.workspace_bytes > NOALLOC
    assert p.tile_m > 0 and p.splits >= 2 and p.workspace_bytes <= NOALLOC


@pytest.mark.parametrize("M", [24, 64, 128, 300, 512])
@pytest.mark.parametrize("out", [na.OUT_S8, na.OUT_S32])
def test_i8_splits_grow_with_the_workspace(M, out):
    """Plans for less and less room fit into it, down to an unsplit one."""
    full = i8_plan(M, 14336, 1024, out_kind=out)
    assert full.splits > 1
    seen = set()
    for slabs in range(full.splits, 0, -1):
        room = full.workspace_bytes - (full.splits - slabs) * M * 1024 * 4
        p = i8_plan(M, 14336, 1024, room, out_kind=out)
        assert p.tile_m > 0 and p.workspace_bytes <= room and p.splits <= slabs
        seen.add(p.splits)
    assert full.splits in seen and 1 in seen


# A call whose workspace is too small is refused before any launch: the
# pointers are never followed.
FAR = 1 << 20


def i8_call(ws, M, K, N, **fields):
    g = na.GemmI8Args()
    g.a, g.b, g.c, g.m, g.n, g.k = FAR, FAR, FAR, M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b, g.out_kind = K, K, N, 1, na.OUT_S8
    g.s_a_scalar = g.s_b_scalar = g.s_out = 1.0
    for k, v in fields.items():
        setattr(g, k, v)
    return g, na.lib().nnops_hip_gemm_i8(C.byref(g), FAR, ws, None)


@pytest.mark.parametrize("M,K,N", [(64, 4096, 4096), (128, 14336, 1024), (333, 14336, 4096), (512, 8192, 1024)])
@pytest.mark.parametrize("fields", [dict(), dict(s_a=FAR), dict(trans_b=0, ldb=4096)])
def test_i8_refuses_a_small_workspace(M, K, N, fields):
    """Between the sums' room and what the splits of the rows' tile take."""
    p = i8_plan(M, K, N, **fields)
    assert p.splits > 1
    sums = (M * 4 + 255) // 256 * 256 + (N * 4 + 255) // 256 * 256
    for ws in (0, sums, sums + M * N * 4):
        assert i8_call(ws, M, K, N, **fields)[1] == na.NOT_INITIALIZED


@pytest.mark.parametrize("M,K,N", [(64, 4096, 4096), (333, 8192, 4096), (512, 14336, 1024)])
def test_f16_refuses_a_small_workspace(M, K, N):
    g = na.GemmFpArgs()
    g.a, g.b, g.c, g.m, g.n, g.k = FAR, FAR, FAR, M, N, K
    g.lda, g.ldb, g.ldc, g.trans_b, g.in_f16, g.out_f16, g.alpha = K, K, N, 1, 1, 1, 1.0
    need = na.lib().nnops_hip_gemm_fp_workspace_size(C.byref(g))
    assert need >= M * N * 4
    for ws in (0, M * N * 4 - 1):
        assert na.lib().nnops_hip_gemm_fp(C.byref(g), FAR, ws, None) == na.NOT_INITIALIZED


@pytest.mark.parametrize("M,K,N,ring", [
    (2, 4096, 4096, False), (3, 512, 1000, False), (4, 1024, 4096, False), (3, 1776, 8192, False), (4, 1792, 4096, True),
    (3, 1536, 14336, True), (4, 4096, 4096, True), (3, 8192, 8192, True), (4, 8192, 14336, False),
    (5, 512, 1024, True), (5, 512, 100, False), (8, 768, 1001, False), (9, 768, 1001, True), (8, 4096, 1001, True)])
def test_f16_few_rows(M, K, N, ring):
    """Where the GEMV is the faster, a call of few rows does not take the ring."""
    assert (f16_plan(M, K, N).tile_m > 0) == ring


@pytest.mark.parametrize("M,K,N,kind,ring", [
    (17, 256, 1024, na.OUT_S8, False), (63, 384, 4096, na.OUT_S32, False), (17, 448, 4096, na.OUT_S8, True),
    (48, 960, 1024, na.OUT_S8, False), (48, 1024, 1024, na.OUT_S8, True), (64, 256, 1024, na.OUT_S8, True),
    (17, 256, 1024, na.OUT_F16, True), (17, 256, 1024, na.OUT_F32, True)])
def test_i8_few_rows_short_k(M, K, N, kind, ring):
    """Where gemm_i8_mfma is the faster, few rows do not take the ring; over a
    [K,N] B, which it would have to copy, they do."""
    assert (i8_plan(M, K, N, out_kind=kind).tile_m > 0) == ring
    assert i8_plan(M, K, N, out_kind=kind, trans_b=False).in_place


def tile(p):
    return p.tile_m, p.tile_n


@pytest.mark.parametrize("M,K,N,nk,kn", pc.I8_TILES)
def test_i8_tile_cases(M, K, N, nk, kn):
    """The GPU tests' shapes take the tiles that they are there for, with every
    destination that is fused and through partials (a scale per row)."""
    for trans_b, want in ((True, nk), (False, kn)):
        for fields in (dict(), dict(out_kind=na.OUT_S32), dict(out_kind=na.OUT_F16), dict(s_a=FAR)):
            p = i8_plan(M, K, N, trans_b=trans_b, **fields)
            assert tile(p) == want and p.in_place == (not trans_b) and p.fused == ("s_a" not in fields)


@pytest.mark.parametrize("M,K,N,tile_m", pc.I8_IN_PLACE_ODD)
def test_i8_in_place_odd_cases(M, K, N, tile_m):
    p = i8_plan(M, K, N, trans_b=False, ldb=(N + 15) // 16 * 16, out_kind=na.OUT_S32)
    assert p.in_place and p.tile_m == tile_m


@pytest.mark.parametrize("M,K,N,want", pc.F16_TILES)
def test_f16_tile_cases(M, K, N, want):
    for trans_b in (True, False):
        p = f16_plan(M, K, N, trans_b=trans_b)
        assert tile(p) == want and p.fused == (N % 8 == 0)


@pytest.mark.parametrize("M,K,N,want,splits", pc.Q41_TILES)
def test_q4_1_tile_cases(M, K, N, want, splits):
    p = q41_plan(M, K, N)
    assert tile(p) == want and p.splits == splits and p.fused == (splits == 1)


@pytest.mark.parametrize("M,K,n,want", pc.Q41_GATED)
def test_q4_1_gated_cases(M, K, n, want):
    p = q41_plan(M, K, 2 * n, L.PLAN_GATED_PASS)
    assert tile(p) == want and p.fused


def test_every_tile_has_its_cases():
    """Nine int8 and f16 tiles (seven of them in place over a [K,N] B), seven
    Q4_1 ones and two gated ones, each with whole stages and a short last one."""
    def forms(cases, k_stage, i):
        return {(c[i], c[1] % k_stage != 0) for c in cases}
    assert len(forms(pc.I8_TILES, 128, 3)) == len(forms(pc.F16_TILES, 64, 3)) == 18
    assert len(forms(pc.I8_TILES, 128, 4)) == 14
    assert len({(c[3], c[4] > 1, c[1] % 64 != 0) for c in pc.Q41_TILES}) == 26
    assert len(forms(pc.Q41_GATED, 64, 3)) == 4


@pytest.mark.parametrize("M,K,N,trans_b,want,splits", [
    (907, 1344, 9680, False, (256, 256), 1),        # 21 us; two rounds of 192 x 128 33
    (1551, 1024, 5904, False, (256, 256), 1),       # 18; 25
    (858, 6144, 11008, False, (256, 256), 1),       # 75; 86
    (218, 14336, 4240, True, (256, 128), 7),        # 31; 41 in 5 splits of 128 x 192
    (97, 11008, 1232, True, (64, 64), 6)])          # 12.5; 15.2 in 12 splits of 128 x 64
def test_i8_cheapest(M, K, N, trans_b, want, splits):
    """Shapes that an estimate without the CUs' fill, the [K,N] steps and the
    reduce of many splits had given slower tiles."""
    p = i8_plan(M, K, N, trans_b=trans_b)
    assert tile(p) == want and p.splits == splits


@pytest.mark.parametrize("M,K,N,splits", [(997, 13056, 4608, 3), (414, 14336, 10096, 3), (929, 7616, 4944, 3)])
def test_f16_splits_past_32_mib(M, K, N, splits):
    """Partials of up to 64 MiB where they are the faster: 126 us in 3 splits
    against 158 unsplit, 159 against 192 in 2, 83 against 108 unsplit."""
    p = f16_plan(M, K, N)
    assert tile(p) == (256, 256) and p.splits == splits and p.workspace_bytes <= 64 << 20


@pytest.mark.parametrize("M,K,n", [(593, 11008, 4592), (593, 11008, 4593), (700, 11008, 3300), (384, 4096, 8192)])
def test_q4_1_gated_tiles_past_half_the_cus(M, K, n):
    """The fused tiles where they fill most of one round: 160 us against 178 in K
    splits and a pass (593 rows)."""
    p = q41_plan(M, K, 2 * n, L.PLAN_GATED_PASS)
    assert p.fused and p.tile_m
