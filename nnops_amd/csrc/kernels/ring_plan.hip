// Which tile and K split a call of the LDS-ring GEMM takes (host code).
#include "gemm_i8_ring.hpp"

namespace nnops_amd {
namespace {

// The ring's tile shapes and the time of one 128-byte k step of one
// workgroup, with one workgroup on every CU (the loop's time over its steps,
// at 512 x 4096 x 4096 and up, int8 and f16 operands alike: the step moves
// the same bytes and runs as many matrix-core cycles). The 192-column tiles
// (not over a [K,N] B in place) are for widths that leave 128 and 256 columns
// with a last round nearly empty: 1000 x 4096 x 11008 f16 115 -> 105 us on 232
// tiles of 256 x 192 against 172 of 256 x 256, 512 rows 67 -> 60 (s8 36 -> 33).
struct RingTile {
    int bm, bn;
    float step_us;
};
constexpr RingTile kRingTiles[] = {
    {64, 64, 0.38f},    {128, 64, 0.48f},   {128, 128, 0.68f},  {192, 128, 0.82f},
    {128, 192, 0.85f}, {256, 128, 1.08f},  {128, 256, 1.08f},  {256, 192, 1.40f}, {256, 256, 1.80f},
};

// The fused output mode a call may take (RING_PART: none): row-uniform
// parameters, no zero-point terms, half-away rounding, N % 4 == 0, 16-byte
// aligned tables and destination; everything else writes raw partials and runs
// gemm_i8_reduce.
int fused_mode(const NnopsGemmI8Args& g)
{
    const bool compensate = g.a_u8 || g.zp_a != nullptr || g.zp_a_scalar != 0 || g.zp_b != nullptr ||
                            g.zp_b_scalar != 0;
    const bool tables16 = ((uintptr_t)g.bias % 16 == 0) && ((uintptr_t)g.s_b % 16 == 0);
    const bool fp_out = g.out_kind == NNOPS_OUT_F32 || g.out_kind == NNOPS_OUT_F16;
    const bool plain = !compensate && g.s_out_rows == nullptr && g.zp_out_rows == nullptr && !g.float_ep &&
                       !g.round_even && !fp_out && tables16 && ((uintptr_t)g.c % 16 == 0);
    const size_t ebytes = g.out_kind == NNOPS_OUT_F16 ? 2 : 4;
    if (g.n % 4 != 0) {
        return RING_PART;
    }
    if (fp_out && !compensate && (g.act == NNOPS_ACT_NONE || g.act == NNOPS_ACT_RELU) && (uintptr_t)g.c % 16 == 0 &&
        (g.ldc * ebytes) % 16 == 0 && ((uintptr_t)g.s_b % 16) == 0 &&
        (g.bias_fp == nullptr || (uintptr_t)g.bias_fp % (4 * ebytes) == 0)) {
        return RING_FP;       // dequantizing output pass fused
    }
    if (plain && g.out_kind == NNOPS_OUT_S32 && (g.ldc * 4) % 16 == 0) {
        return RING_S32;
    }
    if (plain && g.out_kind != NNOPS_OUT_S32 && g.s_a == nullptr && g.ldc % 16 == 0 && g.n % 16 == 0) {
        return RING_S8;
    }
    return RING_PART;
}

}  // namespace

// One tile shape per range of rows, K split to fill the CUs (at least 512 bytes
// of k per split, none below 16 stages); small_tiles: 64 x 64 tiles where that
// gives fewer than 32 tiles. For the calls that it takes (64 rows and more, k in
// whole 64-byte steps, N % 4 == 0) it says how much workspace is enough: callers
// keep buffers of that size, and the library's own fixed one is measured by it.
RingPlan plan_ring_by_rows(const NnopsGemmI8Args& g, const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                           bool trb, bool small_tiles)
{
    RingPlan r;
    if (g.m < 64 || g.k < 64 || g.k % 64 != 0 || g.n % 4 != 0 || !aligned16(a, lda) || !aligned16(b, ldb) ||
        (trb && (g.k * ldb + g.n >= (int64_t)INT32_MAX || ldb < g.n))) {
        return r;
    }
    int bm = 256, bn = 256;
    if (g.m <= 128) {
        bm = 128;
    } else if (g.m <= 256) {
        bn = 128;
    } else if (g.m <= 384) {
        bm = g.k % 128 == 0 ? 192 : 384;
        bn = 128;
    }
    auto tiles = [&] { return ((g.m + bm - 1) / bm) * ((g.n + bn - 1) / bn); };
    if (small_tiles && tiles() < 32) {
        bm = bn = 64;
    }
    if (bm * lda >= (int64_t)INT32_MAX || (!trb && bn * ldb >= (int64_t)INT32_MAX)) {
        return r;
    }
    const int64_t bk = g.k % 128 == 0 ? 128 : 64, kt = g.k / bk;
    r.bm = bm;
    r.bn = bn;
    r.splits = kt < 16 ? 1 : (int)std::max<int64_t>(1, std::min<int64_t>(256 / tiles(), kt / (512 / bk)));
    r.mode = r.splits > 1 ? RING_PART : fused_mode(g);
    r.trb = trb;
    return r;
}

// The ring kernel needs K % 32 == 0 (bytes of k: whole matrix-core slices),
// 16-byte-aligned k-contiguous rows and 32-bit buffer offsets within a row
// panel.
// The tile and the K split are the cheapest by
//   rounds of 256 workgroups x k steps x the tile's step time
//   + (partials: 3 us, and their bytes written and read at 3.5 TB/s),
// since every sweep of tiles and splits (int8 and f16, 24 to 4096 rows) was
// won by a grid just under one workgroup per CU, whichever tile gives it, and
// a second workgroup on a CU doubles the time: 512 x 4096 x 4096 s8 18.4 us on
// 256 tiles of 128 x 64, 21 on 128 of 128 x 128, 27 on 512 of 64 x 64, 35 in
// eight K splits of 256 x 256; 1024 x 4096 x 4096 24.7 us on 256 tiles of
// 128 x 128, 42 on 256 x 256 in four splits. The estimate is within 20 % of
// the measured time where the matrix work or the staging bounds it. The partials
// of K splits stay under 32 MiB (an unsplit call's, where its mode has any, are
// one M x N array of 4 bytes), a split keeps at least 512 bytes of k, a k of fewer than
// 16 steps is not split (the reduce costs more than it gains), and a problem
// of few rows is split over small tiles only, which bounds the partials (and
// so the workspace) by those of one tile per CU. max_splits: what a workspace
// has room for (kMostSplits: all that the plan would take). The fused output
// modes (fused_mode) go without a split.
// trb: B is the caller's [K,N] (row pitch ldb), read in place (its whole
// span within 32-bit buffer offsets).
RingPlan plan_ring(const NnopsGemmI8Args& g, const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, bool trb,
                   int max_splits)
{
    RingPlan r;
    if (g.m < 1 || g.n < 1 || g.m > INT32_MAX || g.n > INT32_MAX - 3 || g.k > INT32_MAX - 127 || g.k < 32 || g.k % 32 != 0 || !aligned16(a, lda) || !aligned16(b, ldb)) {
        return r;
    }
    if (trb && (g.k * ldb + g.n >= (int64_t)INT32_MAX || ldb < g.n)) {
        return r;
    }
    const int fused = fused_mode(g);
    const uint32_t m = (uint32_t)g.m, n = (uint32_t)g.n, kt = (uint32_t)((g.k + 127) / 128);
    const float out_bytes = 4.0f * (float)m * (float)n;
    const uint32_t most = std::min({(uint32_t)max_splits, kt / 4u, (uint32_t)(32.0f * 1024 * 1024 / out_bytes)});
    const int split_area = m <= 256 ? 256 * 128 : m <= 384 ? 192 * 128 : 256 * 256;
    float best = 0.0f;
    for (const RingTile& t : kRingTiles) {
        if ((trb && t.bn == 192) || t.bm * lda >= (int64_t)INT32_MAX ||
            (!trb && t.bn * ldb >= (int64_t)INT32_MAX)) {
            continue;
        }
        const uint64_t tiles = (uint64_t)((m + t.bm - 1) / (uint32_t)t.bm) * ((n + t.bn - 1) / (uint32_t)t.bn);
        auto consider = [&](uint32_t sp, uint64_t rounds) {
            const uint32_t steps = kt - (sp - 1) * (kt / sp);       // the last split's, the longest
            const bool part = sp > 1 || fused == RING_PART;
            const float us = (float)rounds * (float)steps * t.step_us +
                             (part ? 3.0f + 2.0f * (float)sp * out_bytes / 3.5e6f : 0.0f);
            if (r.bm == 0 || us < best) {
                best = us;
                r.bm = t.bm;
                r.bn = t.bn;
                r.splits = (int)sp;
                r.mode = part ? RING_PART : fused;
            }
        };
        consider(1, (tiles + 255) / 256);
        if (tiles <= 128 && kt >= 16 && t.bm * t.bn <= split_area) {
            // the split that fills the CUs, and half of it
            const uint32_t sp = std::min(most, 256u / (uint32_t)tiles);
            if (sp > 1) {
                consider(sp, 1);
            }
            if (sp > 3) {
                consider(sp / 2, 1);
            }
        }
    }
    if (r.bm != 0) {
        r.us = best;
        r.trb = trb;
    }
    return r;
}

}  // namespace nnops_amd
