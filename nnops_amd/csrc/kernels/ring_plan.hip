// Which tile and K split a call of the LDS-ring GEMM takes (host code).
#include "gemm_i8_ring.hpp"

namespace nnops_amd {
namespace {

// The ring's tile shapes and the time of one 128-byte k step of one workgroup
// with one workgroup on every CU, over [N,K] rows of B and over a [K,N] B in
// place (0: not taken there). The 192-column tiles are for widths that leave 128
// and 256 columns with a last round nearly empty: 1000 x 4096 x 11008 f16 115 ->
// 105 us on 232 tiles of 256 x 192 against 172 of 256 x 256, 512 rows 67 -> 60
// (s8 36 -> 33).
struct RingTile {
    int bm, bn;
    float step_us, trb_step_us;
};
constexpr RingTile kRingTiles[] = {
    {64, 64, 0.31f, 0.58f},    {128, 64, 0.40f, 0.48f},  {128, 128, 0.53f, 0.61f},
    {192, 128, 0.74f, 0.84f},  {128, 192, 0.75f, 0.0f},  {256, 128, 0.89f, 1.04f},
    {128, 256, 0.90f, 1.04f},  {256, 192, 1.13f, 0.0f},  {256, 256, 1.28f, 1.30f},
};

// The step time of the 64 x 64 tiles over a [K,N] B that an XCD's L2 holds: their
// stages read 64 bytes of each row of B, from further away at half the rate.
constexpr float kTrbSmallStepUs = 0.37f;
constexpr int64_t kTrbSmallBytes = 6000000;

// The time of `wgs` workgroups of `steps` k steps each: per round of 256 of them
// what the first stages and the output take, by the tile's area, and the steps,
// which take less where a last round leaves CUs idle (the matrix cores' clock and
// the L2s are shared: down to 0.85 of it at half of the CUs, the small tiles
// 0.91). A grid that is no multiple of the 8 XCDs is not remapped to them, so
// that the row tiles of one column band read B into several L2s: 8 % more.
float ring_us(const RingTile& t, float step_us, uint64_t wgs, uint32_t steps, bool bands)
{
    const float area = (float)(t.bm * t.bn);
    const uint64_t full = wgs / 256, rest = wgs % 256;
    const float low = t.bm * t.bn > 128 * 128 ? 0.85f : 0.91f;
    const float last = rest == 0 ? 0.0f : low + (1.0f - low) * std::max(0.0f, (float)rest * (1.0f / 128.0f) - 1.0f);
    const float us = ((float)full + last) * (float)steps * step_us;
    return (wgs % 8 != 0 && bands && wgs > 128 ? 1.08f * us : us) +
           (float)(full + (rest != 0 ? 1 : 0)) * (3.0f + area * (4.3f / 65536.0f));
}

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
// The tile and the K split are the cheapest by ring_us, plus, with partials, 2.4
// us and 0.38 us per MB of them (0.71 past 8 splits of int8, whose reduce is then
// gemm_i8_reduce<16>). That was fitted to 852 shapes of 17 to 2048 rows (int8 s8 /
// s32 / [K,N], f16; k 256 and widths 128 to 14336), each timed in graphs on 3 to
// 20 tiles and splits, 7792 times in all: within 8 % of them (one standard
// deviation). Its choices are 0.9 % slower than the best of each shape's and in 3
// of 100 by more than 10 %; an estimate by rounds and full step times alone had
// left 1.6 % and 6 of 100, 907 x 1344 x 9680 over a [K,N] B 32.6 us for 21.0 and
// 929 x 7616 x 4944 f16 108 for 83.
// The partials of K splits stay under 64 MiB (an unsplit call's, where its mode
// has any, are one M x N array of 4 bytes), a split keeps at least 512 bytes of
// k, a k of fewer than 16 steps is not split (the reduce costs more than it
// gains), and a problem of few rows is split over small tiles only, which bounds
// the partials (and so the workspace) by those of one tile per CU; tiles of 192
// and 256 rows that are over twice its rows are not looked at. max_splits:
// what a workspace has room for (kMostSplits: all that the plan would take). The
// fused output modes (fused_mode) go without a split.
// trb: B is the caller's [K,N] (row pitch ldb), read in place (its whole
// span within 32-bit buffer offsets). f16: f16 operands.
RingPlan plan_ring(const NnopsGemmI8Args& g, const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, bool trb,
                   int max_splits, bool f16)
{
    RingPlan r;
    if (g.m < 1 || g.n < 1 || g.m > INT32_MAX || g.n > INT32_MAX - 3 || g.k > INT32_MAX - 127 || g.k < 32 ||
        g.k % 32 != 0 || !aligned16(a, lda) || !aligned16(b, ldb)) {
        return r;
    }
    if (trb && (g.k * ldb + g.n >= (int64_t)INT32_MAX || ldb < g.n)) {
        return r;
    }
    const int fused = fused_mode(g);
    const uint32_t m = (uint32_t)g.m, n = (uint32_t)g.n, kt = (uint32_t)((g.k + 127) / 128);
    const float out_bytes = 4.0f * (float)m * (float)n;
    const uint32_t most = std::min({(uint32_t)max_splits, kt / 4u, (uint32_t)(64.0f * 1024 * 1024 / out_bytes)});
    const int split_area = m <= 256 ? 256 * 128 : m <= 384 ? 192 * 128 : 256 * 256;
    float best = 0.0f;
    for (const RingTile& t : kRingTiles) {
        float step_us = trb ? t.trb_step_us : t.step_us;
        if (step_us == 0.0f || (t.bm > 128 && (uint32_t)t.bm > 2 * m) || t.bm * lda >= (int64_t)INT32_MAX ||
            (!trb && t.bn * ldb >= (int64_t)INT32_MAX)) {
            continue;
        }
        if (trb && t.bm * t.bn == 64 * 64 && g.k * g.n < kTrbSmallBytes) {
            step_us = kTrbSmallStepUs;
        }
        const uint32_t row_tiles = (m + (uint32_t)t.bm - 1) / (uint32_t)t.bm;
        const uint64_t tiles = (uint64_t)row_tiles * ((n + (uint32_t)t.bn - 1) / (uint32_t)t.bn);
        auto consider = [&](uint32_t sp) {
            const uint32_t steps = kt - (sp - 1) * (kt / sp);       // the last split's, the longest
            const bool part = sp > 1 || fused == RING_PART;
            const float byte_us = !f16 && sp > 8 ? 0.71e-6f : 0.38e-6f;
            const float us = ring_us(t, step_us, tiles * sp, steps, row_tiles > 1) +
                             (part ? 2.4f + (float)sp * out_bytes * byte_us : 0.0f);
            if (r.bm == 0 || us < best) {
                best = us;
                r.bm = t.bm;
                r.bn = t.bn;
                r.splits = (int)sp;
                r.mode = part ? RING_PART : fused;
            }
        };
        consider(1);
        if (tiles <= 128 && kt >= 16 && t.bm * t.bn <= split_area) {
            // the split that fills the CUs, parts of it, and the least
            const uint32_t top = std::min(most, 256u / (uint32_t)tiles);
            for (const uint32_t sp : {top, top / 2, top / 3}) {
                if (sp > 2) {
                    consider(sp);
                }
            }
            if (top >= 2) {
                consider(2);
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
