// ---------------------------------------------------------------------------
// The ring over f16 operands (nnops_hip_gemm_fp's large shapes): the same
// byte staging, K and the row pitches in bytes; B [N][K] rows in place, or a
// [K][N] B transposed into the workspace first. RING_FP writes alpha * acc
// straight to C; K splits write f32 partials that ring_f16_reduce sums.
// ---------------------------------------------------------------------------
#include "gemm_i8_ring.hpp"

namespace nnops_amd {
namespace {

// dst[c][r] = src[r][c] over 64 x 64 tiles in LDS, rows R to Rp of dst's rows
// 0 (an f16 [K][N] B staged as [N][Kp]). Bound: HBM.
__global__ __launch_bounds__(256) void transpose_b16(const uint16_t* src, int64_t lds_, int R, int C,
                                                    uint16_t* dst, int64_t ldd, int Rp)
{
    __shared__ uint16_t tile[64][65];
    const int r0 = blockIdx.y * 64;
    const int c0 = blockIdx.x * 64;
    const int tx = threadIdx.x & 63;
    const int ty = threadIdx.x >> 6;
    for (int i = ty; i < 64; i += 4) {
        const int r = r0 + i, c = c0 + tx;
        tile[i][tx] = (r < R && c < C) ? src[(int64_t)r * lds_ + c] : (uint16_t)0;
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
        const int c = c0 + i, r = r0 + tx;
        if (c < C && r < Rp) {
            dst[(int64_t)c * ldd + r] = tile[tx][i];
        }
    }
}

// C = alpha * (the f16 ring's f32 partials summed in split order): 4 columns
// per thread (the last past N cut), grid.y walking the rows; a group's splits are loaded
// four at a time ahead of their sum. Bound: HBM / MALL.
__global__ __launch_bounds__(256) void ring_f16_reduce(GemmI8Kern p, RingSplit sk)
{
    const int nb = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
    if (nb >= p.n) {
        return;
    }
    const bool f16 = p.ep.out_kind == NNOPS_OUT_F16;
    const int64_t slab = (int64_t)p.m * sk.ldp;
    const int cn = min(4, p.n - nb);
    for (int m = (int)blockIdx.y; m < p.m; m += (int)gridDim.y) {
        const float* src = reinterpret_cast<const float*>(sk.part) + (int64_t)m * sk.ldp + nb;
        v4f v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        int sp = 0;
        for (; sp + 3 < sk.splits; sp += 4) {
            const v4f x0 = *reinterpret_cast<const v4f*>(src + sp * slab);
            const v4f x1 = *reinterpret_cast<const v4f*>(src + (sp + 1) * slab);
            const v4f x2 = *reinterpret_cast<const v4f*>(src + (sp + 2) * slab);
            const v4f x3 = *reinterpret_cast<const v4f*>(src + (sp + 3) * slab);
            v = (((v + x0) + x1) + x2) + x3;
        }
        for (; sp < sk.splits; ++sp) {
            v += *reinterpret_cast<const v4f*>(src + sp * slab);
        }
        char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e >= cn) {
                break;
            }
            const float y = __fmul_rn(v[e], p.ep.s_a_scalar);
            if (f16) {
                reinterpret_cast<_Float16*>(crow)[nb + e] = (_Float16)y;
            } else {
                reinterpret_cast<float*>(crow)[nb + e] = y;
            }
        }
    }
}

struct F16Plan {
    RingPlan ring;          // mode < 0: the ring does not take the call
    bool stage_b = false;
    int64_t kp = 0;         // staged B row bytes
    size_t part_off = 0, total = 0;
};

// Few rows over [N][K] rows of B that the GEMV is the faster for: 1 and 2, and
// 3 and 4 (one pass of it) over a short k or a long one with many columns. GEMV
// against ring, us, weights in the cache and from HBM:
//   2 x 4096 x 4096            9.7 / 13.7
//   3 x 512 x 1000      4.6 /  5.9    4.6 /  5.9
//   3 x 1024 x 1024     5.3 /  6.0    7.1 /  6.7
//   3 x 1536 x 100      5.8 /  6.5    5.8 /  6.4
//   3 x 1792 x 4096                  12.5 /  9.6
//   3 x 4096 x 4096    13.1 / 12.3   19.3 / 14.9
//   3 x 1536 x 14336   12.5 / 11.8   16.4 / 13.4
//   3 x 8192 x 11008                 48.2 / 46.5
//   3 x 8192 x 14336   41.0 / 40.9   53.6 / 57.9
inline bool gemv_f16_faster(const NnopsGemmFpArgs& g)
{
    return g.m < 3 || (g.m <= 4 && ((g.k < 1792 && g.n <= 8192) || (g.k >= 8192 && g.n > 11008)));
}

// From 3 rows over [N][K] rows of B (4096 x 4096: 16 rows 13.7 us against the
// GEMV's 21.4), but where the GEMV is the faster, and from 17 over a [K][N] B,
// whose transposed copy the GEMV needs not (17 to 63 rows on gemm_fp_tile, in
// f32: 475 us). room: the workspace that K splits may use. by_rows: the plan by
// the call's rows alone, whose workspace is enough.
F16Plan plan_f16(const NnopsGemmFpArgs& g, size_t room = SIZE_MAX, bool by_rows = false)
{
    F16Plan f;
    if (!g.in_f16 || (g.trans_b ? gemv_f16_faster(g) : g.m < 17) || 2 * g.k > INT32_MAX || g.m > INT32_MAX ||
        g.n > INT32_MAX) {
        return f;
    }
    NnopsGemmI8Args x{};
    x.m = g.m;
    x.n = g.n;
    x.k = 2 * g.k;
    x.trans_b = 1;
    x.a = g.a;
    x.lda = 2 * g.lda;
    x.c = g.c;
    x.ldc = g.ldc;
    x.out_kind = g.out_f16 ? NNOPS_OUT_F16 : NNOPS_OUT_F32;
    x.act = NNOPS_ACT_NONE;
    x.s_a_scalar = g.alpha;
    x.s_b_scalar = 1.0f;
    const int8_t* b = static_cast<const int8_t*>(g.b);
    int64_t ldb = 2 * g.ldb;
    size_t off = 0;
    if (!g.trans_b) {
        f.stage_b = true;
        f.kp = (2 * g.k + 127) / 128 * 128;
        off += align_up((size_t)g.n * (size_t)f.kp);
        b = nullptr;          // the staged copy: 256-byte aligned, 128-byte rows
        ldb = f.kp;
    }
    const int8_t* a = static_cast<const int8_t*>(g.a);
    if (by_rows) {
        f.ring = plan_ring_by_rows(x, a, x.lda, b, ldb, false, false);
        // (128 x 256 tiles that nearly fill the CUs: no split)
        if (f.ring.splits > 1 && g.m > 128 && ((g.m + 127) / 128) * ((g.n + 255) / 256) >= 192 &&
            (uintptr_t)g.c % 16 == 0 && (g.ldc * (g.out_f16 ? 2 : 4)) % 16 == 0) {
            f.ring.splits = 1;
            f.ring.mode = RING_FP;
        }
    } else {
        f.ring = plan_ring(x, a, x.lda, b, ldb, false, std::max(1, splits_in(room, off, g.m, g.n)), true);
    }
    // up to 8 rows, two passes of the GEMV, over a k too short to split and with
    // a destination that needs the pass over partials (5 x 768 x 1001: GEMV 7.2
    // us, ring and pass 8.0)
    const bool short_pass = g.trans_b && g.m <= 8 && g.k < 1024 && f.ring.mode == RING_PART;
    if (short_pass || (f.ring.mode != RING_FP && f.ring.mode != RING_PART)) {
        f.ring = RingPlan{};
        f.stage_b = false;
        return f;
    }
    if (f.ring.mode == RING_PART) {
        f.part_off = off;
        off += align_up((size_t)f.ring.splits * (size_t)g.m * (size_t)((g.n + 3) / 4) * 16);
    }
    f.total = off;
    return f;
}

// The plan that a call with ws_bytes of workspace runs on (if that holds it).
F16Plan choose_f16(const NnopsGemmFpArgs& g, size_t ws_bytes)
{
    const F16Plan f = plan_f16(g);
    return ws_bytes < f.total ? plan_f16(g, ws_bytes) : f;
}

// The plan's workspace. The destination's alignment (which a size query may not
// see) picks between the fused output and the split partials: room for either.
size_t f16_workspace(const NnopsGemmFpArgs& g, bool by_rows)
{
    NnopsGemmFpArgs x = g;
    const size_t a = plan_f16(x, SIZE_MAX, by_rows).total;
    x.c = reinterpret_cast<void*>(uintptr_t{2});
    return std::max(a, plan_f16(x, SIZE_MAX, by_rows).total);
}

// Shapes that the GEMV and the tile kernel take without a workspace.
inline bool ring_f16_optional(const NnopsGemmFpArgs& g) { return g.m < 64 || g.k % 32 != 0 || g.n % 4 != 0; }

}  // namespace

size_t ring_gemm_f16_workspace(const NnopsGemmFpArgs& g)
{
    return f16_workspace(g, false);
}

extern "C" int nnops_hip_gemm_fp_plan(const NnopsGemmFpArgs* g, size_t ws_bytes, NnopsGemmPlan* out)
{
    if (g == nullptr || out == nullptr || g->m <= 0 || g->n <= 0 || g->k <= 0) {
        return NNOPS_INVALID_ARGUMENT;
    }
    *out = NnopsGemmPlan{};
    const F16Plan f = choose_f16(*g, ws_bytes);
    if (f.ring.mode >= 0 && f.total <= ws_bytes) {
        out->tile_m = f.ring.bm;
        out->tile_n = f.ring.bn;
        out->splits = f.ring.splits;
        out->fused = f.ring.mode != RING_PART;
        out->short_stage = 2 * g->k % 128 != 0;
        out->workspace_bytes = f.total;
    }
    return NNOPS_OK;
}

int ring_gemm_f16(const NnopsGemmFpArgs& g, void* workspace, size_t ws_bytes, hipStream_t s)
{
    const bool optional = ring_f16_optional(g);
    if (workspace == nullptr || (optional && (uintptr_t)workspace % 16 != 0)) {
        ws_bytes = 0;
    }
    const F16Plan f = choose_f16(g, ws_bytes);
    if (f.ring.mode < 0) {
        return NNOPS_UNSUPPORTED;
    }
    if (ws_bytes < f.total) {
        return optional ? NNOPS_UNSUPPORTED : NNOPS_NOT_INITIALIZED;
    }
    if (!optional && ws_bytes < f16_workspace(g, false) && ws_bytes < f16_workspace(g, true)) {
        return NNOPS_NOT_INITIALIZED;       // less than the query's, and than is enough
    }
    if (!optional && (uintptr_t)workspace % 16 != 0) {
        return NNOPS_INVALID_ARGUMENT;   // staged operands and partials are 16-byte vectors
    }
    char* ws = static_cast<char*>(workspace);
    GemmI8Kern k{};
    k.m = (int)g.m;
    k.n = (int)g.n;
    k.k = (int)(2 * g.k);
    k.a = static_cast<const int8_t*>(g.a);
    k.lda = 2 * g.lda;
    k.c = g.c;
    k.ldc_bytes = g.ldc * (g.out_f16 ? 2 : 4);
    if (f.stage_b) {
        uint16_t* bt = reinterpret_cast<uint16_t*>(ws);
        const dim3 grid((unsigned)((g.n + 63) / 64), (unsigned)((f.kp / 2 + 63) / 64));
        NNOPS_LAUNCH(transpose_b16, grid, dim3(256), 0, s, static_cast<const uint16_t*>(g.b), g.ldb,
                           (int)g.k, (int)g.n, bt, f.kp / 2, (int)(f.kp / 2));
        k.b = reinterpret_cast<const int8_t*>(bt);
        k.ldb = f.kp;
    } else {
        k.b = static_cast<const int8_t*>(g.b);
        k.ldb = 2 * g.ldb;
    }
    EpiParams& e = k.ep;
    e.s_a_scalar = g.alpha;
    e.s_b_scalar = 1.0f;
    e.out_kind = g.out_f16 ? NNOPS_OUT_F16 : NNOPS_OUT_F32;
    e.act = NNOPS_ACT_NONE;
    e.min_clip = -INFINITY;
    e.max_clip = INFINITY;
    const RingSplit sk = ring_split(k, f.ring, reinterpret_cast<int32_t*>(ws + f.part_off));
    launch_ring_tiles<true, false>(k, f.ring, sk, s);
    if (f.ring.mode == RING_PART) {
        const dim3 grid((unsigned)((sk.ldp / 4 + 255) / 256), (unsigned)std::min(k.m, 65535));
        NNOPS_LAUNCH(ring_f16_reduce, grid, dim3(256), 0, s, k, sk);
    }
    return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
}

}  // namespace nnops_amd
