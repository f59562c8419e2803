// Dense fp product of nnops' float MatMul / Linear routes (nnops_hip_gemm_fp):
// C = alpha * (A B) for f32 x f32 or f16 x f16 operands, accumulated in f32
// and rounded once to C's type (f32 or f16). nnops' own f16 route keeps its
// accumulator in C between 128-deep k blocks (FpRoute<half>, Acc = half,
// src/backend/cpu/matmul/matmul.cpp:57-62, KC_CAP_F16 = 128 in
// matmul_helper.h:272), so it rounds the partial sums to f16 along the way;
// the single rounding here is the more accurate of the two. The epilogue
// (bias, beta, residual, activation, Linear's gated combine) is the output
// pass of fp_out.hip over this product.
//
// Kernels
//   gemv_fp_nk<AF16,MT>   M <= 16 rows of A in one launch, B [N][K] rows (the
//                         Linear weight): a wave owns 4 rows of B, its lanes
//                         stride 16-byte chunks over K, A read from L2; the
//                         lanes' sums meet by shuffles. Bound: HBM.
//   gemv_fp_kn<AF16,MT>   M <= 16, B [K][N]: a lane owns one 16-byte column
//                         chunk (8 f16 / 4 f32 columns), the block's 4 waves
//                         quarters of its K range (met in LDS); A through the
//                         scalar cache; K split over blockIdx.y into f32
//                         partials summed by fp_split_sum. Bound: HBM.
//   gemm_fp_tile<AF16,TB> the other shapes: 128 x 128 tiles, 4 waves of
//                         64 x 64, v_mfma_f32_32x32x2f32 with A and B staged
//                         in LDS as f32 (32-deep k stages). Bound: f32 MFMA.
//   fp_split_sum          C = alpha * (sum of the K splits in split order).
// The f16 operands of aligned shapes past a few rows take the int8 ring GEMM's byte
// staging with f16 MFMA instead (gemm_f16.hip, nnops_amd::ring_gemm_f16).
#include "common.hpp"

#include <algorithm>
#include <type_traits>

namespace nnops_amd {

// gemm_f16.hip: the ring GEMM over f16 operands (C = alpha A B, f32 or f16 C),
// or NNOPS_UNSUPPORTED, nothing launched, where the shape, the alignment or
// (shapes with another kernel) the workspace does not fit it.
int ring_gemm_f16(const NnopsGemmFpArgs& g, void* workspace, size_t ws_bytes, hipStream_t s);
size_t ring_gemm_f16_workspace(const NnopsGemmFpArgs& g);

namespace {

struct FpKern {
    const void* a;
    const void* b;
    void* c;
    float* part;            // [splits][M][N] f32 partials, or nullptr: write C
    int m, n, k;
    int64_t lda, ldb, ldc;  // elements
    int out_f16;
    float alpha;
    int splits, kper;
};

template <bool AF16>
__device__ __forceinline__ float ld1(const void* base, int64_t i)
{
    if constexpr (AF16) {
        return (float)static_cast<const _Float16*>(base)[i];
    } else {
        return static_cast<const float*>(base)[i];
    }
}

__device__ __forceinline__ void st_out(const FpKern& p, int m, int n, float v)
{
    if (p.out_f16) {
        static_cast<_Float16*>(p.c)[(int64_t)m * p.ldc + n] = (_Float16)v;
    } else {
        static_cast<float*>(p.c)[(int64_t)m * p.ldc + n] = v;
    }
}

// 16 bytes as f32 values: 8 halves or 4 floats.
template <bool AF16>
struct Chunk {
    static constexpr int E = AF16 ? 8 : 4;
};

template <bool AF16>
__device__ __forceinline__ void unpack16(v4i x, float (&f)[Chunk<AF16>::E])
{
    if constexpr (AF16) {
        const v8h h = __builtin_bit_cast(v8h, x);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            f[e] = (float)h[e];
        }
    } else {
        const v4f v = __builtin_bit_cast(v4f, x);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] = v[e];
        }
    }
}

// ---------------------------------------------------------------------------
// GEMV over B [N][K]: wave w of the block owns rows n0 .. n0 + 3; lane l takes
// chunks l, l + 64, ... of each row (16 bytes each), A's MT rows kept packed
// (one 16-byte chunk per row of A); f16 pairs are dotted with v_dot2_f32_f16
// (exact products, f32 sums), f32 with fma. VEC: 16-byte aligned rows of A and
// B, K a whole number of chunks; otherwise element loads.
// ---------------------------------------------------------------------------
template <bool AF16, int MT, bool VEC>
__global__ __launch_bounds__(256) void gemv_fp_nk(FpKern p)
{
    constexpr int E = Chunk<AF16>::E;
    constexpr int R = 4;
    const int lane = threadIdx.x & 63;
    const int n0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * R;
    if (n0 >= p.n) {
        return;
    }
    const int chunks = (p.k + E - 1) / E;
    float acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            acc[r][m] = 0.0f;
        }
    }
    // 16 bytes of row `row` of X from element k0 (zeros past K)
    auto chunk16 = [&](const void* x, int64_t ld, int64_t row, int k0) {
        if constexpr (VEC) {
            return *reinterpret_cast<const v4i*>(static_cast<const char*>(x) + (row * ld + k0) * (AF16 ? 2 : 4));
        } else {
            uint32_t w[4];
            if constexpr (AF16) {
                const uint16_t* src = static_cast<const uint16_t*>(x) + row * ld + k0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint32_t lo = k0 + 2 * q < p.k ? src[2 * q] : 0u;
                    const uint32_t hi = k0 + 2 * q + 1 < p.k ? src[2 * q + 1] : 0u;
                    w[q] = lo | (hi << 16);
                }
            } else {
                const uint32_t* src = static_cast<const uint32_t*>(x) + row * ld + k0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    w[q] = k0 + q < p.k ? src[q] : 0u;
                }
            }
            return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
        }
    };
    for (int c = lane; c < chunks; c += 64) {
        const int k0 = c * E;
        v4i av[MT];
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            av[m] = chunk16(p.a, p.lda, min(m, p.m - 1), k0);
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const v4i bv = chunk16(p.b, p.ldb, min(n0 + r, p.n - 1), k0);
#pragma unroll
            for (int m = 0; m < MT; ++m) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    // the words as scalars first: a bit cast of a subscripted
                    // vector element reads element 0 with this compiler
                    const uint32_t aw = (uint32_t)av[m][q], bw = (uint32_t)bv[q];
                    if constexpr (AF16) {
                        acc[r][m] = __builtin_amdgcn_fdot2(__builtin_bit_cast(v2h, aw), __builtin_bit_cast(v2h, bw),
                                                           acc[r][m], false);
                    } else {
                        acc[r][m] = fmaf(__builtin_bit_cast(float, aw), __builtin_bit_cast(float, bw), acc[r][m]);
                    }
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            float v = acc[r][m];
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                v += __shfl_xor(v, off, 64);
            }
            acc[r][m] = v;
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                if (n0 + r < p.n && m < p.m) {
                    st_out(p, m, n0 + r, acc[r][m] * p.alpha);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// GEMV over B [K][N]: block (bx, split) owns the 64 16-byte column chunks
// bx * 64 .. + 63 (one per lane, E columns each) for rows [split * kper,
// + kper); its 4 waves take a quarter of those rows each and meet in LDS, so
// a split writes one partial per output. A's rows are wave-uniform: read
// through the scalar cache. VEC: 16-byte aligned B rows and N a whole number
// of chunks; otherwise element loads.
// ---------------------------------------------------------------------------
template <bool AF16, int MT, bool VEC>
__global__ __launch_bounds__(256) void gemv_fp_kn(FpKern p)
{
    constexpr int E = Chunk<AF16>::E;
    typedef std::conditional_t<AF16, _Float16, float> T;
    typedef const __attribute__((address_space(4))) T* ConstT;
    __shared__ float red[3][E][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int c0 = (blockIdx.x * 64 + lane) * E;
    const int ks = blockIdx.y * p.kper;
    const int ke = min(p.k, ks + p.kper);
    const int kq = (ke - ks + 3) / 4;
    const int k0 = ks + wave * kq;
    const int k1 = min(ke, k0 + kq);
    float acc[MT][E];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            acc[m][e] = 0.0f;
        }
    }
    ConstT arow[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        arow[m] = (ConstT)(static_cast<const T*>(p.a) + (int64_t)min(m, p.m - 1) * p.lda);
    }
    const int cc = min(c0, (p.n - 1) / E * E);   // a chunk past N re-reads the last one (never stored)
    auto load_row = [&](int k, float (&bv)[E]) {
        if constexpr (VEC) {
            const char* src = static_cast<const char*>(p.b) + ((int64_t)k * p.ldb + cc) * (AF16 ? 2 : 4);
            unpack16<AF16>(*reinterpret_cast<const v4i*>(src), bv);
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                bv[e] = cc + e < p.n ? ld1<AF16>(p.b, (int64_t)k * p.ldb + cc + e) : 0.0f;
            }
        }
    };
    constexpr int U = 4;
    int k = k0;
    for (; k + U <= k1; k += U) {
        float bv[U][E];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            load_row(k + u, bv[u]);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const float a = (float)arow[m][k + u];
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    acc[m][e] = fmaf(a, bv[u][e], acc[m][e]);
                }
            }
        }
    }
    for (; k < k1; ++k) {
        float bv[E];
        load_row(k, bv);
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const float a = (float)arow[m][k];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                acc[m][e] = fmaf(a, bv[e], acc[m][e]);
            }
        }
    }
    // the four quarters meet in LDS (wave order), one row of A at a time
#pragma unroll
    for (int m = 0; m < MT; ++m) {
        if (wave > 0) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                red[wave - 1][e][lane] = acc[m][e];
            }
        }
        __syncthreads();
        if (wave == 0 && m < p.m && c0 < p.n) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float v = ((acc[m][e] + red[0][e][lane]) + red[1][e][lane]) + red[2][e][lane];
                if (c0 + e < p.n) {
                    if (p.part != nullptr) {
                        p.part[((int64_t)blockIdx.y * p.m + m) * p.n + c0 + e] = v;
                    } else {
                        st_out(p, m, c0 + e, v * p.alpha);
                    }
                }
            }
        }
        __syncthreads();
    }
}

// C = alpha * sum of the splits (split order): one thread per output, its
// loads issued 8 splits at a time.
__global__ __launch_bounds__(256) void fp_split_sum(FpKern p)
{
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)p.m * p.n) {
        return;
    }
    const int64_t slab = (int64_t)p.m * p.n;
    float s = 0.0f;
    int sp = 0;
    for (; sp + 8 <= p.splits; sp += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            v[u] = p.part[(sp + u) * slab + i];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            s += v[u];
        }
    }
    for (; sp < p.splits; ++sp) {
        s += p.part[sp * slab + i];
    }
    const int m = (int)(i / p.n);
    st_out(p, m, (int)(i - (int64_t)m * p.n), s * p.alpha);
}

// ---------------------------------------------------------------------------
// MFMA tile GEMM in f32 (f32 operands, or f16 ones widened on the way into
// LDS): 128 x 128 tiles, 4 waves of 64 x 64 (2 x 2 fragments of
// v_mfma_f32_32x32x2f32). Per 32-deep k stage A is staged as [m][k] f32 rows
// and B as [n][k] rows, both with a 4-float pad. Lane group g (lane >> 5)
// owns k = 16 g .. 16 g + 15 of the stage for A and B alike (the MFMA's k
// index is the lane group, so any such assignment sums the same products),
// and a lane reads its 16 operands of a fragment with four 16-byte reads.
// TB: B [N][K] rows (else [K][N]).
// ---------------------------------------------------------------------------
template <bool AF16, bool TB>
__global__ __launch_bounds__(256, 1) void gemm_fp_tile(FpKern p)
{
    constexpr int BM = 128, BN = 128, LD = 36;
    constexpr int ES = AF16 ? 2 : 4;
    __shared__ __attribute__((aligned(16))) float lds_a[2][BM * LD];
    __shared__ __attribute__((aligned(16))) float lds_b[2][BN * LD];

    const int tiles_n = (p.n + BN - 1) / BN;
    const int tm = blockIdx.x / tiles_n;
    const int tn = blockIdx.x - tm * tiles_n;
    const int m0 = tm * BM, n0 = tn * BN;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm0 = (wave >> 1) * 64, wn0 = (wave & 1) * 64;
    // whole 4-element loads where the rows allow them
    const bool a_vec = (p.lda * ES) % (4 * ES) == 0 && ((uintptr_t)p.a % (4 * ES)) == 0;
    const bool b_vec = (p.ldb * ES) % (4 * ES) == 0 && ((uintptr_t)p.b % (4 * ES)) == 0;

    // 4 elements from row `row` of X starting at column col (zero past cols)
    auto load4 = [&](const void* x, int64_t ld, bool vec, int64_t row, int col, int cols, float (&f)[4]) {
        const int64_t base = row * ld + col;
        if (vec && col + 4 <= cols) {
            if constexpr (AF16) {
                const uint2 w = *reinterpret_cast<const uint2*>(static_cast<const _Float16*>(x) + base);
                const _Float16* h = reinterpret_cast<const _Float16*>(&w);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[e] = (float)h[e];
                }
            } else {
                const v4f v = *reinterpret_cast<const v4f*>(static_cast<const float*>(x) + base);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    f[e] = v[e];
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f[e] = col + e < cols ? ld1<AF16>(x, base + e) : 0.0f;
            }
        }
    };

    float ra[4][4], rb[4][4];
    auto load_stage = [&](int k0) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + i * 256;
            const int r = idx >> 3, c = idx & 7;       // 8 chunks of 4 per 32-deep row
            load4(p.a, p.lda, a_vec, min(m0 + r, p.m - 1), k0 + 4 * c, p.k, ra[i]);
            if constexpr (TB) {
                load4(p.b, p.ldb, b_vec, min(n0 + r, p.n - 1), k0 + 4 * c, p.k, rb[i]);
            } else {
                // 32 k rows x 128 columns: row idx >> 5, columns 4 (idx & 31) ..
                const int kr = idx >> 5, cn = idx & 31;
                if (k0 + kr < p.k) {
                    load4(p.b, p.ldb, b_vec, k0 + kr, n0 + 4 * cn, p.n, rb[i]);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        rb[i][e] = 0.0f;
                    }
                }
            }
        }
    };
    auto store_stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int idx = tid + i * 256;
            const int r = idx >> 3, c = idx & 7;
            *reinterpret_cast<v4f*>(&lds_a[buf][r * LD + 4 * c]) = v4f{ra[i][0], ra[i][1], ra[i][2], ra[i][3]};
            if constexpr (TB) {
                *reinterpret_cast<v4f*>(&lds_b[buf][r * LD + 4 * c]) = v4f{rb[i][0], rb[i][1], rb[i][2], rb[i][3]};
            } else {
                const int kr = idx >> 5, cn = idx & 31;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lds_b[buf][(4 * cn + e) * LD + kr] = rb[i][e];
                }
            }
        }
    };

    v16f acc[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[i][j] = v16f{0.0f};
        }
    }
    const int kt = (p.k + 31) / 32;
    const int fr = lane & 31, fg = 16 * (lane >> 5);
    load_stage(0);
    store_stage(0);
    __syncthreads();
    for (int t = 0; t < kt; ++t) {
        const int cur = t & 1;
        if (t + 1 < kt) {
            load_stage((t + 1) * 32);
        }
        v4f fa[2][4], fb[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                fa[i][q] = *reinterpret_cast<const v4f*>(&lds_a[cur][(wm0 + 32 * i + fr) * LD + fg + 4 * q]);
                fb[i][q] = *reinterpret_cast<const v4f*>(&lds_b[cur][(wn0 + 32 * i + fr) * LD + fg + 4 * q]);
            }
        }
#pragma unroll
        for (int s = 0; s < 16; ++s) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][s >> 2][s & 3], fb[j][s >> 2][s & 3],
                                                                    acc[i][j], 0, 0, 0);
                }
            }
        }
        if (t + 1 < kt) {
            store_stage(cur ^ 1);
        }
        __syncthreads();
    }

#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + wn0 + 32 * j + fr;
        if (n >= p.n) {
            continue;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + wm0 + 32 * i + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                if (m < p.m) {
                    st_out(p, m, n, acc[i][j][r] * p.alpha);
                }
            }
        }
    }
}

constexpr int kGemvRows = 16;    // rows of A per GEMV launch
constexpr int64_t kGemvMaxM = 16;

// K split of the [K][N] GEMV: about 512 workgroups (each 1 KiB of columns),
// at least 128 rows (32 per wave) per split
int kn_splits_fp(int64_t n, int64_t k, bool f16)
{
    const int64_t blocks = (n + (f16 ? 8 : 4) * 64 - 1) / ((f16 ? 8 : 4) * 64);
    int64_t s = (512 + blocks - 1) / blocks;
    s = std::min<int64_t>(s, std::max<int64_t>(1, k / 128));
    return (int)std::max<int64_t>(1, std::min<int64_t>(s, 1024));
}

template <bool AF16, int MT>
void launch_gemv(const FpKern& k, bool tb, bool vec, hipStream_t s)
{
    if (tb) {
        const dim3 grid((unsigned)((k.n + 15) / 16));      // 4 waves of 4 rows of B
        if (vec) {
            NNOPS_LAUNCH((gemv_fp_nk<AF16, MT, true>), grid, dim3(256), 0, s, k);
        } else {
            NNOPS_LAUNCH((gemv_fp_nk<AF16, MT, false>), grid, dim3(256), 0, s, k);
        }
    } else {
        const int e = AF16 ? 8 : 4;
        const dim3 grid((unsigned)((k.n + 64 * e - 1) / (64 * e)), (unsigned)k.splits);
        if (vec) {
            NNOPS_LAUNCH((gemv_fp_kn<AF16, MT, true>), grid, dim3(256), 0, s, k);
        } else {
            NNOPS_LAUNCH((gemv_fp_kn<AF16, MT, false>), grid, dim3(256), 0, s, k);
        }
    }
}

template <bool AF16>
void launch_gemv_rows(const FpKern& k, bool tb, bool vec, hipStream_t s)
{
    if (k.m == 1) {
        launch_gemv<AF16, 1>(k, tb, vec, s);
    } else if (k.m == 2) {
        launch_gemv<AF16, 2>(k, tb, vec, s);
    } else if (k.m <= 4) {
        launch_gemv<AF16, 4>(k, tb, vec, s);
    } else if (k.m <= 8) {
        launch_gemv<AF16, 8>(k, tb, vec, s);
    } else {
        launch_gemv<AF16, 16>(k, tb, vec, s);
    }
}

bool use_gemv_fp(const NnopsGemmFpArgs& g)
{
    return g.m <= kGemvMaxM;
}

// the [K][N] GEMV's K-split partials
size_t gemv_fp_workspace(const NnopsGemmFpArgs& g)
{
    if (g.trans_b) {
        return 0;
    }
    const int splits = kn_splits_fp(g.n, g.k, g.in_f16 != 0);
    const int64_t rows = std::min<int64_t>(g.m, kGemvRows);
    return splits > 1 ? (size_t)splits * (size_t)rows * (size_t)g.n * sizeof(float) : 0;
}

}  // namespace
}  // namespace nnops_amd

using namespace nnops_amd;

extern "C" size_t nnops_hip_gemm_fp_workspace_size(const NnopsGemmFpArgs* g)
{
    if (g == nullptr || g->m <= 0 || g->n <= 0 || g->k <= 0) {
        return 0;
    }
    const size_t gemv = use_gemv_fp(*g) ? gemv_fp_workspace(*g) : 0;
    // room for the ring's plan, which pointer alignment (not seen by a size
    // query) may rule out in favour of the GEMV or the tile kernel
    return g->in_f16 ? std::max(gemv, ring_gemm_f16_workspace(*g)) : gemv;
}

extern "C" int nnops_hip_gemm_fp(const NnopsGemmFpArgs* g, void* workspace, size_t ws_bytes, void* stream)
{
    const TimingDisarm disarm;
    if (g == nullptr) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (g->m < 0 || g->n < 0 || g->k < 0) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (g->m == 0 || g->n == 0) {
        return NNOPS_OK;
    }
    if (g->a == nullptr || g->b == nullptr || g->c == nullptr) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (g->m > INT32_MAX || g->n > INT32_MAX || g->k > INT32_MAX) {
        return NNOPS_UNSUPPORTED;
    }
    if (g->lda < g->k || g->ldc < g->n || g->ldb < (g->trans_b ? g->k : g->n)) {
        return NNOPS_INVALID_ARGUMENT;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool f16 = g->in_f16 != 0;
    if (f16 && g->k > 0) {
        // the f16 ring, where it takes the call
        if (const int rc = ring_gemm_f16(*g, workspace, ws_bytes, s); rc != NNOPS_UNSUPPORTED) {
            return rc;
        }
    }
    const size_t need = use_gemv_fp(*g) ? gemv_fp_workspace(*g) : 0;
    if (need > 0 && (workspace == nullptr || ws_bytes < need)) {
        return NNOPS_NOT_INITIALIZED;
    }
    const int es = f16 ? 2 : 4;
    FpKern k{};
    k.a = g->a;
    k.b = g->b;
    k.c = g->c;
    k.m = (int)g->m;
    k.n = (int)g->n;
    k.k = (int)g->k;
    k.lda = g->lda;
    k.ldb = g->ldb;
    k.ldc = g->ldc;
    k.out_f16 = g->out_f16 != 0;
    k.alpha = g->alpha;
    k.splits = 1;
    k.kper = k.k;
    if (g->k == 0) {
        // an empty sum: C = 0
        k.splits = 0;
        NNOPS_LAUNCH(fp_split_sum, dim3((unsigned)((g->m * g->n + 255) / 256)), dim3(256), 0, s, k);
        return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
    }
    if (use_gemv_fp(*g)) {
        const bool tb = g->trans_b != 0;
        // 16-byte chunks along the contiguous dimension
        const bool vec = tb ? ((g->lda * es) % 16 == 0 && (g->ldb * es) % 16 == 0 && (g->k * es) % 16 == 0 &&
                               (uintptr_t)g->a % 16 == 0 && (uintptr_t)g->b % 16 == 0)
                            : ((g->ldb * es) % 16 == 0 && (g->n * es) % 16 == 0 && (uintptr_t)g->b % 16 == 0);
        if (!tb) {
            k.splits = kn_splits_fp(g->n, g->k, f16);
            k.kper = (int)((g->k + k.splits - 1) / k.splits);
            k.splits = (int)((g->k + k.kper - 1) / k.kper);
        }
        for (int m0 = 0; m0 < k.m; m0 += kGemvRows) {
            FpKern kk = k;
            kk.m = std::min(kGemvRows, k.m - m0);
            kk.a = static_cast<const char*>(g->a) + (int64_t)m0 * g->lda * es;
            kk.c = static_cast<char*>(g->c) + (int64_t)m0 * g->ldc * (g->out_f16 ? 2 : 4);
            kk.part = kk.splits > 1 ? static_cast<float*>(workspace) : nullptr;
            if (f16) {
                launch_gemv_rows<true>(kk, tb, vec, s);
            } else {
                launch_gemv_rows<false>(kk, tb, vec, s);
            }
            if (kk.splits > 1) {
                NNOPS_LAUNCH(fp_split_sum, dim3((unsigned)(((int64_t)kk.m * kk.n + 255) / 256)), dim3(256), 0,
                                   s, kk);
            }
        }
        return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
    }
    const int64_t tiles = ((g->m + 127) / 128) * ((g->n + 127) / 128);
    if (tiles > INT32_MAX) {
        return NNOPS_UNSUPPORTED;
    }
    if (f16) {
        if (g->trans_b) {
            NNOPS_LAUNCH((gemm_fp_tile<true, true>), dim3((unsigned)tiles), dim3(256), 0, s, k);
        } else {
            NNOPS_LAUNCH((gemm_fp_tile<true, false>), dim3((unsigned)tiles), dim3(256), 0, s, k);
        }
    } else if (g->trans_b) {
        NNOPS_LAUNCH((gemm_fp_tile<false, true>), dim3((unsigned)tiles), dim3(256), 0, s, k);
    } else {
        NNOPS_LAUNCH((gemm_fp_tile<false, false>), dim3((unsigned)tiles), dim3(256), 0, s, k);
    }
    return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
}
