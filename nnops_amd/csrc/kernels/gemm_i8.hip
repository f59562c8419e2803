// Integer GEMM on gfx950: s8|u8 x s8 -> int32 accumulate on the int8 matrix
// cores, with the nnops output pass (compensate, bias, Relu, requant, or the
// float epilogue) applied to the accumulators in registers.
//
// Kernels
//   gemm_i8_mfma   M > 16: block tile BMxBN, k-step 64, A and B staged through
//                  LDS (k-contiguous rows padded to 80 B, so the 16-byte
//                  fragment reads of 8 consecutive rows hit disjoint banks),
//                  double-buffered global->register->LDS, v_mfma_i32_32x32x32_i8.
//                  Bound: MFMA (4096^3: arithmetic intensity ~2730 op/B).
//   gemv_i8_lds    4 < M <= 16, B [N][K]: 16 rows of B per block staged through
//                  LDS in 1 KiB row pieces, v_mfma_i32_16x16x64_i8.
//   gemv_i8_mfma   M <= 16 otherwise: one 16-column slice of B per block, K split over
//                  the block's 4 waves, fragments loaded straight from HBM into
//                  v_mfma_i32_16x16x64_i8 operands (no LDS on the weight path),
//                  partial tiles summed through LDS. Bound: HBM (weight bytes).
//   transpose_i8   [R][C] -> [C][R'] byte transpose through LDS (k-contiguous
//                  staging of a [K,N] B or a [K,M] A).
//   rowsum_i8      sum_k of each k-contiguous row (zero-point compensation).
//
// The reduction order of the int32 accumulate is irrelevant (integer addition
// is associative), so both kernels are bit-exact whatever the k split.
#include "gemm_i8_ring.hpp"

namespace nnops_amd {
namespace {

constexpr int kBK = 64;        // k bytes per pipeline stage
constexpr int kLdsRow = 80;    // LDS row pitch (64 + 16 pad) in bytes

// ---------------------------------------------------------------------------
// 16-byte fragment loads (ALIGNED: base, pitch and K are multiples of 16).
// ---------------------------------------------------------------------------
template <bool ALIGNED>
__device__ __forceinline__ v4i load16(const int8_t* row, int k0, int K)
{
    if constexpr (ALIGNED) {
        if (k0 < K) {
            return *reinterpret_cast<const v4i*>(row + k0);
        }
        return v4i{0, 0, 0, 0};
    } else {
        uint32_t w[4];
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint32_t v = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const int kk = k0 + d * 4 + b;
                const uint32_t byte = kk < K ? (uint32_t)(uint8_t)row[kk] : 0u;
                v |= byte << (8 * b);
            }
            w[d] = v;
        }
        return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
}

// A u8 operand is fed to the signed MFMA as a - 128 (flip the top bit of every
// byte); the epilogue adds 128 * sum_k b back through a_off. Padding bytes past
// K must stay 0 after the flip, which `valid` takes care of.
__device__ __forceinline__ v4i flip_u8(v4i v, uint32_t x, bool valid)
{
    if (x == 0u || !valid) {
        return v;
    }
    return v4i{(int)((uint32_t)v.x ^ x), (int)((uint32_t)v.y ^ x), (int)((uint32_t)v.z ^ x),
               (int)((uint32_t)v.w ^ x)};
}

// Unaligned path: bytes past K must read as 0 after the flip too, so flip per byte.
template <bool ALIGNED>
__device__ __forceinline__ v4i load16_a(const int8_t* row, int k0, int K, uint32_t x)
{
    v4i v = load16<ALIGNED>(row, k0, K);
    if (x == 0u) {
        return v;
    }
    if constexpr (ALIGNED) {
        return flip_u8(v, x, k0 < K);
    } else {
        uint32_t w[4] = {(uint32_t)v.x, (uint32_t)v.y, (uint32_t)v.z, (uint32_t)v.w};
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            uint32_t mask = 0;
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if (k0 + d * 4 + b < K) {
                    mask |= 0x80u << (8 * b);
                }
            }
            w[d] ^= mask;
        }
        return v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
    }
}

// ---------------------------------------------------------------------------
// Block-index mapping: consecutive logical tiles on one XCD (the hardware
// deals workgroups round-robin over the 8 XCDs), then grouped along M so the
// tiles resident on one XCD share A row panels and B column panels in its L2.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void tile_coords(int tiles_m, int tiles_n, int& tm, int& tn)
{
    int bid = blockIdx.x;
    const int nb = gridDim.x;
    if ((nb & 7) == 0) {
        bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    }
    constexpr int G = 4;
    const int per_group = G * tiles_n;
    const int group = bid / per_group;
    const int first_m = group * G;
    const int gsize = min(tiles_m - first_m, G);
    const int in_group = bid - group * per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// Stage loader: CA/CB 16-byte chunks per thread per 64-byte k stage. FULLK:
// K is a multiple of 64 and every row is 16-byte aligned, so no load needs a
// bound; otherwise chunks past K read as zero (ALIGNED or per byte).
template <int C, bool FULLK, bool ALIGNED, bool FLIP>
__device__ __forceinline__ void load_chunks(v4i (&r)[C], const int8_t* const (&src)[C],
                                            const int (&kc)[C], int k0, int K, uint32_t x)
{
#pragma unroll
    for (int i = 0; i < C; ++i) {
        if constexpr (FULLK) {
            r[i] = *reinterpret_cast<const v4i*>(src[i] + k0 + kc[i]);
            if constexpr (FLIP) {
                r[i] = flip_u8(r[i], x, true);
            }
        } else if constexpr (FLIP) {
            r[i] = load16_a<ALIGNED>(src[i], k0 + kc[i], K, x);
        } else {
            r[i] = load16<ALIGNED>(src[i], k0 + kc[i], K);
        }
    }
}

// ---------------------------------------------------------------------------
// Output pass shared by the MFMA kernels. One 32-row slab of the wave tile at a
// time goes through LDS (32x32 accumulator layout: lane holds column lane & 31,
// rows 8*(r/4) + 4*(lane/32) + (r%4)); then every lane owns 4 consecutive
// columns and walks the slab's rows, so the destination is written with packed
// 4-byte (s8/u8) or 16-byte (s32) stores, 4 rows in flight per lane.
//   EPI_S8   integer requant with row-uniform scales (no zero points, no
//            per-row tables): req = (s_a / s_out) * s_b[n] hoisted per column;
//   EPI_S32  raw accumulate + bias (+ Relu), no zero points;
//   EPI_GENERIC  everything else (compensation, per-row tables, float epilogue).
// The fast modes evaluate exactly the float operations epi_value does.
// ---------------------------------------------------------------------------
enum { EPI_GENERIC = 0, EPI_S8 = 1, EPI_S32 = 2 };

template <int FM, int FN, int TN, int EPI>
__device__ __forceinline__ void output_pass(const GemmI8Kern& p, v16i (&acc)[FM][FN], int32_t* slab,
                                            int row0, int col0, int lane)
{
    constexpr int kEpiPitch = TN + 4;
    constexpr int kColGroups = TN / 4;                   // 4-column groups per slab row
    constexpr int kRowStep = 64 / kColGroups;            // rows covered per pass of the wave
    constexpr int kRowsPerLane = 32 / kRowStep;
    static_assert(kColGroups * kRowStep == 64 && kRowsPerLane * kRowStep == 32, "slab walk");
    const EpiParams& ep = p.ep;
    const int cg = lane % kColGroups;
    const int rsub = lane / kColGroups;
    const int nb = col0 + cg * 4;                        // first of this lane's 4 columns
    EpiCol cols[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        cols[e] = epi_col(ep, min(nb + e, p.n - 1));
    }
    float req[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (EPI == EPI_S8) {
        const float row_k = __fdiv_rn(ep.s_a_scalar, ep.s_out);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            req[e] = __fmul_rn(row_k, cols[e].s_b);
        }
    }
    const bool relu = ep.act == NNOPS_ACT_RELU;
    const bool u8 = ep.out_kind == NNOPS_OUT_U8;
    const bool s32 = ep.out_kind == NNOPS_OUT_S32;
    const bool packed = !epi_is_fp(ep) && (nb + 3 < p.n) && (((uintptr_t)p.c & 15) == 0) &&
                        (s32 ? (p.ldc_bytes % 16 == 0) : (p.ldc_bytes % 4 == 0));
    // Fast modes (host-checked: N % 4 == 0, 16-byte-aligned C, pitch multiple
    // of the packed store, half-away rounding): branch-free per element.
    const int32_t relu_floor = relu ? 0 : INT32_MIN;
    const float zpf = (float)ep.zp_out;
    const float lo = __fsub_rn(u8 ? 0.0f : -128.0f, zpf);
    const float hi = __fsub_rn(u8 ? 255.0f : 127.0f, zpf);
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int row = 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
                slab[row * kEpiPitch + j * 32 + (lane & 31)] = acc[i][j][r];
            }
        }
        __syncthreads();
        const int mbase = row0 + i * 32 + rsub;
        char* cbase = static_cast<char*>(p.c) + (int64_t)mbase * p.ldc_bytes +
                      (int64_t)nb * (s32 ? 4 : 1);
        const int64_t cstep = (int64_t)kRowStep * p.ldc_bytes;
#pragma unroll 4
        for (int t = 0; t < kRowsPerLane; ++t) {
            const int rr = rsub + t * kRowStep;
            const int m = mbase + t * kRowStep;
            char* cptr = cbase + t * cstep;
            if (m >= p.m || nb >= p.n) {
                continue;
            }
            const v4i raw = *reinterpret_cast<const v4i*>(&slab[rr * kEpiPitch + cg * 4]);
            if constexpr (EPI == EPI_S8) {
                uint32_t w = 0;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int32_t v = max(raw[e] + cols[e].bias, relu_floor);
                    float x = __fmul_rn((float)v, req[e]);
                    x = __builtin_fminf(__builtin_fmaxf(x, lo), hi);
                    const int32_t q = (int32_t)round_half_away(x) + ep.zp_out;
                    w |= ((uint32_t)q & 0xffu) << (8 * e);
                }
                *reinterpret_cast<uint32_t*>(cptr) = w;
            } else if constexpr (EPI == EPI_S32) {
                v4i q;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    q[e] = max(raw[e] + cols[e].bias, relu_floor);
                }
                *reinterpret_cast<v4i*>(cptr) = q;
            } else {
                char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
                const EpiRow row = epi_row(ep, m);
                if (packed && s32) {
                    int32_t q[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        q[e] = epi_value(ep, row, cols[e], raw[e], 0);
                    }
                    *reinterpret_cast<v4i*>(crow + (int64_t)nb * 4) = v4i{q[0], q[1], q[2], q[3]};
                } else if (packed) {
                    uint32_t old = 0;
                    if (ep.add_to) {
                        old = *reinterpret_cast<const uint32_t*>(crow + nb);
                    }
                    uint32_t w = 0;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t ob = (old >> (8 * e)) & 0xffu;
                        const int32_t o = u8 ? (int32_t)ob : (int32_t)(int8_t)ob;
                        w |= ((uint32_t)epi_value(ep, row, cols[e], raw[e], o) & 0xffu) << (8 * e);
                    }
                    *reinterpret_cast<uint32_t*>(crow + nb) = w;
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if (nb + e < p.n) {
                            epi_store(ep, row, cols[e], raw[e], crow, nb + e);
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------------------
// Register output pass (EPI_S8 / EPI_S32): the element math runs in the MFMA
// accumulator layout (lane = one column, 4 consecutive rows per register
// group), then each 4x4 block is transposed across the lane quad with DPP so a
// lane holds 4 consecutive columns of one row and writes them with one packed
// store. No LDS round trip and no block barrier.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int quad_bcast(int v, int k)
{
    // quad_perm(k, k, k, k): every lane of the quad reads lane k
    switch (k) {
    case 0: return __builtin_amdgcn_mov_dpp(v, 0x00, 0xf, 0xf, true);
    case 1: return __builtin_amdgcn_mov_dpp(v, 0x55, 0xf, 0xf, true);
    case 2: return __builtin_amdgcn_mov_dpp(v, 0xaa, 0xf, 0xf, true);
    default: return __builtin_amdgcn_mov_dpp(v, 0xff, 0xf, 0xf, true);
    }
}

// Lane qi holds bytes (row 0..3) of column qi; returns (column 0..3) of row qi.
// Two exchange stages: with lane xor 1 (swapping lane bit 0 with byte bit 0),
// then with lane xor 2 (bit 1 with bit 1); each is one DPP move and one
// v_perm whose per-lane byte selectors (sel1, sel2) come from quad_sel.
struct QuadSel {
    uint32_t s1, s2;
};

__device__ __forceinline__ QuadSel quad_sel(int qi)
{
    // v_perm_b32(hi = partner, lo = own, sel): selector byte b picks own.byte[b]
    // (b < 4) or partner.byte[b - 4]
    return QuadSel{(qi & 1) ? 0x03070105u : 0x06020400u, (qi & 2) ? 0x03020706u : 0x05040100u};
}

__device__ __forceinline__ uint32_t quad_transpose_bytes(uint32_t w, const QuadSel& qs)
{
    const uint32_t p1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0xb1, 0xf, 0xf, true);   // quad_perm(1,0,3,2)
    w = __builtin_amdgcn_perm(p1, w, qs.s1);
    const uint32_t p2 = (uint32_t)__builtin_amdgcn_mov_dpp((int)w, 0x4e, 0xf, 0xf, true);   // quad_perm(2,3,0,1)
    return __builtin_amdgcn_perm(p2, w, qs.s2);
}

// 4x4 dword transpose across the quad: v[r] = (row r, column qi) in,
// v[c] = (row qi, column c) out. Two exchange stages (lane xor 1, xor 2).
__device__ __forceinline__ void quad_transpose_dwords(int32_t (&v)[4], int qi)
{
    const bool odd = qi & 1;
#pragma unroll
    for (int a = 0; a < 4; a += 2) {
        const int send = odd ? v[a] : v[a + 1];
        const int recv = __builtin_amdgcn_mov_dpp(send, 0xb1, 0xf, 0xf, true);  // quad_perm(1,0,3,2)
        if (odd) {
            v[a] = recv;
        } else {
            v[a + 1] = recv;
        }
    }
    const bool hi = qi & 2;
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int send = hi ? v[a] : v[a + 2];
        const int recv = __builtin_amdgcn_mov_dpp(send, 0x4e, 0xf, 0xf, true);  // quad_perm(2,3,0,1)
        if (hi) {
            v[a] = recv;
        } else {
            v[a + 2] = recv;
        }
    }
}

// BIAS_IN_ACC: the accumulators started from bias[n], so it is not added again.
template <int FM, int FN, int EPI, bool BIAS_IN_ACC = false>
__device__ __forceinline__ void output_pass_regs(const GemmI8Kern& p, v16i (&acc)[FM][FN], int row0,
                                                 int col0, int lane)
{
    static_assert(EPI == EPI_S8 || EPI == EPI_S32, "register pass: fast modes only");
    const EpiParams& ep = p.ep;
    const int qi = lane & 3;
    const QuadSel qs = quad_sel(qi);
    const int colq = (lane & 31) & ~3;
    int32_t relu_floor = ep.act == NNOPS_ACT_RELU ? 0 : INT32_MIN;
    asm("" : "+s"(relu_floor));   // one max per element, not max + select on the flag
    const bool u8 = ep.out_kind == NNOPS_OUT_U8;
    const int32_t lo_i = (u8 ? 0 : -128) - ep.zp_out;
    const int32_t hi_i = (u8 ? 255 : 127) - ep.zp_out;
    const float row_k = __fdiv_rn(ep.s_a_scalar, ep.s_out);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        const int n_own = col0 + j * 32 + (lane & 31);       // column held before the transpose
        const EpiCol col = epi_col(ep, min(n_own, p.n - 1));
        const float req = __fmul_rn(row_k, col.s_b);
        const int n_st = col0 + j * 32 + colq;               // first column stored by this lane
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int m = row0 + i * 32 + 8 * g + 4 * (lane >> 5) + qi;
                char* cptr = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
                if constexpr (EPI == EPI_S8) {
                    uint32_t q[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int32_t v = max(acc[i][j][4 * g + e] + (BIAS_IN_ACC ? 0 : col.bias), relu_floor);
                        const float x = __fmul_rn((float)v, req);
                        // round half away from zero (the conversion truncates, as
                        // trunc() would), then clamp in the integer domain: lo and
                        // hi are integers and rounding is monotonic, so this equals
                        // clamping x first; |x| past 2^31 saturates the conversion.
                        const int32_t r = (int32_t)__fadd_rn(x, __builtin_copysignf(0.5f, x));
                        q[e] = (uint32_t)(med3_i32(r, lo_i, hi_i) + ep.zp_out);
                    }
                    // low bytes of q[0..3] -> one word (0x0c selects a zero byte)
                    const uint32_t w01 = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u);
                    const uint32_t w23 = __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
                    const uint32_t w = quad_transpose_bytes(w01 | w23, qs);
                    if (m < p.m && n_st < p.n) {
                        *reinterpret_cast<uint32_t*>(cptr + n_st) = w;
                    }
                } else {
                    int32_t v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = max(acc[i][j][4 * g + e] + (BIAS_IN_ACC ? 0 : col.bias), relu_floor);
                    }
                    quad_transpose_dwords(v, qi);
                    if (m < p.m && n_st < p.n) {
                        *reinterpret_cast<v4i*>(cptr + (int64_t)n_st * 4) = v4i{v[0], v[1], v[2], v[3]};
                    }
                }
            }
        }
    }
}

template <int BM, int BN, int WM, int WN, int WPE, bool FULLK, bool ALIGNED, bool FLIP, int EPI>
__global__ __launch_bounds__(WM * WN * 64) __attribute__((amdgpu_waves_per_eu(WPE, WPE)))
void gemm_i8_mfma(GemmI8Kern p)
{
    constexpr int T = WM * WN * 64;
    constexpr int TM = BM / WM;           // wave tile rows
    constexpr int TN = BN / WN;           // wave tile cols
    constexpr int FM = TM / 32;           // 32x32 fragments per wave
    constexpr int FN = TN / 32;
    constexpr int CA = BM * (kBK / 16) / T;   // 16-byte chunks per thread per stage
    constexpr int CB = BN * (kBK / 16) / T;
    static_assert(CA >= 1 && CB >= 1 && CA * T == BM * 4 && CB * T == BN * 4, "tile/threads");

    constexpr int kStageBytes = 2 * (BM + BN) * kLdsRow;
    constexpr int kEpiPitch = TN + 4;                      // int32 per staged output row
    constexpr int kEpiBytes = WM * WN * 32 * kEpiPitch * 4;
    static_assert(kEpiBytes <= kStageBytes, "epilogue staging must fit the stage buffers");
    __shared__ __attribute__((aligned(16))) int8_t lds_raw[kStageBytes];
    int8_t (*lds_a)[BM * kLdsRow] = reinterpret_cast<int8_t (*)[BM * kLdsRow]>(lds_raw);
    int8_t (*lds_b)[BN * kLdsRow] = reinterpret_cast<int8_t (*)[BN * kLdsRow]>(lds_raw + 2 * BM * kLdsRow);

    int tm, tn;
    tile_coords((p.m + BM - 1) / BM, (p.n + BN - 1) / BN, tm, tn);
    const int m0 = tm * BM;
    const int n0 = tn * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int wm0 = (wave / WN) * TM;
    const int wn0 = (wave % WN) * TN;

    // Per-thread stage chunks (rows past M/N are clamped: computed, never stored).
    const int8_t* a_src[CA];
    const int8_t* b_src[CB];
    int a_lds[CA], b_lds[CB], a_kc[CA], b_kc[CB];
#pragma unroll
    for (int i = 0; i < CA; ++i) {
        const int idx = tid + i * T;
        const int r = idx >> 2, c = idx & 3;
        a_src[i] = p.a + (int64_t)min(m0 + r, p.m - 1) * p.lda;
        a_kc[i] = c * 16;
        a_lds[i] = r * kLdsRow + c * 16;
    }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        const int idx = tid + i * T;
        const int r = idx >> 2, c = idx & 3;
        b_src[i] = p.b + (int64_t)min(n0 + r, p.n - 1) * p.ldb;
        b_kc[i] = c * 16;
        b_lds[i] = r * kLdsRow + c * 16;
    }

    v4i ra[CA], rb[CB];
    v16i acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            acc[i][j] = v16i{0};
        }
    }

    const int frag_row = lane & 31;
    const int frag_k = (lane >> 5) * 16;
    const int kt = (p.k + kBK - 1) / kBK;

    load_chunks<CA, FULLK, ALIGNED, FLIP>(ra, a_src, a_kc, 0, p.k, p.a_xor);
    load_chunks<CB, FULLK, ALIGNED, false>(rb, b_src, b_kc, 0, p.k, 0u);
#pragma unroll
    for (int i = 0; i < CA; ++i) {
        *reinterpret_cast<v4i*>(&lds_a[0][a_lds[i]]) = ra[i];
    }
#pragma unroll
    for (int i = 0; i < CB; ++i) {
        *reinterpret_cast<v4i*>(&lds_b[0][b_lds[i]]) = rb[i];
    }
    __syncthreads();

    for (int t = 0; t < kt; ++t) {
        const int cur = t & 1;
        const bool more = t + 1 < kt;
        if (more) {
            load_chunks<CA, FULLK, ALIGNED, FLIP>(ra, a_src, a_kc, (t + 1) * kBK, p.k, p.a_xor);
            load_chunks<CB, FULLK, ALIGNED, false>(rb, b_src, b_kc, (t + 1) * kBK, p.k, 0u);
        }
        const int8_t* la = &lds_a[cur][(wm0 + frag_row) * kLdsRow + frag_k];
        const int8_t* lb = &lds_b[cur][(wn0 + frag_row) * kLdsRow + frag_k];
#pragma unroll
        for (int ks = 0; ks < kBK; ks += 32) {
            v4i fa[FM], fb[FN];
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                fa[i] = *reinterpret_cast<const v4i*>(la + i * 32 * kLdsRow + ks);
            }
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                fb[j] = *reinterpret_cast<const v4i*>(lb + j * 32 * kLdsRow + ks);
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) {
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fa[i], fb[j], acc[i][j], 0, 0, 0);
                }
            }
        }
        if (more) {
#pragma unroll
            for (int i = 0; i < CA; ++i) {
                *reinterpret_cast<v4i*>(&lds_a[cur ^ 1][a_lds[i]]) = ra[i];
            }
#pragma unroll
            for (int i = 0; i < CB; ++i) {
                *reinterpret_cast<v4i*>(&lds_b[cur ^ 1][b_lds[i]]) = rb[i];
            }
        }
        __syncthreads();
    }

    if constexpr (EPI == EPI_GENERIC) {
        output_pass<FM, FN, TN, EPI>(p, acc, reinterpret_cast<int32_t*>(lds_raw) + wave * 32 * kEpiPitch,
                                     m0 + wm0, n0 + wn0, lane);
    } else {
        output_pass_regs<FM, FN, EPI>(p, acc, m0 + wm0, n0 + wn0, lane);
    }
}

// The output pass of 4 consecutive columns nb..nb+3 of row m: its row and
// column constants and the residual word, loaded before the raw sums arrive
// (out4_prepare), then the pass itself (out4_store).
struct Out4 {
    EpiRow row;
    EpiCol cols[4];
    uint32_t oldw;
    char* crow;
    int8_t* c8;
    int cn;            // columns within N
    bool word8;
};

__device__ __forceinline__ Out4 out4_prepare(const GemmI8Kern& p, int m, int nb)
{
    const EpiParams& ep = p.ep;
    Out4 o{};
    o.crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
    o.c8 = reinterpret_cast<int8_t*>(o.crow) + nb;
    o.cn = min(4, p.n - nb);
    o.word8 = !epi_is_fp(ep) && ep.out_kind != NNOPS_OUT_S32 && o.cn == 4 && ((uintptr_t)o.c8 & 3) == 0;
    o.row = epi_row(ep, m);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        o.cols[e] = epi_col(ep, min(nb + e, p.n - 1));
    }
    if (o.word8 && ep.add_to) {
        o.oldw = *reinterpret_cast<const uint32_t*>(o.c8);
    }
    return o;
}

__device__ __forceinline__ void out4_store(const GemmI8Kern& p, const Out4& o, int nb, v4i raw)
{
    const EpiParams& ep = p.ep;
    const bool u8 = ep.out_kind == NNOPS_OUT_U8;
    if (epi_is_fp(ep)) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e < o.cn) {
                epi_store(ep, o.row, o.cols[e], raw[e], o.crow, nb + e);
            }
        }
        return;
    }
    if (ep.out_kind == NNOPS_OUT_S32) {
        int32_t* c32 = reinterpret_cast<int32_t*>(o.crow) + nb;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e < o.cn) {
                c32[e] = epi_value(ep, o.row, o.cols[e], raw[e], 0);
            }
        }
        return;
    }
    if (o.word8) {
        // one 4-byte read of the residual (in out4_prepare) and one 4-byte store
        uint32_t outw = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t ob = (o.oldw >> (8 * e)) & 0xffu;
            const int32_t old = u8 ? (int32_t)ob : (int32_t)(int8_t)ob;
            outw |= ((uint32_t)epi_value(ep, o.row, o.cols[e], raw[e], old) & 0xffu) << (8 * e);
        }
        *reinterpret_cast<uint32_t*>(o.c8) = outw;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (e >= o.cn) {
            break;
        }
        const int32_t old = ep.add_to ? (u8 ? (int32_t)((const uint8_t*)o.c8)[e] : (int32_t)o.c8[e]) : 0;
        o.c8[e] = (int8_t)epi_value(ep, o.row, o.cols[e], raw[e], old);
    }
}

// Sum of the K-split partial accumulators and the full output pass
// (compensation, bias, Relu, requant or the float epilogue, add_to). TPG
// threads share a group of 4 consecutive columns of a row (the last past N is cut), each
// summing every TPG-th split with its loads in flight together, then combine
// with lane shuffles; the first of them runs the output pass. TPG = 16 suits
// many splits of a small output (each thread's loads in one round trip), TPG =
// 1 a few splits of a large one.
template <int TPG>
__global__ __launch_bounds__(256) void gemm_i8_reduce(GemmI8Kern p, RingSplit sk)
{
    const int groups = sk.ldp / 4;
    const int64_t gid = ((int64_t)blockIdx.x * 256 + threadIdx.x) / TPG;
    const int j = threadIdx.x % TPG;
    const bool in = gid < (int64_t)p.m * groups;
    const int m = in ? (int)(gid / groups) : 0;
    const int nb = in ? (int)(gid - (int64_t)m * groups) * 4 : 0;
    const int64_t slab = (int64_t)p.m * sk.ldp;
    const int32_t* src = sk.part + (int64_t)m * sk.ldp + nb;
    // the output pass's constants and the residual word, loaded with the
    // partials rather than after them
    Out4 o{};
    if (in && j == 0) {
        o = out4_prepare(p, m, nb);
    }
    v4i raw = v4i{0, 0, 0, 0};
    if (in) {
        int s = j;
        for (; s + 3 * TPG < sk.splits; s += 4 * TPG) {
            const v4i x0 = *reinterpret_cast<const v4i*>(src + s * slab);
            const v4i x1 = *reinterpret_cast<const v4i*>(src + (s + TPG) * slab);
            const v4i x2 = *reinterpret_cast<const v4i*>(src + (s + 2 * TPG) * slab);
            const v4i x3 = *reinterpret_cast<const v4i*>(src + (s + 3 * TPG) * slab);
            raw += (x0 + x1) + (x2 + x3);
        }
        for (; s < sk.splits; s += TPG) {
            raw += *reinterpret_cast<const v4i*>(src + s * slab);
        }
    }
    if constexpr (TPG > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
            for (int o = 1; o < TPG; o <<= 1) {
                raw[e] += __shfl_xor(raw[e], o);
            }
        }
    }
    if (!in || j != 0) {
        return;
    }
    out4_store(p, o, nb, raw);
}

// round(gelu_tanh(x) / s_out), clamped, where a cheap evaluation settles it:
// gelu(x) = x / (1 + 2^(-2 log2(e) c (x + 0.044715 x^3))) on the hardware's
// exponential and reciprocal. With T = 1 + tanh its error against gelu_tanh's
// T is below 5e-7 + 5e-7 T: the exponent's rounding moves T by at most 8e-8
// (2 |a| e / (1 + e)^2 2^-23 over all e = 2^a), the exponential, the sum and the
// reciprocal by 4e-7 T, and gelu_tanh's own tanh and sum are within 2.4e-7; the
// products and the quotient add 3e-7 of the value. `sure` is set where the
// quotient is further from the next rounding boundary (a half-integer, in
// either rounding) than twice all of that, |x / s_out| (5e-7 + 8e-7 T); NaN and
// overflow compare as not sure. A third of gelu_tanh's instructions.
__device__ __forceinline__ float gelu_quotient(float x, float inv_out, bool& sure)
{
    const float x3 = __fmul_rn(__fmul_rn(__fmul_rn(0.044715f, x), x), x);
    const float e = __builtin_amdgcn_exp2f((x + x3) * (-2.0f * 1.44269504f * 0.7978845608f));
    const float r = __builtin_amdgcn_rcpf(1.0f + e);          // T / 2
    const float z = x * inv_out;
    const float y = z * r;
    const float off = __builtin_fabsf(__builtin_amdgcn_fractf(__builtin_fabsf(y)) - 0.5f);
    sure = off > __builtin_fabsf(z) * __builtin_fmaf(r, 16e-7f, 5e-7f);
    return y;
}

// The same sum and output pass for s8 / u8 destinations with row-uniform
// parameters (per-tensor s_a, s_out and zp_out, no zero-point terms, 16-byte
// aligned tables, 4-byte aligned destination rows), with the activation,
// float epilogue and residual order fixed at compile time: every load a
// thread needs (its splits' partial groups, the column tables and the
// residual word) is issued before the first is used, and the arithmetic is
// straight-line. One thread per 4-column group, grid.y walking the rows (no
// per-thread division for the row); element for element the operations of
// epi_value, so the bytes equal gemm_i8_reduce's.
template <int ACT, bool FEP, bool ADD, bool PRE>
__global__ __launch_bounds__(256) void gemm_i8_reduce_q(GemmI8Kern p, RingSplit sk)
{
    const EpiParams& ep = p.ep;
    const int nb = ((int)blockIdx.x * 256 + (int)threadIdx.x) * 4;
    if (nb >= p.n) {
        return;
    }
    const v4f sb = ep.s_b != nullptr ? *reinterpret_cast<const v4f*>(ep.s_b + nb)
                                     : v4f{ep.s_b_scalar, ep.s_b_scalar, ep.s_b_scalar, ep.s_b_scalar};
    const v4i bias = ep.bias != nullptr ? *reinterpret_cast<const v4i*>(ep.bias + nb) : v4i{0, 0, 0, 0};
    const bool u8 = ep.out_kind == NNOPS_OUT_U8;
    const bool even = ep.round_even != 0;
    const float row_k = sk.row_k;
    const float inv_out = sk.inv_out;
    const bool clip = !(ep.min_clip == -__builtin_inff() && ep.max_clip == __builtin_inff());
    const int64_t slab = (int64_t)p.m * p.n;              // N % 4 == 0: the partials' pitch is N
    for (int m = (int)blockIdx.y; m < p.m; m += (int)gridDim.y) {
        const int32_t* src = sk.part + (int64_t)m * p.n + nb;
        v4i raw = v4i{0, 0, 0, 0};
        int s = 0;
        for (; s + 3 < sk.splits; s += 4) {
            const v4i x0 = *reinterpret_cast<const v4i*>(src + s * slab);
            const v4i x1 = *reinterpret_cast<const v4i*>(src + (s + 1) * slab);
            const v4i x2 = *reinterpret_cast<const v4i*>(src + (s + 2) * slab);
            const v4i x3 = *reinterpret_cast<const v4i*>(src + (s + 3) * slab);
            raw += (x0 + x1) + (x2 + x3);
        }
        for (; s < sk.splits; ++s) {
            raw += *reinterpret_cast<const v4i*>(src + s * slab);
        }
        int8_t* c8 = static_cast<int8_t*>(p.c) + (int64_t)m * p.ldc_bytes + nb;
        uint32_t oldw = 0;
        if constexpr (ADD) {
            oldw = *reinterpret_cast<const uint32_t*>(c8);
        }
        uint32_t outw = 0;
        if constexpr (FEP && ACT == NNOPS_ACT_GELU && !ADD) {
            // the cheap evaluation, where it settles all four roundings
            bool sure = true;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float f = __fmul_rn((float)(raw[e] + bias[e]), __fmul_rn(ep.s_a_scalar, sb[e]));
                if (clip) {
                    f = f < ep.min_clip ? ep.min_clip : f;
                    f = ep.max_clip < f ? ep.max_clip : f;
                }
                bool s1;
                const int32_t q = requant_clamped(gelu_quotient(f, inv_out, s1), ep.zp_out, u8, even);
                outw |= ((uint32_t)q & 0xffu) << (8 * e);
                sure = sure && s1;
            }
            if (sure) {
                *reinterpret_cast<uint32_t*>(c8) = outw;
                continue;
            }
            outw = 0;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            int32_t v = raw[e] + bias[e];
            int32_t q;
            if constexpr (!FEP) {
                if constexpr (ACT == NNOPS_ACT_RELU) {
                    v = v < 0 ? 0 : v;
                }
                q = requant_clamped(__fmul_rn((float)v, __fmul_rn(row_k, sb[e])), ep.zp_out, u8, even);
            } else {
                float f = __fmul_rn((float)v, __fmul_rn(ep.s_a_scalar, sb[e]));
                float res = 0.0f;
                if constexpr (ADD) {
                    const uint32_t ob = (oldw >> (8 * e)) & 0xffu;
                    const int32_t old = u8 ? (int32_t)ob : (int32_t)(int8_t)ob;
                    res = __fmul_rn((float)(old - ep.zp_out), ep.s_out);
                    if constexpr (PRE) {
                        f = __fadd_rn(f, res);
                    }
                }
                if (clip) {   // the default -inf / +inf clip is the identity
                    f = f < ep.min_clip ? ep.min_clip : f;
                    f = ep.max_clip < f ? ep.max_clip : f;
                }
                if constexpr (ACT == NNOPS_ACT_RELU) {
                    f = f > 0.0f ? f : 0.0f;
                } else if constexpr (ACT == NNOPS_ACT_GELU) {
                    f = gelu_tanh(f);
                }
                if constexpr (ADD && !PRE) {
                    f = __fadd_rn(f, res);
                }
                q = requant_clamped(div_by_fixed(f, ep.s_out, inv_out), ep.zp_out, u8, even);
            }
            outw |= ((uint32_t)q & 0xffu) << (8 * e);
        }
        *reinterpret_cast<uint32_t*>(c8) = outw;
    }
}

// ---------------------------------------------------------------------------
// GEMV / skinny GEMM, M <= 16.
// ---------------------------------------------------------------------------
template <int U, bool ALIGNED>
__global__ __launch_bounds__(256) void gemv_i8_mfma(GemmI8Kern p)
{
    constexpr int W = 4;                  // waves per block, splitting K
    __shared__ v4i red[W - 1][64];

    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int n0 = blockIdx.x * 16;
    const int col = min(n0 + (lane & 15), p.n - 1);
    const int arow = lane & 15;
    const bool a_live = arow < p.m;
    const int kg = (lane >> 4) * 16;
    const int8_t* brow = p.b + (int64_t)col * p.ldb;
    const int8_t* a_row = p.a + (int64_t)(a_live ? arow : 0) * p.lda;

    const int ksteps = (p.k + 63) / 64;
    v4i acc = {0, 0, 0, 0};
    for (int s0 = wave * U; s0 < ksteps; s0 += W * U) {
        v4i fb[U], fa[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k0 = (s0 + u) * 64 + kg;
            const bool live = (s0 + u) < ksteps;
            fb[u] = live ? load16<ALIGNED>(brow, k0, p.k) : v4i{0, 0, 0, 0};
            fa[u] = (live && a_live) ? load16_a<ALIGNED>(a_row, k0, p.k, p.a_xor)
                                     : v4i{0, 0, 0, 0};
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[u], fb[u], acc, 0, 0, 0);
        }
    }

    if (wave > 0) {
        red[wave - 1][lane] = acc;
    }
    __syncthreads();
    if (wave != 0) {
        return;
    }
#pragma unroll
    for (int w = 0; w < W - 1; ++w) {
        acc += red[w][lane];
    }
    // 16x16 layout: lane holds column (lane & 15), rows 4*(lane/16) + r.
    const int n = n0 + (lane & 15);
    if (n >= p.n) {
        return;
    }
    const EpiCol c = epi_col(p.ep, n);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = 4 * (lane >> 4) + r;
        if (m < p.m) {
            const EpiRow row = epi_row(p.ep, m);
            char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
            epi_store(p.ep, row, c, acc[r], crow, n);
        }
    }
}

// ---------------------------------------------------------------------------
// Skinny GEMM, 4 < M <= 16, B k-contiguous ([N][K], 16-byte aligned rows):
// one block per 16 rows of B (16 output columns), its W waves splitting K in
// 1 KiB pieces (wave w: k = 1024 w + 1024 W j). Each wave moves its 16 rows x
// 1 KiB of B into LDS with one direct-to-LDS load per row (1 KiB of whole
// cache lines per instruction, where the register-fed GEMV's fragment loads
// fetch 64-byte half lines) while its A fragments (16 rows x 1 KiB, from L2)
// go to registers; then 16 v_mfma_i32_16x16x64_i8 read B back from LDS (row
// pitch 1040 bytes: a fragment read's 16 rows fall in distinct bank groups).
// K tails: A reads zero past K; B reads past the block's last row come back
// zero from the buffer's range check. Bound: HBM (the B stream).
// ---------------------------------------------------------------------------
template <int W>
__global__ __launch_bounds__(W * 64) void gemv_i8_lds(GemmI8Kern p)
{
    constexpr int KW = 1024;                         // k bytes per wave piece
    constexpr int PITCH = KW + 16;                   // LDS row pitch
    constexpr int T = KW / 64;                       // MFMAs per piece
    __shared__ __attribute__((aligned(16))) int8_t stage[W][16 * PITCH];
    __shared__ v4i red[W - 1][64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int n0 = blockIdx.x * 16;
    const int rows = min(16, p.n - n0);
    const int64_t span = (int64_t)(rows - 1) * p.ldb + p.k;
#if __HIP_DEVICE_COMPILE__
    const BufRsrc rs = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.b + (int64_t)n0 * p.ldb), 0,
                                                         (int)span, 0x00020000);
#else
    (void)span;
    const BufRsrc rs{};
#endif
    const int arow = lane & 15;
    const bool a_live = arow < p.m;
    const int8_t* a_row = p.a + (int64_t)(a_live ? arow : 0) * p.lda;
    const int kq = (lane >> 4) * 16;
    int8_t* st = stage[wave];
    // A plain int32 destination (no zero-point terms) takes only the bias and
    // Relu; its bias word is loaded now, off the output pass's critical path
    const bool plain32 = p.ep.out_kind == NNOPS_OUT_S32 && !p.ep.compensate;
    const int n_out = n0 + (lane & 15);
    int32_t bias_n = 0;
    if (plain32 && wave == 0 && p.ep.bias != nullptr && n_out < p.n) {
        bias_n = p.ep.bias[n_out];
    }
    // the general output pass's column and row constants, likewise up front
    EpiCol col{};
    EpiRow rws[4]{};
    if (!plain32 && wave == 0 && n_out < p.n) {
        col = epi_col(p.ep, n_out);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            rws[r] = epi_row(p.ep, min(4 * (lane >> 4) + r, p.m - 1));
        }
    }

    v4i acc = {0, 0, 0, 0};
    for (int kb = wave * KW; kb < p.k; kb += W * KW) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            buffer_load_lds16<2>(rs, st + r * PITCH, (int)((int64_t)r * p.ldb) + kb + lane * 16, 0);
        }
        v4i fa[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            fa[t] = a_live ? load16_a<true>(a_row, kb + 64 * t + kq, p.k, p.a_xor) : v4i{0, 0, 0, 0};
        }
        wait_vmcnt<0>();
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const v4i fb = *reinterpret_cast<const v4i*>(st + arow * PITCH + 64 * t + kq);
            acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[t], fb, acc, 0, 0, 0);
        }
        // the next piece's loads overwrite this stage: its reads must be done
        __builtin_amdgcn_s_waitcnt(0xc07f);
        asm volatile("" ::: "memory");
    }

    if (wave > 0) {
        red[wave - 1][lane] = acc;
    }
    __syncthreads();
    if (wave != 0) {
        return;
    }
#pragma unroll
    for (int w = 0; w < W - 1; ++w) {
        acc += red[w][lane];
    }
    // 16x16 layout: lane holds column (lane & 15), rows 4*(lane/16) + r.
    const int n = n_out;
    if (n >= p.n) {
        return;
    }
    if (plain32) {
        const bool relu = p.ep.act == NNOPS_ACT_RELU;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = 4 * (lane >> 4) + r;
            if (m < p.m) {
                const int32_t v = acc[r] + bias_n;
                reinterpret_cast<int32_t*>(static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes)[n] =
                    (relu && v < 0) ? 0 : v;
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = 4 * (lane >> 4) + r;
        if (m < p.m) {
            char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
            epi_store(p.ep, rws[r], col, acc[r], crow, n);
        }
    }
}

// ---------------------------------------------------------------------------
// Row GEMV, M <= 4, B k-contiguous ([N][K]). A wave owns R consecutive rows of
// B; lane l reads the 16-byte chunks k = 16*(l + 64c), so every wave load
// instruction streams 1 KiB of one row contiguously (non-temporal: the
// weights are read once). Dots on v_dot4_i32_i8, A kept in registers per
// 4 KiB k block, cross-lane sum at the end. Bound: HBM.
// ---------------------------------------------------------------------------
__device__ __forceinline__ int wave_sum(int v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        v += __shfl_xor(v, off, 64);
    }
    return v;
}

template <int MT, int R, bool FLIP, int WPB = 4, int SPLIT = 1>
__global__ __launch_bounds__(WPB * 64) void gemv_i8_rows(GemmI8Kern p)
{
    // SPLIT > 1: SPLIT consecutive waves share one row (R = 1), each taking an
    // interleaved 1/SPLIT of its 1 KiB k chunks; partial sums meet in LDS.
    static_assert(SPLIT == 1 || R == 1, "split rows are single rows");
    static_assert(WPB % SPLIT == 0, "a row's waves share a block");
    constexpr int C = 4;                       // 16-byte chunks per lane per row per k block
    __shared__ int part[SPLIT > 1 ? WPB : 1][R * MT];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int sub = wave % SPLIT;
    const int n0 = ((blockIdx.x * WPB + wave) / SPLIT) * R;
    const bool row_live = n0 < p.n;
    const int8_t* brow[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        brow[r] = p.b + (int64_t)min(n0 + r, p.n - 1) * p.ldb;
    }
    int acc[R][MT];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            acc[r][m] = 0;
        }
    }
    for (int kb = 0; kb < p.k; kb += 64 * 16 * C) {
        v4i w[R][C], a[MT][C];
        // weights first (the HBM stream is the long pole), then A from cache
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int k = kb + (lane + 64 * c) * 16;
            const bool live = row_live && (c % SPLIT == sub) && k < p.k;
#pragma unroll
            for (int r = 0; r < R; ++r) {
                w[r][c] = live ? __builtin_nontemporal_load(reinterpret_cast<const v4i*>(brow[r] + k))
                               : v4i{0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
            const int k = kb + (lane + 64 * c) * 16;
            const bool live = row_live && (c % SPLIT == sub) && k < p.k;
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int mm = min(m, p.m - 1);
                v4i x = live ? *reinterpret_cast<const v4i*>(p.a + (int64_t)mm * p.lda + k) : v4i{0, 0, 0, 0};
                if constexpr (FLIP) {
                    x = flip_u8(x, p.a_xor, live);
                }
                a[m][c] = x;
            }
        }
#pragma unroll
        for (int c = 0; c < C; ++c) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
#pragma unroll
                for (int m = 0; m < MT; ++m) {
                    int s = acc[r][m];
                    s = __builtin_amdgcn_sdot4(a[m][c].x, w[r][c].x, s, false);
                    s = __builtin_amdgcn_sdot4(a[m][c].y, w[r][c].y, s, false);
                    s = __builtin_amdgcn_sdot4(a[m][c].z, w[r][c].z, s, false);
                    s = __builtin_amdgcn_sdot4(a[m][c].w, w[r][c].w, s, false);
                    acc[r][m] = s;
                }
            }
        }
    }
    int mine = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int m = 0; m < MT; ++m) {
            const int v = wave_sum(acc[r][m]);
            if (lane == r * MT + m) {
                mine = v;
            }
        }
    }
    if constexpr (SPLIT > 1) {
        if (lane < R * MT) {
            part[wave][lane] = mine;
        }
        __syncthreads();
        if (sub != 0) {
            return;
        }
        if (lane < R * MT) {
#pragma unroll
            for (int q = 1; q < SPLIT; ++q) {
                mine += part[wave + q][lane];
            }
        }
    }
    if (row_live && lane < R * MT) {
        const int r = lane / MT, m = lane % MT;
        const int n = n0 + r;
        if (n < p.n && m < p.m) {
            char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
            epi_store(p.ep, epi_row(p.ep, m), epi_col(p.ep, n), mine, crow, n);
        }
    }
}

// ---------------------------------------------------------------------------
// Column GEMV, M <= 16, B n-contiguous ([K][N], the MatMul weight without
// transpose_b), consumed in place. Lane l of a wave owns CPL consecutive
// columns (the launch takes CPL = 4: one 4-byte load per row; the template
// also takes 16), so every wave load streams 64 * CPL contiguous bytes of one row. Four
// rows k..k+3 are transposed in registers (two v_perm per column) into one
// dword of 4 k-bytes per column, which v_dot4 multiplies with A[m][k..k+3]
// read through the scalar cache (A is uniform across the wave). Split s of S
// takes k-quads [s Q / S, (s + 1) Q / S) of a column chunk, and the W waves of
// its workgroup equal parts of that range, summed by LDS atomic adds (W = 4
// or 8); the workgroups write raw
// int32 partials that gemm_i8_reduce sums and passes through the output pass.
// (Meeting the splits inside the kernel, the last-arriving split summing the
// others through device-coherent loads, measured slower: the handoff costs
// more than the second launch.) Bound: HBM.
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(4))) int32_t* ScalarI32Ptr;

struct KnSplit {
    int chunks;       // column chunks of 64 * CPL
};

// 4 rows (one dword each, byte c = column c) -> 4 column dwords (byte i = row i)
__device__ __forceinline__ void transpose4x4_bytes(uint32_t r0, uint32_t r1, uint32_t r2, uint32_t r3,
                                                   uint32_t (&col)[4])
{
    const uint32_t t0 = __builtin_amdgcn_perm(r1, r0, 0x05010400u);   // r0b0 r1b0 r0b1 r1b1
    const uint32_t t1 = __builtin_amdgcn_perm(r3, r2, 0x05010400u);   // r2b0 r3b0 r2b1 r3b1
    const uint32_t t2 = __builtin_amdgcn_perm(r1, r0, 0x07030602u);   // r0b2 r1b2 r0b3 r1b3
    const uint32_t t3 = __builtin_amdgcn_perm(r3, r2, 0x07030602u);
    col[0] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
    col[1] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
    col[2] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
    col[3] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
}

// ---------------------------------------------------------------------------
// Skinny GEMM over a [K,N] B in place, M <= 16 (A rows padded to 16):
// v_mfma_i32_16x16x64_i8 with each B fragment built by two transposed LDS
// reads (lds_read_tr8) from k rows staged as they lie in memory. A workgroup
// of 4 waves owns a group of 16 CB columns and one of sk.splits K ranges;
// wave w streams its own contiguous run of 64-row steps (16 CB bytes per
// row, whole cache lines, in 1 KiB DMA instructions) through an NSW-slot
// ring of its own, with the step's A fragments (16 bytes per lane, from L2)
// loaded beside it. The waves meet in LDS. With one K range the workgroup
// runs the output pass; with several it writes its int32 partials
// [split][M][N] (device-coherent sc1 stores), then its flag (the launch
// epoch), then reads every split's flag: a workgroup that finds them all set
// sums the column group's splits in split order and runs the output pass --
// the last to arrive always does, and one that reads the flags at the same
// moment writes the same bits -- then clears the flags, so a replayed graph
// (same epoch) finds them clear. No second launch.
// ---------------------------------------------------------------------------
template <int NSW, int CB>
__global__ __launch_bounds__(256) void gemv_i8_kn_tr(GemmI8Kern p, RingSplit sk, int groups)
{
    constexpr int CW = 16 * CB;             // columns per workgroup: CB blocks of 16
    constexpr int STEP = 64 * CW;           // bytes per 64-row step
    constexpr int Q = STEP / 1024;          // DMA instructions per step
    constexpr int RPQ = 1024 / CW;          // rows per DMA instruction
    constexpr int L = Q + 1;                // vector-memory ops per step: the DMA + 1 A load
    static_assert(CB == 8, "128-byte row segments (lds_tr8_ready ties 8 column blocks)");
    static_assert(NSW >= 1 && (NSW - 1) * L < 64, "vmcnt range");
    __shared__ __attribute__((aligned(1024))) int8_t ring[4][NSW][STEP];
    static_assert(3 * CB * 64 * 16 <= 4 * NSW * STEP, "the waves' partial tiles fit the ring");
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int cg = blockIdx.x % groups, sp = blockIdx.x / groups;
    const int n0 = cg * CW;
    const int T = p.k / 64;
    const int s0 = (int)((int64_t)T * sp / sk.splits), s1 = (int)((int64_t)T * (sp + 1) / sk.splits);
    const int w0 = s0 + (s1 - s0) * wave / 4, w1 = s0 + (s1 - s0) * (wave + 1) / 4;
    const int nst = w1 - w0;

    // slot of 16-byte chunk c in k row r: the transposed reads of 32 lanes
    // (rows r0..r0+7 and r0+16..r0+23 of one chunk) fall in 16 distinct
    // 16-byte bank groups (128-byte rows: two rows per 256-byte bank row)
    auto swz = [](int r) {
        return CB == 8 ? ((((r >> 1) & 3) << 1) | ((r >> 4) & 1)) : (((r & 7) << 1) | ((r >> 4) & 1));
    };
    // the descriptor ends at B's last byte: chunks past column N of the last
    // row read 0 (earlier rows' read the next row: never stored)
    const BufRsrc rsb = buffer_rsrc(p.b + n0, (int)((int64_t)(p.k - 1) * p.ldb + (p.n - n0)));
    int b_off[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int r = q * RPQ + lane / CB;
        b_off[q] = r * (int)p.ldb + (((lane % CB) ^ swz(r)) << 4);
    }
    const int arow = lane & 15;
    const int8_t* a_row = p.a + (int64_t)min(arow, p.m - 1) * p.lda;
    const int kq = 16 * (lane >> 4);
    v4i fa[NSW];
    auto issue = [&](int st, int u) {
        int8_t* dst = ring[wave][u];
        fa[u] = *reinterpret_cast<const v4i*>(a_row + st * 64 + kq);
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            buffer_load_lds16<2>(rsb, dst + q * 1024, b_off[q], st * 64 * (int)p.ldb);
        }
    };
    // B fragment of column block cb (16 columns) from a staged step: lane
    // (group g, index i) reads k row 16 g + (i >> 1) (+8), columns 16 cb +
    // 8 (i & 1); lane l receives column 16 cb + (l & 15) at k 16 g + 0..15
    const int tr_k = 16 * (lane >> 4) + ((lane & 15) >> 1);
    const int tr_b = 8 * (lane & 1);
    v4i acc[CB];
#pragma unroll
    for (int cb = 0; cb < CB; ++cb) {
        acc[cb] = v4i{0, 0, 0, 0};
    }
#pragma unroll
    for (int u = 0; u < NSW; ++u) {
        if (u < nst) {
            issue(w0 + u, u);
        }
    }
    for (int t = 0; t < nst; t += NSW) {
#pragma unroll
        for (int u = 0; u < NSW; ++u) {
            if (t + u < nst) {
                const int ahead = min(nst - 1 - (t + u), NSW - 1);
                if (ahead <= 0) {
                    wait_vmcnt<0>();
                } else if (NSW >= 2 && ahead == 1) {
                    wait_vmcnt<(NSW >= 2 ? L : 0)>();
                } else if (NSW >= 3 && ahead == 2) {
                    wait_vmcnt<(NSW >= 3 ? 2 * L : 0)>();
                } else {
                    wait_vmcnt<(NSW >= 4 ? 3 * L : 0)>();
                }
                asm volatile("" ::: "memory");
                const int8_t* st = ring[wave][u];
                v2i lo[CB], hi[CB];
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    // the column block is chunk cb of the staged row
                    const int k0 = tr_k;
                    lo[cb] = lds_read_tr8_asm(st + k0 * CW + ((cb ^ swz(k0)) << 4) + tr_b);
                    hi[cb] = lds_read_tr8_asm(st + (k0 + 8) * CW + ((cb ^ swz(k0 + 8)) << 4) + tr_b);
                }
                lds_tr8_ready(lo, hi);
#pragma unroll
                for (int cb = 0; cb < CB; ++cb) {
                    acc[cb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(fa[u], v4i{lo[cb].x, lo[cb].y, hi[cb].x, hi[cb].y},
                                                                   acc[cb], 0, 0, 0);
                }
                // the slot's reads are done before the next step's DMA reuses it
                __builtin_amdgcn_s_waitcnt(0xc07f);
                asm volatile("" ::: "memory");
                if (t + u + NSW < nst) {
                    issue(w0 + t + u + NSW, u);
                }
            }
        }
    }
    __syncthreads();
    v4i* red = reinterpret_cast<v4i*>(&ring[0][0][0]);
    if (wave > 0) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            red[((wave - 1) * CB + cb) * 64 + lane] = acc[cb];
        }
    }
    __syncthreads();
    // 16x16 layout: lane holds column (lane & 15) of the block, rows 4 (lane >> 4) + r
    if (sk.splits == 1) {
        if (wave != 0) {
            return;
        }
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const v4i v = acc[cb] + red[(0 * CB + cb) * 64 + lane] + red[(1 * CB + cb) * 64 + lane] +
                          red[(2 * CB + cb) * 64 + lane];
            const int n = n0 + 16 * cb + (lane & 15);
            if (n < p.n) {
                const EpiCol c = epi_col(p.ep, n);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int m = 4 * (lane >> 4) + r;
                    if (m < p.m) {
                        epi_store(p.ep, epi_row(p.ep, m), c, v[r],
                                  static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes, n);
                    }
                }
            }
        }
        return;
    }
    // the split's partials (byte offsets fit 32 bits: splits * M * N * 4 <
    // 2^31, checked by the plan), then its flag
    const BufRsrc rpart = buffer_rsrc(sk.part);
    const BufRsrc rflag = buffer_rsrc(sk.flag + (int64_t)cg * sk.splits);
    __shared__ int s_all;
    if (wave == 0) {
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
            const v4i v = acc[cb] + red[(0 * CB + cb) * 64 + lane] + red[(1 * CB + cb) * 64 + lane] +
                          red[(2 * CB + cb) * 64 + lane];
            const int n = n0 + 16 * cb + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int m = 4 * (lane >> 4) + r;
                if (n < p.n && m < p.m) {
                    buffer_store4_sc1(rpart, v[r], ((sp * p.m + m) * p.n + n) * 4);
                }
            }
        }
        wait_vmcnt<0>();
        if (lane == 0) {
            buffer_store8_sc1(rflag, sk.epoch, sp * 8);
        }
        wait_vmcnt<0>();
        bool all = true;
        for (int f0 = 0; f0 < sk.splits; f0 += 64) {
            const uint64_t f = f0 + lane < sk.splits ? buffer_load8_sc1(rflag, (f0 + lane) * 8) : sk.epoch;
            all = all && __builtin_amdgcn_ballot_w64(f != sk.epoch) == 0;
        }
        if (lane == 0) {
            s_all = all;
        }
    }
    __syncthreads();
    if (!s_all) {
        return;
    }
    // every split has published: 4 consecutive columns of one row per
    // thread, the splits summed in split order (exact: integers)
    const int q = threadIdx.x & (CW / 4 - 1);
    const int n = n0 + 4 * q;
    if (n < p.n) {
        const EpiCol c[4] = {epi_col(p.ep, n), epi_col(p.ep, n + 1), epi_col(p.ep, n + 2), epi_col(p.ep, n + 3)};
        const bool plain32 = p.ep.out_kind == NNOPS_OUT_S32 && !p.ep.compensate;
        for (int m = threadIdx.x / (CW / 4); m < p.m; m += 256 / (CW / 4)) {
            // four splits' loads in flight at a time
            v4i sum = v4i{0, 0, 0, 0};
            int sp2 = 0;
            for (; sp2 + 3 < sk.splits; sp2 += 4) {
                const int o = ((sp2 * p.m + m) * p.n + n) * 4, st = p.m * p.n * 4;
                const v4i x0 = buffer_load16_sc1(rpart, o), x1 = buffer_load16_sc1(rpart, o + st);
                const v4i x2 = buffer_load16_sc1(rpart, o + 2 * st), x3 = buffer_load16_sc1(rpart, o + 3 * st);
                sum += (x0 + x1) + (x2 + x3);
            }
            for (; sp2 < sk.splits; ++sp2) {
                sum += buffer_load16_sc1(rpart, ((sp2 * p.m + m) * p.n + n) * 4);
            }
            char* crow = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes;
            if (plain32) {
                // an int32 destination without zero-point terms: bias and Relu
                const bool relu = p.ep.act == NNOPS_ACT_RELU;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int32_t v = sum[e] + c[e].bias;
                    reinterpret_cast<int32_t*>(crow)[n + e] = (relu && v < 0) ? 0 : v;
                }
                continue;
            }
            const EpiRow row = epi_row(p.ep, m);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                epi_store(p.ep, row, c[e], sum[e], crow, n + e);
            }
        }
    }
    for (int f = (int)threadIdx.x; f < sk.splits; f += (int)blockDim.x) {
        buffer_store8_sc1(rflag, 0ull, f * 8);
    }
}

template <int MT, int CPL, int W, int U>
__global__ __launch_bounds__(W * 64) void gemv_i8_kn(GemmI8Kern p, RingSplit sk, KnSplit ks)
{
    constexpr int D = CPL / 4;                   // dwords per lane per row
    // U k-quads per batch (4 U rows in flight); the waves' sums meet in one
    // LDS array through integer atomic adds (exact in any order)
    __shared__ int32_t red[MT * CPL][64];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = threadIdx.x; i < MT * CPL * 64; i += W * 64) {
        (&red[0][0])[i] = 0;
    }
    const int chunk = blockIdx.x % ks.chunks;
    const int split = blockIdx.x / ks.chunks;
    const int n = chunk * 64 * CPL + lane * CPL;
    const bool live = n < p.n;
    // split s of S takes k-quads [s Q / S, (s + 1) Q / S) and its W waves
    // equal parts of that range, so any S fills the CUs evenly
    const int nquad = p.k / 4;
    const int qs0 = (int)((int64_t)split * nquad / sk.splits);
    const int qs1 = (int)((int64_t)(split + 1) * nquad / sk.splits);
    const int qw0 = qs0 + (int)((int64_t)wave * (qs1 - qs0) / W);
    const int qw1 = qs0 + (int)((int64_t)(wave + 1) * (qs1 - qs0) / W);

    int32_t acc[MT][CPL];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            acc[m][c] = 0;
        }
    }
    const int8_t* bcol = p.b + (live ? n : 0);
    for (int q = qw0; q < qw1; q += U) {
        const int nq = min(U, qw1 - q);       // wave-uniform
        const int k = 4 * q;
        uint32_t rows[4 * U][D];
#pragma unroll
        for (int r = 0; r < 4 * U; ++r) {
            const int8_t* src = bcol + (int64_t)(k + r) * p.ldb;
            if (r < 4 * nq) {
                if constexpr (D == 4) {
                    const v4i v = __builtin_nontemporal_load(reinterpret_cast<const v4i*>(src));
#pragma unroll
                    for (int d = 0; d < 4; ++d) {
                        rows[r][d] = (uint32_t)v[d];
                    }
                } else {
                    rows[r][0] = __builtin_nontemporal_load(reinterpret_cast<const uint32_t*>(src));
                }
            } else {
#pragma unroll
                for (int d = 0; d < D; ++d) {
                    rows[r][d] = 0u;
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= nq) {
                break;
            }
            int32_t aq[MT];
#pragma unroll
            for (int m = 0; m < MT; ++m) {
                const int mm = m < p.m ? m : 0;
                aq[m] = *reinterpret_cast<ScalarI32Ptr>((uintptr_t)(p.a + (int64_t)mm * p.lda + k + 4 * u));
            }
#pragma unroll
            for (int d = 0; d < D; ++d) {
                uint32_t col[4];
                transpose4x4_bytes(rows[4 * u][d], rows[4 * u + 1][d], rows[4 * u + 2][d], rows[4 * u + 3][d], col);
#pragma unroll
                for (int m = 0; m < MT; ++m) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        acc[m][4 * d + c] = __builtin_amdgcn_sdot4(aq[m], (int)col[c], acc[m][4 * d + c], false);
                    }
                }
            }
        }
    }
    __syncthreads();   // red is cleared
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            if (m < p.m) {
                atomicAdd(&red[m * CPL + c][lane], acc[m][c]);
            }
        }
    }
    __syncthreads();
    // Thread t takes chunk column r = t % (64 CPL) (lane r / CPL, element
    // r % CPL) of row t / (64 CPL), so consecutive threads store consecutive
    // int32 partials.
    const int nc0 = chunk * 64 * CPL;
    int32_t* part = sk.part + (int64_t)split * p.m * p.n;
    for (int idx = threadIdx.x; idx < MT * CPL * 64; idx += W * 64) {
        const int m = idx / (CPL * 64);
        const int r = idx % (CPL * 64);
        if (m < p.m && nc0 + r < p.n) {
            part[(int64_t)m * p.n + nc0 + r] = red[m * CPL + r % CPL][r / CPL];
        }
    }
}

// ---------------------------------------------------------------------------
// Prepasses
// ---------------------------------------------------------------------------
// dst[c][r] = src[r][c] for r < R, c < C; dst columns r in [R, Rp) are zeroed.
// The same transpose in 256-row x 64-column tiles with 16-byte accesses on
// both sides (source rows, pitch, destination and its pitch 16-byte aligned,
// Rp % 16 == 0): each thread loads four 16-byte row pieces into LDS (row
// pitch 17 dwords), then reads a 16-row x 4-column block as 16 dwords,
// transposes it in registers (v_perm, 4 x 4 bytes at a time) and stores four
// 16-byte destination pieces (the byte-wise kernel below, kept for unaligned
// operands, moves one byte per load and store).
__global__ __launch_bounds__(256) void transpose_i8_v(const int8_t* src, int64_t lds_, int R, int C,
                                                      int8_t* dst, int64_t ldd, int Rp)
{
    constexpr int TR = 256, TC = 64, P = TC / 4 + 1;   // rows, columns, LDS pitch in dwords
    __shared__ uint32_t tile[TR * P];
    const int r0 = blockIdx.y * TR;
    const int c0 = blockIdx.x * TC;
    const int t = threadIdx.x;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int idx = q * 256 + t;
        const int row = idx >> 2, seg = idx & 3;
        const int r = r0 + row, c = c0 + 16 * seg;
        v4i v = v4i{0, 0, 0, 0};
        if (r < R && c < C) {
            const int8_t* sp = src + (int64_t)r * lds_ + c;
            if (c + 16 <= C) {
                v = *reinterpret_cast<const v4i*>(sp);
            } else {
                uint32_t w[4] = {0u, 0u, 0u, 0u};
                for (int b = 0; b < C - c; ++b) {
                    w[b >> 2] |= (uint32_t)(uint8_t)sp[b] << (8 * (b & 3));
                }
                v = v4i{(int)w[0], (int)w[1], (int)w[2], (int)w[3]};
            }
        }
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            tile[row * P + 4 * seg + d] = (uint32_t)v[d];
        }
    }
    __syncthreads();
    const int c4 = t & 15, r16 = t >> 4;
    uint32_t w[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        w[i] = tile[(16 * r16 + i) * P + c4];
    }
    uint32_t col[4][4];   // [column j][row quad g]
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        uint32_t cq[4];
        transpose4x4_bytes(w[4 * g], w[4 * g + 1], w[4 * g + 2], w[4 * g + 3], cq);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            col[j][g] = cq[j];
        }
    }
    const int r = r0 + 16 * r16;
    if (r >= Rp) {
        return;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = c0 + 4 * c4 + j;
        if (c < C) {
            *reinterpret_cast<v4i*>(dst + (int64_t)c * ldd + r) =
                v4i{(int)col[j][0], (int)col[j][1], (int)col[j][2], (int)col[j][3]};
        }
    }
}

__global__ __launch_bounds__(256) void transpose_i8(const int8_t* src, int64_t lds_, int R, int C,
                                                   int8_t* dst, int64_t ldd, int Rp)
{
    __shared__ int8_t tile[64][65];
    const int r0 = blockIdx.y * 64;
    const int c0 = blockIdx.x * 64;
    const int tx = threadIdx.x & 63;
    const int ty = threadIdx.x >> 6;
    for (int i = ty; i < 64; i += 4) {
        const int r = r0 + i, c = c0 + tx;
        tile[i][tx] = (r < R && c < C) ? src[(int64_t)r * lds_ + c] : (int8_t)0;
    }
    __syncthreads();
    for (int i = ty; i < 64; i += 4) {
        const int c = c0 + i, r = r0 + tx;
        if (c < C && r < Rp) {
            dst[(int64_t)c * ldd + r] = tile[tx][i];
        }
    }
}

// dst[c][r] = src[r][c] (r < R, c < C; columns r in [R, Rp) zeroed): the
// 16-byte tiled kernel where its alignment holds, else the byte-wise one.
void launch_transpose_i8(const int8_t* src, int64_t lds_, int R, int C, int8_t* dst, int64_t ldd, int Rp,
                         hipStream_t s)
{
    if (((uintptr_t)src % 16) == 0 && lds_ % 16 == 0 && ((uintptr_t)dst % 16) == 0 && ldd % 16 == 0 &&
        Rp % 16 == 0) {
        const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((Rp + 255) / 256));
        NNOPS_LAUNCH(transpose_i8_v, grid, dim3(256), 0, s, src, lds_, R, C, dst, ldd, Rp);
    } else {
        const dim3 grid((unsigned)((C + 63) / 64), (unsigned)((Rp + 63) / 64));
        NNOPS_LAUNCH(transpose_i8, grid, dim3(256), 0, s, src, lds_, R, C, dst, ldd, Rp);
    }
}

// out[r] = sum_k row r (u8 reads unsigned). One wave per row.
__global__ __launch_bounds__(256) void rowsum_i8(const int8_t* src, int64_t ld, int R, int K, int u8,
                                                int32_t* out)
{
    const int lane = threadIdx.x & 63;
    const int r = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (r >= R) {
        return;
    }
    const int8_t* row = src + (int64_t)r * ld;
    int32_t s = 0;
    for (int k = lane; k < K; k += 64) {
        s += u8 ? (int32_t)(uint8_t)row[k] : (int32_t)row[k];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_xor(s, off, 64);
    }
    if (lane == 0) {
        out[r] = s;
    }
}

// Row copy into a wider, zero-padded pitch (the prepack of an [N,K] B):
// 16 bytes per thread where source and destination allow it.
__global__ __launch_bounds__(256) void pad_rows_i8(const int8_t* src, int64_t lds_, int R, int C,
                                                  int8_t* dst, int64_t ldd)
{
    const int64_t chunks = ldd / 16;
    const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (t >= (int64_t)R * chunks) {
        return;
    }
    const int r = (int)(t / chunks);
    const int c0 = (int)(t - (int64_t)r * chunks) * 16;
    const int8_t* s = src + (int64_t)r * lds_;
    int8_t v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        v[i] = c0 + i < C ? s[c0 + i] : (int8_t)0;
    }
    int4 o;
    __builtin_memcpy(&o, v, 16);
    *reinterpret_cast<int4*>(dst + (int64_t)r * ldd + c0) = o;
}

// ---------------------------------------------------------------------------
// Host side: workspace plan and dispatch.
// ---------------------------------------------------------------------------
inline int64_t round16(int64_t x) { return (x + 15) / 16 * 16; }

// Column GEMV plan ([K,N] B consumed in place, M <= 16).
struct KnPlan {
    int cpl = 0;            // columns per lane (0: not taken)
    int w = 0;              // waves per workgroup
    int chunks = 0, splits = 0;
    bool tr = false;        // gemv_i8_kn_tr (chunks: its 128-column groups)
};

inline int kn_mt(int64_t m) { return m <= 1 ? 1 : m <= 2 ? 2 : m <= 4 ? 4 : m <= 8 ? 8 : 16; }

struct WsPlan {
    size_t r_a = 0, r_b = 0, a_t = 0, b_t = 0, part = 0, flag = 0, total = 0;
    size_t full = 0;        // the total of the plan with all the room it would take (choose_plan)
    int64_t kp = 0;
    RingPlan ring;
    KnPlan kn;
};


// M <= 16 with a [K,N] B: 16-byte (M <= 2) or 4-byte column groups per lane,
// K % 16 == 0, dword-aligned A rows (scalar loads), no term that needs the
// column sums of B (u8 A, A zero points). About 512 workgroups of 8 (or 4)
// waves, row ranges a multiple of 16.
KnPlan plan_kn(const NnopsGemmI8Args& g)
{
    KnPlan r;
    if (g.trans_b || g.trans_a || g.m > 16 || g.k % 16 != 0 || g.a_u8 || g.zp_a != nullptr || g.zp_a_scalar != 0) {
        return r;
    }
    // (8 columns per lane with 32 rows in flight measured slower for
    // 4 <= M <= 16: 17.1 / 32.1 us against 14.8 / 28.3 at M = 4 / 16)
    // 3 <= M <= 16, 64-row steps, 16-byte rows: the transposed-read MFMA
    // kernel, K split so about two workgroups per CU stream at once
    // (measured at config 3, N = 11008, call totals with the reduce: 128-byte
    // row segments and ~512 workgroups 15.2 / 16.6 us at M = 4 / 16; 256-byte
    // segments 18.7 / 20.0 (256 workgroups) and 21.8 / 27.0 (512); no K split
    // (86 workgroups) 37.8 / 38.5; at M = 1..2 the column GEMV stays faster,
    // 13.8 against 14.9 us). With the splits meeting in the launch: 14.6 /
    // 16.5 us at 5 splits, the same at 4, 16.6 / 18.8 at 3, 19.7 / 21.8 at 6
    // (516 workgroups: a second round), 17.3 / 18.8 at 8.
    if (g.m >= 3 && g.k % 64 == 0 && g.n % 4 == 0 && aligned16(g.b, g.ldb) &&
        aligned16(static_cast<const int8_t*>(g.a), g.lda) && g.k * g.ldb + g.n < (int64_t)INT32_MAX) {
        r.tr = true;
        r.cpl = 8;          // column blocks of 16 per workgroup
        r.w = 4;
        r.chunks = (int)((g.n + 127) / 128);
        r.splits = (int)std::max<int64_t>(1, std::min<int64_t>(512 / r.chunks, g.k / 64 / 4));
        if ((int64_t)r.splits * g.m * g.n * 4 >= INT32_MAX) {
            return KnPlan{};
        }
        return r;
    }
    const int cpl = 4;
    if (g.n % cpl != 0 || g.n % 4 != 0 || ((uintptr_t)g.b % cpl) != 0 || (g.ldb % cpl) != 0 ||
        ((uintptr_t)g.a % 4) != 0 || (g.lda % 4) != 0) {
        return r;
    }
    const int mt = kn_mt(g.m);
    r.cpl = cpl;
    r.chunks = (int)((g.n + 64 * cpl - 1) / (64 * cpl));
    // 256-column chunks (4 columns per lane: every wave load is 256 bytes of
    // one row, two whole lines). K is split so the workgroups fill the CUs
    // about twice, each split at least 16 rows per wave. (Config 3, M = 1:
    // 43 chunks x 11 splits, 13.0 us per call; 1024-column chunks of 16-byte
    // lanes, 11 chunks x 23 splits of 16 waves, ran 13.6 at M = 1 and 15.1
    // against 13.5 at M = 2.)
    r.w = (mt * cpl >= 64) ? 4 : 8;
    const int per_cu = 2;
    const int64_t max_splits = std::max<int64_t>(1, g.k / (16 * r.w));
    r.splits = (int)std::min<int64_t>(max_splits, std::max(1, 256 * per_cu / r.chunks));
    if ((int64_t)r.splits * g.m * g.n * 4 >= INT32_MAX) {
        return KnPlan{};    // the partials' 32-bit buffer offsets
    }
    return r;
}


// Shapes that gemm_i8_mfma, which writes no partials, also takes at a tolerable
// rate: they run without the ring where the workspace has no room for it.
inline bool ring_optional(const NnopsGemmI8Args& g) { return g.m < 64 || g.k % 64 != 0 || g.n % 4 != 0; }

// How a call is planned: with as many K splits as `room` bytes hold, or by its
// rows alone (plan_ring_by_rows), or without the ring.
struct PlanFor {
    size_t room = SIZE_MAX;
    bool by_rows = false;
    bool ring = true;
};

WsPlan plan_workspace(const NnopsGemmI8Args& g, const PlanFor& f = PlanFor{})
{
    WsPlan w;
    size_t off = 0;
    w.kp = round16(g.k);
    w.r_a = off; off += align_up((size_t)g.m * 4);
    w.r_b = off; off += align_up((size_t)g.n * 4);
    const int8_t* a = static_cast<const int8_t*>(g.a);
    const int8_t* b = g.b;
    int64_t lda = g.lda, ldb = g.ldb;
    if (g.trans_a) {
        w.a_t = off; off += align_up((size_t)g.m * (size_t)w.kp);
        a = nullptr;      // staged copies are 256-byte aligned with a 16-byte pitch
        lda = w.kp;
    }
    w.kn = plan_kn(g);
    if (w.kn.cpl != 0) {
        w.part = off; off += align_up((size_t)w.kn.splits * (size_t)g.m * (size_t)g.n * 4);
        if (w.kn.tr && w.kn.splits > 1) {
            // the splits' completion flags (gemv_i8_kn_tr meets them in the launch)
            w.flag = off; off += align_up((size_t)w.kn.chunks * (size_t)w.kn.splits * 8);
        }
        w.total = off;
        return w;
    }
    // a [K,N] B goes to the ring in place when it takes it and no column
    // sums of B are needed (they are summed over the staged copy's rows)
    const bool need_rb = g.a_u8 || g.zp_a != nullptr || g.zp_a_scalar != 0;
    // (from 17 rows: 24 x 11008 x 4096 s8 14.1 us on 64 x 64 tiles in four
    // splits, 52 us on gemm_i8_mfma's 64 workgroups of the whole K)
    const bool ring = g.m > 16 && f.ring;
    auto plan = [&](bool trb) {
        return f.by_rows ? plan_ring_by_rows(g, a, lda, b, ldb, trb, true)
                         : plan_ring(g, a, lda, b, ldb, trb, std::max(1, splits_in(f.room, off, g.m, g.n)), false);
    };
    if (!g.trans_b && !need_rb && ring) {
        w.ring = plan(true);
    }
    if (!g.trans_b && w.ring.mode < 0) {
        w.b_t = off; off += align_up((size_t)g.n * (size_t)w.kp);
        b = nullptr;
        ldb = w.kp;
    }
    if (!w.ring.trb && ring) {
        w.ring = plan(false);
    }
    // few rows over a short k, B's rows k-contiguous: gemm_i8_mfma before the
    // ring, where the general output pass is needed (one launch, 2.2 us and 0.3 per
    // 64 bytes of k, before the ring and its reduce: 34 x 1024 x 677 11.3 against
    // 12.2 us) and where an integer destination is written without a split (us,
    // gemm_i8_mfma / ring, s8: 17 x 256 x 1024 3.4 / 3.8, 17 x 384 x 4096 4.4 /
    // 4.5, 17 x 512 x 4096 5.2 / 5.0, 48 x 768 x 1024 5.0 / 5.2, 17 x 1024 x 1024
    // 6.8 / 6.1; an f16 one 17 x 256 x 1024 8.2 / 4.3)
    const bool short_k = w.ring.mode == RING_PART
                             ? w.ring.splits == 1 && 2.2f + 0.3f * (float)(g.k / 64) < w.ring.us
                             : w.ring.mode != RING_FP && (g.k <= 384 || (g.k < 1024 && g.n <= 1024));
    if (!f.by_rows && !w.ring.trb && g.m < 64 && short_k) {
        w.ring = RingPlan{};
    }
    if (w.ring.mode == RING_PART) {
        w.part = off; off += align_up((size_t)w.ring.splits * (size_t)g.m * (size_t)((g.n + 3) / 4) * 16);
    }
    w.total = off;
    return w;
}

// The plan that a call with ws_bytes of workspace runs on.
WsPlan choose_plan(const NnopsGemmI8Args& g, size_t ws_bytes)
{
    WsPlan w = plan_workspace(g);
    const size_t full = w.total;
    if (ws_bytes < full) {
        w = plan_workspace(g, {.room = ws_bytes});
        if (ws_bytes < w.total && ring_optional(g)) {
            w = plan_workspace(g, {.ring = false});
        }
    }
    w.full = full;
    return w;
}

template <int BM, int BN, int WM, int WN, int WPE, bool FULLK, bool ALIGNED>
void launch_gemm_epi(const GemmI8Kern& k, int epi, hipStream_t s)
{
    const int tiles = ((k.m + BM - 1) / BM) * ((k.n + BN - 1) / BN);
    const dim3 grid(tiles), block(WM * WN * 64);
    if (k.a_xor != 0u) {
        NNOPS_LAUNCH((gemm_i8_mfma<BM, BN, WM, WN, WPE, FULLK, ALIGNED, true, EPI_GENERIC>), grid, block, 0, s, k);
    } else if (epi == EPI_S8) {
        NNOPS_LAUNCH((gemm_i8_mfma<BM, BN, WM, WN, WPE, FULLK, ALIGNED, false, EPI_S8>), grid, block, 0, s, k);
    } else if (epi == EPI_S32) {
        NNOPS_LAUNCH((gemm_i8_mfma<BM, BN, WM, WN, WPE, FULLK, ALIGNED, false, EPI_S32>), grid, block, 0, s, k);
    } else {
        NNOPS_LAUNCH((gemm_i8_mfma<BM, BN, WM, WN, WPE, FULLK, ALIGNED, false, EPI_GENERIC>), grid, block, 0, s, k);
    }
}

template <int BM, int BN, int WM, int WN, int WPE>
void launch_gemm(const GemmI8Kern& k, bool aligned, bool fullk, int epi, hipStream_t s)
{
    if (fullk) {
        launch_gemm_epi<BM, BN, WM, WN, WPE, true, true>(k, epi, s);
    } else if (aligned) {
        launch_gemm_epi<BM, BN, WM, WN, WPE, false, true>(k, epi, s);
    } else {
        launch_gemm_epi<BM, BN, WM, WN, WPE, false, false>(k, epi, s);
    }
}

template <int MT>
void launch_kn_mt(const GemmI8Kern& k, const RingSplit& sk, const KnSplit& ks, int cpl, int w, hipStream_t s)
{
    const dim3 grid((unsigned)(ks.chunks * sk.splits));
    (void)cpl;                              // the plan takes 4 columns per lane
    if (w == 4) {
        NNOPS_LAUNCH((gemv_i8_kn<MT, 4, 4, 4>), grid, dim3(256), 0, s, k, sk, ks);
    } else {
        NNOPS_LAUNCH((gemv_i8_kn<MT, 4, 8, 4>), grid, dim3(512), 0, s, k, sk, ks);
    }
}

// gemm_i8_reduce_q's conditions: an s8 / u8 destination with row-uniform
// parameters and no zero-point terms, 16-byte-aligned tables and 4-byte
// aligned destination rows, an identity / Relu / GELU activation (GELU only
// with the float epilogue).
bool reduce_q_ok(const GemmI8Kern& k)
{
    const EpiParams& e = k.ep;
    return (e.out_kind == NNOPS_OUT_S8 || e.out_kind == NNOPS_OUT_U8) && !e.compensate && e.s_a == nullptr &&
           e.s_out_rows == nullptr && e.zp_out_rows == nullptr && k.n % 4 == 0 && ((uintptr_t)e.s_b % 16) == 0 &&
           ((uintptr_t)e.bias % 16) == 0 && ((uintptr_t)k.c % 4) == 0 && (k.ldc_bytes % 4) == 0 &&
           (e.act == NNOPS_ACT_NONE || e.act == NNOPS_ACT_RELU || (e.act == NNOPS_ACT_GELU && e.float_ep));
}

template <int ACT>
void launch_reduce_q_act(const GemmI8Kern& k, const RingSplit& sk, const dim3& grid, hipStream_t s)
{
    const EpiParams& e = k.ep;
    if (!e.float_ep) {
        if constexpr (ACT != NNOPS_ACT_GELU) {
            NNOPS_LAUNCH((gemm_i8_reduce_q<ACT, false, false, false>), grid, dim3(256), 0, s, k, sk);
        }
    } else if (!e.add_to) {
        NNOPS_LAUNCH((gemm_i8_reduce_q<ACT, true, false, false>), grid, dim3(256), 0, s, k, sk);
    } else if (e.residual_pre) {
        NNOPS_LAUNCH((gemm_i8_reduce_q<ACT, true, true, true>), grid, dim3(256), 0, s, k, sk);
    } else {
        NNOPS_LAUNCH((gemm_i8_reduce_q<ACT, true, true, false>), grid, dim3(256), 0, s, k, sk);
    }
}

void launch_reduce(const GemmI8Kern& k, const RingSplit& sk, hipStream_t s)
{
    const int64_t groups = (int64_t)k.m * (sk.ldp / 4);
    if (sk.splits <= 8 && reduce_q_ok(k)) {
        const dim3 grid((unsigned)((k.n / 4 + 255) / 256), (unsigned)std::min<int64_t>(k.m, 65535));
        RingSplit q = sk;
        q.row_k = k.ep.s_a_scalar / k.ep.s_out;
        q.inv_out = 1.0f / k.ep.s_out;
        if (k.ep.act == NNOPS_ACT_GELU) {
            launch_reduce_q_act<NNOPS_ACT_GELU>(k, q, grid, s);
        } else if (k.ep.act == NNOPS_ACT_RELU) {
            launch_reduce_q_act<NNOPS_ACT_RELU>(k, q, grid, s);
        } else {
            launch_reduce_q_act<NNOPS_ACT_NONE>(k, q, grid, s);
        }
        return;
    }
    if (sk.splits > 8) {
        NNOPS_LAUNCH(gemm_i8_reduce<16>, dim3((unsigned)((groups * 16 + 255) / 256)), dim3(256), 0, s, k, sk);
    } else {
        NNOPS_LAUNCH(gemm_i8_reduce<1>, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, k, sk);
    }
}

void launch_kn(const GemmI8Kern& k, const KnPlan& r, int32_t* part, uint64_t* flag, hipStream_t s)
{
    RingSplit sk{};
    sk.splits = r.splits;
    sk.kt_per = 0;
    sk.part = part;
    sk.ldp = k.n;
    if (r.tr) {
        sk.flag = flag;
        sk.epoch = next_launch_epoch();
        NNOPS_LAUNCH((gemv_i8_kn_tr<2, 8>), dim3((unsigned)(r.chunks * r.splits)), dim3(256), 0, s, k, sk,
                     r.chunks);
        return;
    }
    KnSplit ks;
    ks.chunks = r.chunks;
    switch (k.m) {
    case 1: launch_kn_mt<1>(k, sk, ks, r.cpl, r.w, s); break;
    case 2: launch_kn_mt<2>(k, sk, ks, r.cpl, r.w, s); break;
    case 3: case 4: launch_kn_mt<4>(k, sk, ks, r.cpl, r.w, s); break;
    case 5: case 6: case 7: case 8: launch_kn_mt<8>(k, sk, ks, r.cpl, r.w, s); break;
    default: launch_kn_mt<16>(k, sk, ks, r.cpl, r.w, s); break;
    }
    launch_reduce(k, sk, s);
}

void launch_ring(const GemmI8Kern& k, const RingPlan& r, int32_t* part, hipStream_t s)
{
    const RingSplit sk = ring_split(k, r, part);
    if (r.trb) {
        launch_ring_trb(k, r, sk, s);
    } else {
        launch_ring_nk(k, r, sk, s);
    }
    if (r.mode == RING_PART) {
        launch_reduce(k, sk, s);
    }
}

// Which output-pass specialisation a call can take: the fast modes need
// row-uniform parameters, no zero-point terms, half-away rounding, and a
// destination that takes packed stores for every 4-column group.
int choose_epi(const NnopsGemmI8Args& g, const EpiParams& e)
{
    if (e.compensate || g.s_out_rows != nullptr || g.zp_out_rows != nullptr || g.float_ep ||
        g.round_even || (g.n % 4) != 0 || ((uintptr_t)g.c & 15) != 0 || epi_is_fp(e)) {
        return EPI_GENERIC;
    }
    if (g.out_kind == NNOPS_OUT_S32) {
        return (g.ldc * 4) % 16 == 0 ? EPI_S32 : EPI_GENERIC;
    }
    return (g.s_a == nullptr && g.ldc % 4 == 0) ? EPI_S8 : EPI_GENERIC;
}

}  // namespace
}  // namespace nnops_amd

using namespace nnops_amd;

namespace {
int64_t prepack_pitch(int64_t k) { return (k + 127) / 128 * 128; }

// The LDS skinny GEMM: M 5..16 (M <= 4 streams faster through the row GEMV),
// a block's 16 rows within a 32-bit buffer range.
bool gemv_lds_ok(const NnopsGemmI8Args& g)
{
    return g.m > 4 && (int64_t)16 * g.ldb + g.k < (int64_t)INT32_MAX;
}
}  // namespace

extern "C" size_t nnops_hip_prepack_i8_bytes(int64_t k, int64_t n)
{
    if (k < 0 || n < 0) {
        return 0;
    }
    return align_up((size_t)n * (size_t)prepack_pitch(k)) + (size_t)n * 4;
}

extern "C" int nnops_hip_prepack_i8(const int8_t* b, int64_t k, int64_t n, int64_t ldb, int32_t trans_b,
                                    void* out, void* stream)
{
    const TimingDisarm disarm;
    if (k < 0 || n < 0 || k > INT32_MAX || n > INT32_MAX) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (k == 0 || n == 0) {
        return NNOPS_OK;
    }
    if (b == nullptr || out == nullptr || (uintptr_t)out % 256 != 0 || ldb < (trans_b ? k : n)) {
        return NNOPS_INVALID_ARGUMENT;
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int64_t kp = prepack_pitch(k);
    int8_t* rows = static_cast<int8_t*>(out);
    int32_t* sums = reinterpret_cast<int32_t*>(static_cast<char*>(out) + align_up((size_t)n * (size_t)kp));
    if (trans_b) {
        const int64_t threads = n * (kp / 16);
        NNOPS_LAUNCH(pad_rows_i8, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, s, b, ldb, (int)n,
                           (int)k, rows, kp);
    } else {
        launch_transpose_i8(b, ldb, (int)k, (int)n, rows, kp, (int)kp, s);
    }
    NNOPS_LAUNCH(rowsum_i8, dim3((unsigned)((n + 3) / 4)), dim3(256), 0, s, rows, kp, (int)n, (int)k, 0,
                       sums);
    return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
}

extern "C" size_t nnops_hip_gemm_i8_workspace_size(const NnopsGemmI8Args* g)
{
    if (g == nullptr) {
        return 0;
    }
    return plan_workspace(*g).total;
}

extern "C" int nnops_hip_gemm_i8_plan(const NnopsGemmI8Args* g, size_t ws_bytes, NnopsGemmPlan* out)
{
    if (g == nullptr || out == nullptr || g->m <= 0 || g->n <= 0 || g->k <= 0 || g->k > 65535 || g->m > INT32_MAX ||
        g->n > INT32_MAX) {
        return NNOPS_INVALID_ARGUMENT;
    }
    *out = NnopsGemmPlan{};
    const WsPlan w = choose_plan(*g, ws_bytes);
    out->workspace_bytes = w.total;
    if (w.kn.cpl == 0 && w.ring.mode >= 0) {
        out->tile_m = w.ring.bm;
        out->tile_n = w.ring.bn;
        out->splits = w.ring.splits;
        out->fused = w.ring.mode != RING_PART;
        out->short_stage = g->k % 128 != 0;
        out->in_place = w.ring.trb;
    }
    return NNOPS_OK;
}

size_t nnops_amd::gemm_i8_least_workspace(const NnopsGemmI8Args& g)
{
    return std::min(plan_workspace(g).total, plan_workspace(g, {.by_rows = true}).total);
}

namespace nnops_amd {
namespace {

// any_workspace: also with less than the least that the query's callers give.
int run_gemm_i8(const NnopsGemmI8Args* g, void* workspace, size_t ws_bytes, hipStream_t s, bool any_workspace)
{
    if (g == nullptr || g->m < 0 || g->n < 0 || g->k < 0) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (g->m == 0 || g->n == 0) {
        return NNOPS_OK;
    }
    if (g->a == nullptr || g->b == nullptr || g->c == nullptr) {
        return NNOPS_INVALID_ARGUMENT;
    }
    const bool fp_out = g->out_kind == NNOPS_OUT_F32 || g->out_kind == NNOPS_OUT_F16;
    if (g->out_kind != NNOPS_OUT_S32 && g->out_kind != NNOPS_OUT_S8 && g->out_kind != NNOPS_OUT_U8 && !fp_out) {
        return NNOPS_UNSUPPORTED;
    }
    if (g->float_ep && g->out_kind == NNOPS_OUT_S32) {
        return NNOPS_UNSUPPORTED;
    }
    if (g->act < NNOPS_ACT_NONE || g->act > NNOPS_ACT_RELU6 ||
        (!fp_out && g->act != NNOPS_ACT_NONE && g->act != NNOPS_ACT_RELU && g->act != NNOPS_ACT_GELU)) {
        return NNOPS_UNSUPPORTED;
    }
    if ((fp_out && g->bias != nullptr) || (!fp_out && g->bias_fp != nullptr)) {
        return NNOPS_INVALID_ARGUMENT;   // an f32/f16 destination takes its bias in its own type
    }
    // int32 accumulate: |sum| <= K * 128 * 255 must stay below 2^31.
    if (g->k > 65535 || g->m > INT32_MAX || g->n > INT32_MAX) {
        return NNOPS_UNSUPPORTED;
    }
    const int64_t min_lda = g->trans_a ? g->m : g->k;
    const int64_t min_ldb = g->trans_b ? g->k : g->n;
    if (g->lda < min_lda || g->ldb < min_ldb || g->ldc < g->n) {
        return NNOPS_INVALID_ARGUMENT;
    }
    const WsPlan w = choose_plan(*g, ws_bytes);
    if (!any_workspace && ws_bytes < w.full && ws_bytes < plan_workspace(*g, {.by_rows = true}).total) {
        return NNOPS_NOT_INITIALIZED;
    }
    if (w.total > 0 && (workspace == nullptr || ws_bytes < w.total)) {
        return NNOPS_NOT_INITIALIZED;
    }
    if ((uintptr_t)workspace % 16 != 0) {
        return NNOPS_INVALID_ARGUMENT;   // staged operands and partials are 16-byte vectors
    }
    char* ws = static_cast<char*>(workspace);

    GemmI8Kern k{};
    k.m = (int)g->m;
    k.n = (int)g->n;
    k.k = (int)g->k;
    k.c = g->c;
    k.ldc_bytes = g->ldc * out_elem_bytes(g->out_kind);
    k.a_xor = g->a_u8 ? 0x80808080u : 0u;

    // k-contiguous operands (stage a transposed copy where needed)
    if (g->trans_a) {
        int8_t* at = reinterpret_cast<int8_t*>(ws + w.a_t);
        launch_transpose_i8(static_cast<const int8_t*>(g->a), g->lda, (int)g->k, (int)g->m, at, (int64_t)w.kp,
                            (int)w.kp, s);
        k.a = at;
        k.lda = w.kp;
    } else {
        k.a = static_cast<const int8_t*>(g->a);
        k.lda = g->lda;
    }
    if (w.kn.cpl != 0 || w.ring.trb) {
        k.b = g->b;               // [K,N], consumed in place by the column GEMV or the TRB ring
        k.ldb = g->ldb;
    } else if (!g->trans_b) {
        int8_t* bt = reinterpret_cast<int8_t*>(ws + w.b_t);
        launch_transpose_i8(g->b, g->ldb, (int)g->k, (int)g->n, bt, (int64_t)w.kp, (int)w.kp, s);
        k.b = bt;
        k.ldb = w.kp;
    } else {
        k.b = g->b;
        k.ldb = g->ldb;
    }

    // zero-point compensation terms
    EpiParams& e = k.ep;
    e.bias = g->bias;
    e.s_a = g->s_a; e.s_a_scalar = g->s_a_scalar;
    e.zp_a = g->zp_a; e.zp_a_scalar = g->zp_a_scalar;
    e.s_b = g->s_b; e.s_b_scalar = g->s_b_scalar;
    e.zp_b = g->zp_b; e.zp_b_scalar = g->zp_b_scalar;
    e.s_out_rows = g->s_out_rows; e.zp_out_rows = g->zp_out_rows;
    e.s_out = g->s_out; e.zp_out = g->zp_out;
    e.k = (int32_t)g->k;
    e.out_kind = g->out_kind;
    e.act = g->act;
    e.round_even = g->round_even;
    e.float_ep = g->float_ep;
    e.min_clip = g->min_clip;
    e.max_clip = g->max_clip;
    e.add_to = g->add_to;
    e.residual_pre = g->residual_pre;
    e.bias_fp = fp_out ? g->bias_fp : nullptr;
    e.act_alpha = g->act_alpha;
    e.act_beta = g->act_beta;
    if (fp_out) {
        e.float_ep = 0;
        e.round_even = 0;
    }
    e.a_off = g->a_u8 ? -128 : 0;
    const bool need_rb = g->a_u8 || g->zp_a != nullptr || g->zp_a_scalar != 0;
    const bool need_ra = g->zp_b != nullptr || g->zp_b_scalar != 0;
    e.compensate = need_ra || need_rb;
    if (need_rb && g->b_col_sums != nullptr) {
        e.r_b = g->b_col_sums;
    } else if (need_rb) {
        int32_t* rb = reinterpret_cast<int32_t*>(ws + w.r_b);
        NNOPS_LAUNCH(rowsum_i8, dim3((unsigned)((g->n + 3) / 4)), dim3(256), 0, s, k.b, k.ldb,
                           (int)g->n, (int)g->k, 0, rb);
        e.r_b = rb;
    }
    if (need_ra) {
        int32_t* ra = reinterpret_cast<int32_t*>(ws + w.r_a);
        NNOPS_LAUNCH(rowsum_i8, dim3((unsigned)((g->m + 3) / 4)), dim3(256), 0, s, k.a, k.lda,
                           (int)g->m, (int)g->k, (int)g->a_u8, ra);
        e.r_a = ra;
    }

    const bool aligned = aligned16(k.a, k.lda) && aligned16(k.b, k.ldb) && (g->k % 16 == 0);
    const bool fullk = aligned && (g->k % 64 == 0);
    const int epi = choose_epi(*g, e);
    if (w.kn.cpl != 0) {
        launch_kn(k, w.kn, reinterpret_cast<int32_t*>(ws + w.part), reinterpret_cast<uint64_t*>(ws + w.flag), s);
    } else if (g->m <= 16 && aligned && g->k % 64 == 0 && gemv_lds_ok(*g)) {
        NNOPS_LAUNCH((gemv_i8_lds<4>), dim3((unsigned)((g->n + 15) / 16)), dim3(256), 0, s, k);
    } else if (g->m <= 4 && aligned) {
        const bool flip = k.a_xor != 0u;
        // two rows per wave from M = 3: halves the A re-reads per weight byte
        const int rsel = g->m >= 3 ? 2 : 1;
#define NNOPS_ROWS_R(MT, R)                                                                         \
        {                                                                                           \
            const unsigned blocks = (unsigned)((g->n + 4 * R - 1) / (4 * R));                      \
            if (flip) {                                                                             \
                NNOPS_LAUNCH((gemv_i8_rows<MT, R, true>), dim3(blocks), dim3(256), 0, s, k);  \
            } else {                                                                                \
                NNOPS_LAUNCH((gemv_i8_rows<MT, R, false>), dim3(blocks), dim3(256), 0, s, k); \
            }                                                                                       \
        }
#define NNOPS_ROWS(MT)                                                                              \
        if (rsel == 2) NNOPS_ROWS_R(MT, 2) else NNOPS_ROWS_R(MT, 1)
        if (g->m == 1) {
            NNOPS_ROWS(1)
        } else if (g->m == 2) {
            NNOPS_ROWS(2)
        } else {
            NNOPS_ROWS(4)
        }
#undef NNOPS_ROWS_R
#undef NNOPS_ROWS
    } else if (g->m <= 16) {
        const unsigned blocks = (unsigned)((g->n + 15) / 16);
        if (aligned) {
            NNOPS_LAUNCH((gemv_i8_mfma<4, true>), dim3(blocks), dim3(256), 0, s, k);
        } else {
            NNOPS_LAUNCH((gemv_i8_mfma<4, false>), dim3(blocks), dim3(256), 0, s, k);
        }
    } else if (w.ring.mode >= 0) {
        launch_ring(k, w.ring, reinterpret_cast<int32_t*>(ws + w.part), s);
    } else if (g->m >= 1024 && g->n >= 1024) {
        launch_gemm<256, 256, 2, 2, 1>(k, aligned, fullk, epi, s);
    } else if (g->m >= 64) {
        launch_gemm<128, 128, 2, 2, 2>(k, aligned, fullk, epi, s);
    } else {
        launch_gemm<32, 64, 1, 2, 4>(k, aligned, fullk, epi, s);
    }
    return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
}

}  // namespace

int gemm_i8_in(const NnopsGemmI8Args& g, void* workspace, size_t ws_bytes, hipStream_t stream)
{
    const TimingDisarm disarm;
    return run_gemm_i8(&g, workspace, ws_bytes, stream, true);
}

}  // namespace nnops_amd

extern "C" int nnops_hip_gemm_i8(const NnopsGemmI8Args* g, void* workspace, size_t ws_bytes, void* stream)
{
    const TimingDisarm disarm;
    return run_gemm_i8(g, workspace, ws_bytes, static_cast<hipStream_t>(stream), false);
}
