// The LDS-ring GEMM kernel (int8 and f16 operands) and its launch, shared by
// gemm_i8_nk.hip ([N,K] B), gemm_i8_trb.hip ([K,N] B read in place) and
// gemm_f16.hip (f16 operands), which instantiate it side by side.
#pragma once

#include "common.hpp"

#include <type_traits>
#include <utility>

#include <algorithm>

namespace nnops_amd {

struct GemmI8Kern {
    const int8_t* a;     // [M][lda] k-contiguous
    const int8_t* b;     // [N][ldb] k-contiguous
    void* c;
    int m, n, k;
    int64_t lda, ldb, ldc_bytes;
    uint32_t a_xor;      // 0x80808080 when A is u8 (read as a - 128)
    EpiParams ep;
};

enum { RING_S8 = 0, RING_S32 = 1, RING_PART = 2, RING_FP = 3 };

struct RingSplit {
    int splits;        // K ranges per output tile
    int kt_per;        // staged k steps per split (the last split takes the rest)
    int32_t* part;     // RING_PART: [splits][M][ldp] raw accumulators
    int ldp;           // the partials' row pitch: N rounded up to 4
    float row_k;       // gemm_i8_reduce_q: RN(s_a / s_out) and RN(1 / s_out), the
    float inv_out;     // host's correctly rounded f32 quotients (the device's bits)
    uint64_t* flag;    // gemv_i8_kn_tr: [column groups][splits] split-completion flags
    uint64_t epoch;    // the launch's flag value (graph replays repeat it), never 0
};

// Which ring-kernel configuration a call takes (all zero: another kernel).
struct RingPlan {
    int bm = 0, bn = 0;     // block tile
    int splits = 0;         // K splits (1: no split)
    int mode = -1;          // RING_S8 / RING_S32 / RING_PART
    bool trb = false;       // B is [K,N] row-major, read in place (TRB)
    float us = 0.0f;        // the estimate it won by
};

constexpr int kMostSplits = 16;     // K splits at most

// The ring plan of an int8 call (ring_plan.hip), and the one by its rows alone;
// an f16 call asks with its K and row pitches in bytes.
RingPlan plan_ring(const NnopsGemmI8Args& g, const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb, bool trb,
                   int max_splits, bool f16);
RingPlan plan_ring_by_rows(const NnopsGemmI8Args& g, const int8_t* a, int64_t lda, const int8_t* b, int64_t ldb,
                           bool trb, bool small_tiles);

// How many splits' partials of an M x N output `room` bytes hold past `off`.
inline int splits_in(size_t room, size_t off, int64_t m, int64_t n)
{
    if (room == SIZE_MAX) {
        return kMostSplits;
    }
    const size_t slab = (size_t)m * (size_t)((n + 3) / 4) * 16;
    return room <= off ? 0 : (int)std::min<size_t>(kMostSplits, (room - off) / 256 * 256 / slab);
}

inline bool aligned16(const void* p, int64_t ld) { return ((uintptr_t)p % 16 == 0) && (ld % 16 == 0); }

// The ring of a plan over [N,K] rows of B (gemm_i8_nk.hip) and over a [K,N] B
// in place (gemm_i8_trb.hip).
void launch_ring_nk(const GemmI8Kern& k, const RingPlan& r, const RingSplit& sk, hipStream_t s);
void launch_ring_trb(const GemmI8Kern& k, const RingPlan& r, const RingSplit& sk, hipStream_t s);

constexpr size_t kAlign = 256;
inline size_t align_up(size_t x) { return (x + kAlign - 1) / kAlign * kAlign; }

namespace {

// min(max(x, lo), hi) for lo <= hi in one v_med3_i32 (the compiler only forms
// it when it can prove lo <= hi).
__device__ __forceinline__ int32_t med3_i32(int32_t x, int32_t lo, int32_t hi)
{
    int32_t r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(x), "v"(lo), "v"(hi));
    return r;
}

// ---------------------------------------------------------------------------
// Large-tile kernel with an asynchronous LDS ring (K % 32 == 0, 16-byte-aligned
// operands). Stages are filled by buffer_load_dwordx4 ... lds: each wave
// instruction writes 1 KiB of LDS contiguously (lane l -> bytes 16l..16l+15),
// i.e. 16 tile rows of 64 bytes, so the 16-byte chunk a lane fetches from HBM
// is chosen to land in a swizzled slot: row r's logical chunk c lives in slot
// c ^ ((r >> 2) & 3). A fragment read serves 16 lanes (16 consecutive rows,
// one logical chunk) per LDS cycle; with 64 four-byte banks those 16 reads land
// on 16 distinct 16-byte bank groups, so the read is conflict-free with no
// padding. NS stages are in flight, so each load has NS-1 k-steps of MFMA work
// to land before it is needed. The buffer form (32-bit offsets against a
// per-tile descriptor) costs fewer issue cycles than the 64-bit-address form.
//
// The MFMA takes the B fragment as its first operand, so the 32x32 accumulator
// holds C transposed: lane l owns output row (l & 31) and, in register group g,
// the 4 consecutive columns 8g + 4(l >> 5) + 0..3. Each lane therefore packs
// 4 output bytes (or one 16-byte int32 group) with no cross-lane transpose.
//
// Output modes:
//   RING_S8    fused requant (row-uniform s_a/s_out, per-column s_b, bias in
//              the accumulator init, Relu folded into the integer clamp);
//              bytes are staged per wave in LDS and written as 16-byte rows.
//   RING_S32   fused bias + Relu, int32 written straight from the accumulators.
//   RING_PART  raw int32 accumulators of this K split to a workspace slab;
//              gemm_i8_reduce sums the splits and runs the full output pass.
// ---------------------------------------------------------------------------
#define NNOPS_LPTR(x) ((__attribute__((address_space(3))) void*)(x))

// Buffer resource over [base, base + 2 GiB) with raw 32-bit offsets. The
// buffer builtins exist only in the device pass; the host pass sees a
// placeholder (kernels are never compiled for the host).
#if __HIP_DEVICE_COMPILE__
typedef __amdgpu_buffer_rsrc_t BufRsrc;
#else
struct BufRsrc {
    int w[4];
};
#endif

__device__ __forceinline__ BufRsrc buffer_rsrc(const void* base, int bytes = 0x7fffffff)
{
#if __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000);
#else
    (void)base, (void)bytes;
    return BufRsrc{};
#endif
}

// ds_read_b64_tr_b8: each 16-lane group reads 16 rows of 8 bytes (one address
// per lane) and lane L of the group receives byte L & 7 of rows 2j + (L >> 3),
// j = 0..7. With lane i addressing row k0 + (i >> 1), columns c0 + 8 (i & 1)
// of a row-major byte tile, lane L receives column c0 + L at rows k0 .. k0 + 7:
// a k-contiguous fragment of a tile stored n-contiguous.
typedef int v2i __attribute__((ext_vector_type(2)));
__device__ __forceinline__ v2i lds_read_tr8(const int8_t* p)
{
#if __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) v2i*)(p));
#else
    (void)p;
    return v2i{0, 0};
#endif
}

// The same read as inline assembly, for loops whose LDS stages arrive by DMA:
// the compiler cannot tell the intrinsic's reads from the stages still in
// flight and puts a full vmcnt(0) before them, which drains the DMA ring every
// stage. The assembly is not tracked, so its results are pending until
// lds_tr8_ready ties them to an explicit lgkmcnt(0).
__device__ __forceinline__ v2i lds_read_tr8_asm(const int8_t* p)
{
    v2i r;
#if __HIP_DEVICE_COMPILE__
    const uint32_t a = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) int8_t*)(p);
    asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(r) : "v"(a) : "memory");
#else
    (void)p;
    r = v2i{0, 0};
#endif
    return r;
}

// lgkmcnt(0) with the fragments built from lds_read_tr8_asm as in/out
// operands: their uses cannot move above it.
template <int N>
__device__ __forceinline__ void lds_tr8_ready_frags(v4i (&f)[N])
{
    static_assert(N == 1 || N == 2, "one or two fragments");
#if __HIP_DEVICE_COMPILE__
    if constexpr (N == 1) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]) : : "memory");
    } else {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f[0]), "+v"(f[1]) : : "memory");
    }
#else
    (void)f;
#endif
}

// Waits until at most S stages of L vector-memory operations each are in
// flight (S wave-uniform, clamped to MAXS).
template <int L, int MAXS>
__device__ __forceinline__ void wait_stages(int s)
{
    if constexpr (MAXS <= 0) {
        wait_vmcnt<0>();
    } else {
        if (s >= MAXS) {
            wait_vmcnt<MAXS * L>();
        } else {
            wait_stages<L, MAXS - 1>(s);
        }
    }
}

// Waits for every outstanding LDS read of the wave and makes the 16 values
// read by lds_read_tr8_asm depend on that wait, so no use moves above it.
__device__ __forceinline__ void lds_tr8_ready(v2i (&lo)[8], v2i (&hi)[8])
{
#if __HIP_DEVICE_COMPILE__
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(lo[0]), "+v"(lo[1]), "+v"(lo[2]), "+v"(lo[3]), "+v"(lo[4]), "+v"(lo[5]), "+v"(lo[6]),
                   "+v"(lo[7]), "+v"(hi[0]), "+v"(hi[1]), "+v"(hi[2]), "+v"(hi[3]), "+v"(hi[4]), "+v"(hi[5]),
                   "+v"(hi[6]), "+v"(hi[7])
                 :
                 : "memory");
#else
    (void)lo;
    (void)hi;
#endif
}

// Exchanges x's lanes 32..63 with y's lanes 0..31 (v_permlane32_swap): with
// x = a word of lane half h = 0 / 1 and y the same for another word, lane
// l < 32 ends with (x, y) = (x_l, x_{l+32}) and lane l + 32 with
// (y_l, y_{l+32}).
__device__ __forceinline__ void swap_half_waves(uint32_t& x, uint32_t& y)
{
#if __HIP_DEVICE_COMPILE__
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
#else
    (void)x, (void)y;
#endif
}

// 16 bytes per lane from base + voff + soff into LDS at lds + 16 * lane.
// AUX: the cache policy bits (2: non-temporal, for data read once).
template <int AUX = 0>
__device__ __forceinline__ void buffer_load_lds16(BufRsrc r, int8_t* lds, int voff, int soff)
{
#if __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, NNOPS_LPTR(lds), 16, voff, soff, 0, AUX);
#else
    (void)r, (void)lds, (void)voff, (void)soff;
#endif
}

// Stores and loads with the sc1 cache policy: coherent at device scope (the
// lowering of an agent-scope atomic store / load) without a cache-wide fence;
// how the K splits of a one-launch kernel hand their partial sums over.
__device__ __forceinline__ void buffer_store4_sc1(BufRsrc r, int32_t v, int voff)
{
#if __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_buffer_store_b32(v, r, voff, 0, 16);
#else
    (void)r, (void)v, (void)voff;
#endif
}

__device__ __forceinline__ void buffer_store8_sc1(BufRsrc r, uint64_t v, int voff)
{
#if __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(v2i, v), r, voff, 0, 16);
#else
    (void)r, (void)v, (void)voff;
#endif
}

__device__ __forceinline__ uint64_t buffer_load8_sc1(BufRsrc r, int voff)
{
#if __HIP_DEVICE_COMPILE__
    return __builtin_bit_cast(uint64_t, __builtin_amdgcn_raw_buffer_load_b64(r, voff, 0, 16));
#else
    (void)r, (void)voff;
    return 0;
#endif
}

__device__ __forceinline__ v4i buffer_load16_sc1(BufRsrc r, int voff)
{
#if __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, 0, 16);
#else
    (void)r, (void)voff;
    return v4i{0, 0, 0, 0};
#endif
}

// 16 zero bytes in global memory (never written): the address a lane loads
// from when its table value is absent, so the load needs no branch.
static __device__ __attribute__((aligned(16))) int32_t kZero16[4];

__device__ __forceinline__ void block_barrier()
{
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");  // no LDS access moves across the barrier
}

// Logical order: the hardware deals workgroups round-robin over the 8 XCDs,
// so consecutive logical ids are gathered on one XCD. Splits are outermost (a
// band of one XCD shares one K range of A), then tiles grouped 4 along M
// (neighbours share B column panels in that XCD's L2).
__device__ __forceinline__ void ring_coords(int tiles_m, int tiles_n, int& tm, int& tn, int& sp)
{
    int bid = blockIdx.x;
    const int nb = gridDim.x;
    if ((nb & 7) == 0) {
        bid = (bid & 7) * (nb >> 3) + (bid >> 3);
    }
    const int tiles = tiles_m * tiles_n;
    sp = bid / tiles;
    bid -= sp * tiles;
    constexpr int G = 4;
    const int per_group = G * tiles_n;
    const int group = bid / per_group;
    const int first_m = group * G;
    const int gsize = min(tiles_m - first_m, G);
    const int in_group = bid - group * per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}

// F16: the operands are f16 (the same byte staging: K, lda and ldb in bytes,
// a 16-byte lane fragment is 8 halves of v_mfma_f32_32x32x16_f16 as it is 16
// int8 of v_mfma_i32_32x32x32_i8), the accumulators f32; RING_FP then writes
// acc * s_a_scalar (alpha) and RING_PART the f32 partials' bits.
//
// TRB: B is [K,N] row-major (ldb its row pitch in bytes), staged as it lies: a
// stage holds BK k rows of BN bytes, 16-byte chunk c of row r in slot
// c ^ swzb(r), and the B fragments are built by lds_read_tr8 (two per
// fragment: k rows +0..7 and +8..15 of the lane's 16). No transposed copy.
//
// TAIL: K % 128 != 0 (a multiple of 32): the last stage holds fewer than four
// 32-byte slices of k. Its staging reads past a row's k (into the next row's,
// or past the operand's end, where the descriptors make it 0); only the slices
// of k run on the matrix cores.
template <int BM, int BN, int WM, int WN, int NS, int MODE, bool FLIP, bool F16 = false, bool TRB = false,
          bool TAIL = false>
__global__ __launch_bounds__(WM * WN * 64)
__attribute__((amdgpu_waves_per_eu((WM * WN + 3) / 4, BM + BN <= 192 ? 4 : (WM * WN + 3) / 4)))
void gemm_i8_ring(GemmI8Kern p, RingSplit sk)
{
    static_assert(!F16 || MODE == RING_FP || MODE == RING_PART, "f16 operands: fp or partial outputs");
    static_assert(!TRB || !F16, "row-major B: int8 operands");
    constexpr int BK = 128;                       // k bytes per stage and row
    constexpr int W = WM * WN;
    constexpr int TM = BM / WM, TN = BN / WN;
    constexpr int FM = TM / 32, FN = TN / 32;
    constexpr int CPR = BK / 16;                  // 16-byte chunks per staged row
    constexpr int RPI = 1024 / BK;                // rows per 1 KiB load instruction
    constexpr int QA = BM / RPI / W;              // load instructions per wave per stage (A)
    constexpr int QB = BN / RPI / W;
    constexpr int L = QA + QB;                    // vector-memory ops per wave per stage
    // TRB rings of 128 rows and more: the transposed reads as untracked
    // assembly, per-stage counted waits to the end and step 0 peeled, so no
    // full vmcnt(0) drains the ring (4096^3: 73 -> 69 us; 333 x 4096 x
    // 14336: 46 -> 40 us). The 64 x 64 tiles (a handful of stages, latency
    // bound) and the [N,K] rings measured faster without.
    constexpr bool kTrAsm = TRB && BM >= 128;
    constexpr int S = BK / 32;                    // 32-k MFMA slices per stage
    constexpr int kStage = (BM + BN) * BK;
    constexpr int kPitch8 = TN + 16;              // staged byte row pitch: 2-way bank conflicts at most
    static_assert(QA * W * RPI == BM && QB * W * RPI == BN, "rows per stage");
    // TRB staging: 1024 / BN k rows per load instruction, CPRB chunks per row
    constexpr int RPIB = TRB ? 1024 / BN : 1;
    constexpr int CPRB = BN / 16;
    static_assert(!TRB || (1024 % BN == 0 && BN >= 64 && (BK / RPIB) == QB * W), "row-major B staging");
    static_assert(FM * 32 == TM && FN * 32 == TN, "wave tile");
    static_assert(W * TM * kPitch8 <= NS * kStage, "byte staging fits the ring");
    static_assert(NS >= 2 && (NS - 1) * L < 64, "vmcnt range");
    static_assert(MODE == RING_PART || !FLIP, "u8 A needs the compensating output pass");

    // the output pass's per-column scales, staged at the start (their load
    // latency then hides behind the first stage's) where the LDS holds them;
    // RING_FP: the bias in the destination's type, widened to f32, likewise.
    // One array holds the ring and both tables: with tables of their own the
    // compiler tells the LDS arrays apart, tracks the DMA per array and puts a
    // vmcnt(0) before a fragment read in the K loop, which drains the ring
    // every stage (RING_FP in every tile shape, RING_S8 in those of three
    // slots). One array, per call: 1000 x 4096 x 11008 f16 133 -> 115 us,
    // 512 x 4096 x 11008 s8 on 128 x 256 tiles 54 -> 36 us, 48 x 4096 x 14336
    // f16 on 64 x 64 tiles 58 -> 28 us.
    constexpr bool kSbl = (MODE == RING_S8 || MODE == RING_FP) && NS * kStage + BN * 4 <= 160 * 1024;
    constexpr bool kBl = MODE == RING_FP && kSbl && NS * kStage + BN * 8 <= 160 * 1024;
    constexpr int kTables = (kSbl ? BN * 4 : 0) + (kBl ? BN * 4 : 0);
    __shared__ __attribute__((aligned(1024))) int8_t ring[NS * kStage + kTables];
    float* const sbl = reinterpret_cast<float*>(ring + NS * kStage);
    float* const biasl = sbl + BN;

    int tm, tn, sp;
    ring_coords(ceil_div(p.m, BM), ceil_div(p.n, BN), tm, tn, sp);
    const int m0 = tm * BM, n0 = tn * BN;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wm0 = (wave / WN) * TM, wn0 = (wave % WN) * TN;
    const int kt0 = sp * sk.kt_per;
    const int kt = (sp == sk.splits - 1) ? (p.k + BK - 1) / BK - kt0 : sk.kt_per;
    // the stages of whole slices, and the slices of a last, shorter one
    const int tail = TAIL && sp == sk.splits - 1 ? (p.k % BK) / 32 : 0;
    const int kf = tail != 0 ? kt - 1 : kt;

    // Staged rows are BK bytes; chunk c of row r sits in slot c ^ swz(r), so
    // the 16 rows a fragment read serves per LDS cycle hit 16 distinct 16-byte
    // bank groups (2 rows per 256 bytes).
    auto swz = [](int r) { return (r >> 1) & 7; };
    // TRB: a transposed read serves 8 k rows x two 16-byte chunks per 32
    // lanes; rows sharing a 256-byte bank row (256 / BN of them) keep their
    // slots, and the bank rows' 8 slot pairs differ in slot bits 1.., so the
    // 16 chunks fall in 16 distinct 16-byte bank groups.
    auto swzb = [](int r) { return ((r / (BN >= 256 ? 1 : 256 / BN)) & (CPRB / 2 - 1)) << 1; };

    // Descriptors over this tile's row panels from this split's first k; rows
    // past M/N are clamped to the last row (computed, never stored).
    // They end at the last row's last k.
    const int a_end = (min(BM, p.m - m0) - 1) * (int)p.lda + p.k - kt0 * BK;
    const BufRsrc rsa = buffer_rsrc(p.a + (int64_t)m0 * p.lda + (int64_t)kt0 * BK, a_end);
    // TRB: the descriptor ends with the dword of B's last byte, so chunks past
    // column N of the last k row read 0 (earlier rows' read the next row: never
    // stored). Whole dwords: the range check makes one that is only partly in
    // range 0, N % 4 valid columns with it (ldb and B are multiples of 16).
    const BufRsrc rsb = TRB ? buffer_rsrc(p.b + (int64_t)kt0 * BK * p.ldb + n0,
                                          (int)((int64_t)(p.k - kt0 * BK - 1) * p.ldb + ceil_div(p.n - n0, 4) * 4))
                            : buffer_rsrc(p.b + (int64_t)n0 * p.ldb + (int64_t)kt0 * BK,
                                          (min(BN, p.n - n0) - 1) * (int)p.ldb + p.k - kt0 * BK);
    int a_off[QA], b_off[QB];
#pragma unroll
    for (int q = 0; q < QA; ++q) {
        const int r = (wave * QA + q) * RPI + lane / CPR;
        const int c = (lane % CPR) ^ swz(r);
        a_off[q] = min(r, p.m - 1 - m0) * (int)p.lda + c * 16;
    }
#pragma unroll
    for (int q = 0; q < QB; ++q) {
        if constexpr (TRB) {
            const int r = (wave * QB + q) * RPIB + lane / CPRB;
            const int c = (lane % CPRB) ^ swzb(r);
            b_off[q] = r * (int)p.ldb + c * 16;
        } else {
            const int r = (wave * QB + q) * RPI + lane / CPR;
            const int c = (lane % CPR) ^ swz(r);
            b_off[q] = min(r, p.n - 1 - n0) * (int)p.ldb + c * 16;
        }
    }
    const int b_step = TRB ? BK * (int)p.ldb : BK;     // bytes from one stage's B rows to the next's
    auto issue = [&](int s) {
        int8_t* base = ring + (s % NS) * kStage;
#pragma unroll
        for (int q = 0; q < QA; ++q) {
            buffer_load_lds16(rsa, base + (wave * QA + q) * 1024, a_off[q], s * BK);
        }
#pragma unroll
        for (int q = 0; q < QB; ++q) {
            buffer_load_lds16(rsb, base + BM * BK + (wave * QB + q) * 1024, b_off[q], s * b_step);
        }
    };

    // Accumulators (transposed layout), initialised after the first stage loads.
    std::conditional_t<F16, v16f, v16i> acc[FM][FN];

    // Fragment reads of slice ks: row (lane & 31) of each 32-row fragment,
    // logical chunk 2 ks + (lane >> 5).
    const int fr = lane & 31;
    auto frag = [&](const int8_t* st, int row, int ks) {
        const int c = (2 * ks + (lane >> 5)) ^ swz(row);
        return *reinterpret_cast<const v4i*>(st + row * BK + c * 16);
    };
    // TRB: the B fragment of columns col .. col + 31 at slice ks from the
    // row-major stage: lane (group g, index i) addresses k row 32 ks + 16 (g
    // >> 1) + (i >> 1) (+8 for the second read), columns col + 16 (g & 1) +
    // 8 (i & 1); lane l receives column col + (l & 31) at k 32 ks + 16 (l >>
    // 5) + 0..15, the layout of the A fragments.
    const int tr_k = 16 * (lane >> 5) + ((lane & 15) >> 1);
    const int tr_c = 16 * ((lane >> 4) & 1) + 8 * (lane & 1);
    auto frag_tr = [&](const int8_t* stb, int col, int ks) {
        const int k0 = 32 * ks + tr_k;
        const int c = col + tr_c;
        const int8_t* plo = stb + k0 * BN + (((c >> 4) ^ swzb(k0)) << 4) + (c & 15);
        const int8_t* phi = stb + (k0 + 8) * BN + (((c >> 4) ^ swzb(k0 + 8)) << 4) + (c & 15);
        if constexpr (kTrAsm) {
            // untracked reads: step() ties them to an lgkmcnt(0) before their use
            const v2i lo = lds_read_tr8_asm(plo);
            const v2i hi = lds_read_tr8_asm(phi);
            return v4i{lo.x, lo.y, hi.x, hi.y};
        } else {
            const v2i lo = lds_read_tr8(plo);
            const v2i hi = lds_read_tr8(phi);
            return v4i{lo.x, lo.y, hi.x, hi.y};
        }
    };
    auto read_frags = [&](const int8_t* st, int ks, v4i (&fa)[FM], v4i (&fb)[FN]) {
        if constexpr (TRB) {
            fb[0] = frag_tr(st + BM * BK, wn0, ks);
        } else {
            fb[0] = frag(st + BM * BK, wn0 + fr, ks);
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            fa[i] = frag(st, wm0 + i * 32 + fr, ks);
        }
#pragma unroll
        for (int j = 1; j < FN; ++j) {
            if constexpr (TRB) {
                fb[j] = frag_tr(st + BM * BK, wn0 + j * 32, ks);
            } else {
                fb[j] = frag(st + BM * BK, wn0 + j * 32 + fr, ks);
            }
        }
    };
    auto mfma_all = [&](v4i (&fa)[FM], const v4i (&fb)[FN]) {
        if constexpr (FLIP) {  // u8 A enters the signed MFMA as a - 128
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                fa[i] ^= v4i{(int)0x80808080u, (int)0x80808080u, (int)0x80808080u, (int)0x80808080u};
            }
        }
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                if constexpr (F16) {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, fb[j]),
                                                                      __builtin_bit_cast(v8h, fa[i]), acc[i][j], 0,
                                                                      0, 0);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(fb[j], fa[i], acc[i][j], 0, 0, 0);
                }
            }
        }
    };
    // One fragment read after each of the first FM + FN MFMAs, so every read
    // has part of a slice of matrix work to land before it is needed; with
    // loads, they go on the last MFMAs of the slice.
    constexpr int NR = FM + (TRB ? 2 : 1) * FN;     // LDS reads per slice
    auto schedule = [&](bool loads) {
#pragma unroll
        for (int q = 0; q < FM * FN; ++q) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (q < NR) {
                if (q + 1 < FM * FN) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                } else {
                    // the last MFMA takes the reads left over
                    __builtin_amdgcn_sched_group_barrier(0x100, NR - FM * FN + 1, 0);
                }
            }
            if (loads && q >= FM * FN - L && q - (FM * FN - L) < L) {
                __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
            }
        }
    };

    // The output pass's column tables: bias[n] (whose values start the
    // accumulators of the fused modes), the staged s_b and fp bias.
    // kTrAsm: bias[n] and s_b are loaded before the first stages are issued
    // and used after (with step 0 peeled the first use then waits for these
    // loads alone); every lane loads unconditionally, from a 16-byte zero
    // stand-in where a value is absent, since a load under a branch is waited
    // for where the branch joins. Elsewhere they follow the first stages
    // (measured as fast or faster there).
    const int32_t* const zero16 = kZero16;
    v4i bpre[kTrAsm ? FN : 1][4];
    const int nsb = n0 + 4 * (int)threadIdx.x;
    const bool sb_live = kTrAsm && kSbl && threadIdx.x < BN / 4 && p.ep.s_b != nullptr && nsb < p.n;
    v4f sbpre = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (kTrAsm) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                bpre[j][g] = v4i{0, 0, 0, 0};
                if constexpr (MODE != RING_PART) {
                    const int n = n0 + wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
                    const bool live = p.ep.bias != nullptr && n < p.n;
                    bpre[j][g] = *reinterpret_cast<const v4i*>(live ? p.ep.bias + n : zero16);
                }
            }
        }
        if constexpr (kSbl) {
            sbpre = *reinterpret_cast<const v4f*>(sb_live ? p.ep.s_b + nsb : reinterpret_cast<const float*>(zero16));
        }
        // keep those loads ahead of the stages
        asm volatile("" ::: "memory");
    }

    // Ring: stage s goes to slot s % NS; nothing is issued past this split's
    // last stage, so the vmcnt waits count only the stages really in flight.
#pragma unroll
    for (int s = 0; s < NS - 1; ++s) {
        if (s < kt) {
            issue(s);
        }
    }
    // Accumulators (transposed layout); the fused modes start from bias[n].
#pragma unroll
    for (int j = 0; j < FN && F16; ++j) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            acc[i][j] = std::conditional_t<F16, v16f, v16i>{0};
        }
    }
#pragma unroll
    for (int j = 0; j < FN && !F16; ++j) {
        int32_t b0[16];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            v4i bv = v4i{0, 0, 0, 0};
            if constexpr (kTrAsm) {
                bv = bpre[j][g];
            } else if constexpr (MODE != RING_PART) {
                const int n = n0 + wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
                if (p.ep.bias != nullptr && n < p.n) {
                    bv = *reinterpret_cast<const v4i*>(p.ep.bias + n);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                b0[4 * g + e] = bv[e];
            }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                acc[i][j][r] = b0[r];
            }
        }
    }
    if constexpr (kSbl) {
        if (threadIdx.x < BN / 4) {
            const int n = n0 + 4 * (int)threadIdx.x;
            v4f v = v4f{p.ep.s_b_scalar, p.ep.s_b_scalar, p.ep.s_b_scalar, p.ep.s_b_scalar};
            if constexpr (kTrAsm) {
                if (sb_live) {
                    v = sbpre;
                }
            } else if (p.ep.s_b != nullptr && n < p.n) {
                v = *reinterpret_cast<const v4f*>(p.ep.s_b + n);
            }
            *reinterpret_cast<v4f*>(&sbl[4 * threadIdx.x]) = v;
        }
    }
    if constexpr (kBl) {
        if (threadIdx.x >= BN / 4 && threadIdx.x < BN / 2) {
            const int t = (int)threadIdx.x - BN / 4;
            const int n = n0 + 4 * t;
            v4f v = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (p.ep.bias_fp != nullptr && n < p.n) {
                if (p.ep.out_kind == NNOPS_OUT_F16) {
                    const _Float16* b16 = static_cast<const _Float16*>(p.ep.bias_fp) + n;
                    v = v4f{(float)b16[0], (float)b16[1], (float)b16[2], (float)b16[3]};
                } else {
                    v = *reinterpret_cast<const v4f*>(static_cast<const float*>(p.ep.bias_fp) + n);
                }
            }
            *reinterpret_cast<v4f*>(&biasl[4 * t]) = v;
        }
    }
    // stage 0 landed; the others issued (up to NS - 2) may stay in flight
    if constexpr (kTrAsm) {
        wait_stages<L, NS - 2>(min(kt, NS - 1) - 1);
    } else if (kt >= NS - 1) {
        wait_vmcnt<(NS - 2) * L>();
    } else {
        wait_vmcnt<0>();
    }
    block_barrier();

    v4i f0a[FM], f0b[FN], f1a[FM], f1b[FN];
    read_frags(ring, 0, f0a, f0b);
    // One stage: stage t+NS-1 is issued into the slot read in step t-1 (freed
    // by that step's barrier); slice ks runs on the matrix cores while slice
    // ks+1's fragments load; after the last slice, wait for stage t+1 (its
    // later stages may stay in flight) and for every wave's reads of stage t
    // (lgkmcnt, then the barrier), then read slice 0 of stage t+1.
    auto step = [&](int t) {
        const int8_t* st = ring + (t % NS) * kStage;
        const bool more = t + NS - 1 < kt;
        if (more) {
            issue(t + NS - 1);
        }
#pragma unroll
        for (int ks = 0; ks < S; ++ks) {
            v4i (&ca)[FM] = (ks & 1) ? f1a : f0a;
            v4i (&cb)[FN] = (ks & 1) ? f1b : f0b;
            v4i (&na)[FM] = (ks & 1) ? f0a : f1a;
            v4i (&nb)[FN] = (ks & 1) ? f0b : f1b;
            if constexpr (kTrAsm) {
                lds_tr8_ready_frags(cb);
            }
            if (ks + 1 < S) {
                read_frags(st, ks + 1, na, nb);
                mfma_all(ca, cb);
                schedule(false);
            } else {
                mfma_all(ca, cb);
                if constexpr (kTrAsm) {
                    // stage t + 1 landed; the ones after it may stay in
                    // flight (all issued: kt - 2 - t of them)
                    wait_stages<L, NS - 2>(more ? NS - 2 : kt - 2 - t);
                } else if (more) {
                    wait_vmcnt<(NS - 2) * L>();
                } else {
                    wait_vmcnt<0>();
                }
                __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): this wave's reads of stage t are done
                block_barrier();
                if (t + 1 < kt) {
                    read_frags(ring + ((t + 1) % NS) * kStage, 0, na, nb);
                }
            }
        }
    };
    // kTrAsm: step 0 outside the loop (the accumulators start from loaded
    // values, and a loop that uses loaded values while issuing loads of its
    // own gets a full vmcnt(0) before it)
    int t0 = 0;
    if constexpr (kTrAsm) {
        if (kf > 0) {
            step(0);
        }
        t0 = 1;
    }
    for (int t = t0; t < kf; ++t) {
        step(t);
    }
    if constexpr (TAIL) {
        // slice 0 of the last stage is read already
        const int8_t* st = ring + ((kt - 1) % NS) * kStage;
        auto tail_slice = [&](int ks, v4i (&fa)[FM], v4i (&fb)[FN]) {
            if (ks < tail) {
                if (ks > 0) {
                    read_frags(st, ks, fa, fb);
                }
                if constexpr (kTrAsm) {
                    lds_tr8_ready_frags(fb);
                }
                mfma_all(fa, fb);
            }
        };
        // (an even stage ends with slice 0 of the next in f0a / f0b)
        tail_slice(0, f0a, f0b);
        tail_slice(1, f1a, f1b);
        tail_slice(2, f0a, f0b);
    }
    // The output pass's per-column scales: from the LDS copy staged at the
    // start, or else a lane's 8 loads issued together with one wait. They are
    // not read during the last stage: that would raise the loop's register
    // peak past the 256 of two waves per SIMD.
    const EpiParams& ep = p.ep;
    v4f sbp[FN][4];
    if constexpr (MODE == RING_S8 || MODE == RING_FP) {
#pragma unroll
        for (int j = 0; j < FN; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int nl = wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
                if constexpr (kSbl) {
                    sbp[j][g] = *reinterpret_cast<const v4f*>(&sbl[nl]);
                } else {
                    sbp[j][g] = v4f{ep.s_b_scalar, ep.s_b_scalar, ep.s_b_scalar, ep.s_b_scalar};
                    if (ep.s_b != nullptr && n0 + nl < p.n) {
                        sbp[j][g] = *reinterpret_cast<const v4f*>(ep.s_b + n0 + nl);
                    }
                }
            }
        }
    }
    __syncthreads();   // every wave is done with the ring before it is reused for staging

    if constexpr (MODE == RING_S8) {
        // Requant in the transposed layout: per lane 4 consecutive columns of
        // one row per register group. Relu is folded into the clamp: with
        // req >= 0 a negative v gives r <= 0 and Relu's 0 gives r = 0, so
        // raising the low bound to 0 yields the same code; with req < 0 the high
        // bound drops to 0 instead. The integer clamp equals nnops' float clamp
        // before rounding (the bounds are integers and rounding is monotonic).
        const bool relu = ep.act == NNOPS_ACT_RELU;
        const bool u8 = ep.out_kind == NNOPS_OUT_U8;
        const int32_t lo_i = (u8 ? 0 : -128) - ep.zp_out;
        const int32_t hi_i = (u8 ? 255 : 127) - ep.zp_out;
        const float row_k = __fdiv_rn(ep.s_a_scalar, ep.s_out);
        // the whole [BM][BN] byte tile staged at once where the ring holds it,
        // so the stores are whole rows of the tile (BN bytes: whole 128-byte
        // lines) rather than each wave's TN-byte segments
        constexpr int kWholeP = BN + 16;
        constexpr bool kWhole = BM * kWholeP <= NS * kStage && (BN % 64) == 0 && (BM * BN / 16) % (W * 64) == 0;
        constexpr int kSP = kWhole ? kWholeP : kPitch8;
        int8_t* stage8 = kWhole ? ring + wm0 * kSP + wn0 : ring + wave * (TM * kPitch8);
        // Two instructions per element are dropped where the parameters
        // allow: with Relu, only the rounding of values on the unclamped side
        // of 0 reaches the output (the other side clamps to 0 whichever way it
        // rounds), so the half-away addend is the column's constant
        // +-0.5 (the sign of req) instead of copysign(0.5, x); and a zero
        // output zero point needs no add.
        // Each lane packs one row's 4 columns per register group g (columns
        // 8g + 4h .. +3, h = lane / 32); a permlane32 swap of groups (0, 2)
        // and (1, 3) then gives lane h the row's 16 contiguous columns 16h ..
        // 16h + 15 of the fragment, written to the stage as one 16-byte LDS
        // store (four 4-byte stores with 2-way bank conflicts before: the
        // largest part of the output pass).
        auto requant = [&](auto relu_c, auto zp_c) {
            constexpr bool kRelu = decltype(relu_c)::value;
            constexpr bool kZp = decltype(zp_c)::value;
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                uint32_t w[FM][4];
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const v4f sb = sbp[j][g];
                    float req[4], half[4];
                    int32_t lo[4], hi[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        req[e] = __fmul_rn(row_k, sb[e]);
                        lo[e] = (kRelu && req[e] >= 0.0f) ? max(lo_i, 0) : lo_i;
                        hi[e] = (kRelu && !(req[e] >= 0.0f)) ? min(hi_i, 0) : hi_i;
                        half[e] = req[e] >= 0.0f ? 0.5f : -0.5f;
                    }
#pragma unroll
                    for (int i = 0; i < FM; ++i) {
                        uint32_t q[4];
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const float x = __fmul_rn((float)acc[i][j][4 * g + e], req[e]);
                            // round half away from zero: the conversion truncates as trunc() does
                            const float h = kRelu ? half[e] : __builtin_copysignf(0.5f, x);
                            const int32_t r = (int32_t)__fadd_rn(x, h);
                            q[e] = (uint32_t)(kZp ? med3_i32(r, lo[e], hi[e]) + ep.zp_out : med3_i32(r, lo[e], hi[e]));
                        }
                        w[i][g] = __builtin_amdgcn_perm(q[1], q[0], 0x0c0c0400u) |
                                  __builtin_amdgcn_perm(q[3], q[2], 0x04000c0cu);
                    }
                }
#pragma unroll
                for (int i = 0; i < FM; ++i) {
                    swap_half_waves(w[i][0], w[i][2]);
                    swap_half_waves(w[i][1], w[i][3]);
                    const v4i v = v4i{(int)w[i][0], (int)w[i][2], (int)w[i][1], (int)w[i][3]};
                    *reinterpret_cast<v4i*>(stage8 + (i * 32 + (lane & 31)) * kSP + j * 32 + 16 * (lane >> 5)) = v;
                }
            }
        };
        using TrueC = std::integral_constant<bool, true>;
        using FalseC = std::integral_constant<bool, false>;
        if (relu && ep.zp_out == 0) {
            requant(TrueC{}, FalseC{});
        } else if (relu) {
            requant(TrueC{}, TrueC{});
        } else if (ep.zp_out == 0) {
            requant(FalseC{}, FalseC{});
        } else {
            requant(FalseC{}, TrueC{});
        }
        if constexpr (kWhole) {
            __syncthreads();
            // 16-byte chunks of whole tile rows, wave w taking rows w, w + W, ...
            constexpr int CPRW = BN / 16;
#pragma unroll
            for (int q = 0; q < BM * CPRW / (W * 64); ++q) {
                const int idx = (q * W + wave) * 64 + lane, r = idx / CPRW, c = idx % CPRW;
                const int m = m0 + r, n = n0 + c * 16;
                const v4i v = *reinterpret_cast<const v4i*>(ring + r * kSP + c * 16);
                if (m < p.m && n < p.n) {
                    char* cptr = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes + n;
                    __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(cptr));
                }
            }
            return;
        }
        __builtin_amdgcn_wave_barrier();
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        // 16-byte row chunks of the wave tile (host-checked: N % 16 == 0,
        // 16-byte-aligned C and pitch)
        constexpr int CPR = TN / 16;
#pragma unroll
        for (int q = 0; q < TM * CPR / 64; ++q) {
            const int idx = q * 64 + lane, r = idx / CPR, c = idx % CPR;
            const int m = m0 + wm0 + r, n = n0 + wn0 + c * 16;
            const v4i v = *reinterpret_cast<const v4i*>(stage8 + r * kPitch8 + c * 16);
            if (m < p.m && n < p.n) {
                char* cptr = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes + n;
                __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(cptr));
            }
        }
    } else if constexpr (MODE == RING_FP) {
        // f32 / f16 destination, plain operands (no zero points) and an
        // identity or Relu activation (host-checked): f = v * (s_a * s_b[n])
        // [+ bias[n]] [+ C_old before / after the clip], clip, Relu -- the
        // operation order of the generic pass (epi_value_fp). Host-checked:
        // N % 4 == 0, 16-byte-aligned C and pitch.
        const bool f16 = ep.out_kind == NNOPS_OUT_F16;
        const bool relu = ep.act == NNOPS_ACT_RELU;
        const bool pre = ep.add_to && ep.residual_pre, post = ep.add_to && !ep.residual_pre;
        // per 4-column group (j, g): the columns' scales and bias, loaded once
        // for the FM row fragments that share them
        struct ColFp {
            v4f sb, bias;
            int n;
        };
        auto col_fp = [&](int j, int g) {
            ColFp cp;
            cp.n = n0 + wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
            cp.sb = sbp[j][g];
            cp.bias = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if constexpr (kBl) {
                cp.bias = *reinterpret_cast<const v4f*>(&biasl[cp.n - n0]);
            } else if (cp.n < p.n && ep.bias_fp != nullptr) {
                if (f16) {
                    const _Float16* b16 = static_cast<const _Float16*>(ep.bias_fp) + cp.n;
                    cp.bias = v4f{(float)b16[0], (float)b16[1], (float)b16[2], (float)b16[3]};
                } else {
                    cp.bias = *reinterpret_cast<const v4f*>(static_cast<const float*>(ep.bias_fp) + cp.n);
                }
            }
            return cp;
        };
        // the 4 values of (i, j, g) for this lane: row wm0 + 32 i + (lane & 31),
        // columns cp.n .. + 3
        // CLIP: a finite clip range (the default -inf / +inf clip is the
        // identity for every value, NaN included, and is left out)
        // FORM (host-known) > 0: no residual and no clip, so the value is
        // v * (s_a * s_b[n]) [+ bias[n]] [Relu] with no per-element branches
        // (1: neither, 2: bias, 3: Relu, 4: both), the general order's
        // operations; 0: the general pass
        auto values = [&](int i, int j, int g, const ColFp& cp, float sa, auto clip_c, auto form_c) {
            constexpr bool kClip = decltype(clip_c)::value;
            constexpr int kForm = decltype(form_c)::value;
            constexpr bool kPlain = kForm > 0;
            const int n = cp.n;
            const int m = m0 + wm0 + i * 32 + (lane & 31);
            v4f o = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (n >= p.n || m >= p.m) {
                return o;
            }
            v4f old = v4f{0.0f, 0.0f, 0.0f, 0.0f};
            if (!kPlain && ep.add_to) {
                const char* cptr = static_cast<const char*>(p.c) + (int64_t)m * p.ldc_bytes + (int64_t)n * (f16 ? 2 : 4);
                if (f16) {
                    const _Float16* o16 = reinterpret_cast<const _Float16*>(cptr);
                    old = v4f{(float)o16[0], (float)o16[1], (float)o16[2], (float)o16[3]};
                } else {
                    old = *reinterpret_cast<const v4f*>(cptr);
                }
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float f = __fmul_rn((float)acc[i][j][4 * g + e], __fmul_rn(sa, cp.sb[e]));
                if constexpr (kPlain) {
                    if constexpr (kForm == 2 || kForm == 4) {
                        f = __fadd_rn(f, cp.bias[e]);
                    }
                    if constexpr (kForm == 3 || kForm == 4) {
                        f = f > 0.0f ? f : 0.0f;
                    }
                    o[e] = f;
                    continue;
                }
                if (ep.bias_fp != nullptr) {
                    f = __fadd_rn(f, cp.bias[e]);
                }
                if (pre) {
                    f = __fadd_rn(f, old[e]);
                }
                if constexpr (kClip) {
                    f = f < ep.min_clip ? ep.min_clip : f;
                    f = ep.max_clip < f ? ep.max_clip : f;
                }
                if (relu) {
                    f = f > 0.0f ? f : 0.0f;
                }
                if (post) {
                    if (f16) {
                        f = (float)(_Float16)f;
                    }
                    f = __fadd_rn(f, old[e]);
                }
                o[e] = f;
            }
            return o;
        };
        float sa_i[FM];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int m = min(m0 + wm0 + i * 32 + (lane & 31), p.m - 1);
            sa_i[i] = ep.s_a != nullptr ? ep.s_a[m] : ep.s_a_scalar;
        }
        if constexpr (W * TM * 128 <= NS * kStage) {
            // Staged through LDS so the global stores are 16-byte chunks
            // along rows (whole 128-byte lines per 8 lanes): per wave a
            // [TM][128-byte] tile of one slab of columns (32 f32 or 64 f16),
            // entries of 4 columns at slot q ^ (row % groups) in the row.
            int8_t* tile = ring + wave * (TM * 128);
            auto slab = [&](auto esz_c, auto clip_c, auto form_c) {
                constexpr int ESZ = decltype(esz_c)::value;          // output element bytes
                // columns per slab: 128 bytes of a row where they divide the wave tile
                constexpr int SC = TN < 128 / ESZ ? TN : TN % (128 / ESZ) == 0 ? 128 / ESZ : 32;
                constexpr int GPS = SC / 4;                          // 4-column entries per slab row
                constexpr int E = 4 * ESZ;                           // entry bytes
                constexpr int RB = GPS * E;                          // slab row bytes
                constexpr int CPRW = RB / 16;                        // 16-byte chunks per row
#pragma unroll
                for (int s0 = 0; s0 < TN / SC; ++s0) {
#pragma unroll
                    for (int jj = 0; jj < SC / 32; ++jj) {
                        const int j = s0 * (SC / 32) + jj;
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const int q = jj * 8 + 2 * g + (lane >> 5);
                            const ColFp cp = col_fp(j, g);
#pragma unroll
                            for (int i = 0; i < FM; ++i) {
                                const int r = i * 32 + (lane & 31);
                                const v4f o = values(i, j, g, cp, sa_i[i], clip_c, form_c);
                                int8_t* dst = tile + r * RB + ((q ^ (r % GPS)) * E);
                                if constexpr (ESZ == 4) {
                                    *reinterpret_cast<v4f*>(dst) = o;
                                } else {
                                    _Float16 h[4] = {(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]};
                                    uint2 w;
                                    __builtin_memcpy(&w, h, 8);
                                    *reinterpret_cast<uint2*>(dst) = w;
                                }
                            }
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
                    for (int t = 0; t < TM * CPRW / 64; ++t) {
                        const int idx = t * 64 + lane, r = idx / CPRW, cc = idx % CPRW;
                        const int m = m0 + wm0 + r;
                        const int n = n0 + wn0 + s0 * SC + cc * (16 / ESZ);
                        v4i v;
                        if constexpr (ESZ == 4) {
                            v = *reinterpret_cast<const v4i*>(tile + r * RB + ((cc ^ (r % GPS)) * E));
                        } else {
                            const uint2 lo = *reinterpret_cast<const uint2*>(tile + r * RB + (((2 * cc) ^ (r % GPS)) * E));
                            const uint2 hi = *reinterpret_cast<const uint2*>(tile + r * RB + (((2 * cc + 1) ^ (r % GPS)) * E));
                            v = v4i{(int)lo.x, (int)lo.y, (int)hi.x, (int)hi.y};
                        }
                        if (m < p.m && n < p.n) {
                            char* cptr = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes + (int64_t)n * ESZ;
                            if (n + 16 / ESZ <= p.n) {
                                __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(cptr));
                            } else {
                                // a row's last group of 4 columns (N % 8 == 4, f16)
                                *reinterpret_cast<uint2*>(cptr) = uint2{(uint32_t)v.x, (uint32_t)v.y};
                            }
                        }
                    }
                    __builtin_amdgcn_wave_barrier();
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                }
            };
            using TrueC = std::integral_constant<bool, true>;
            using FalseC = std::integral_constant<bool, false>;
            const bool clip = !(ep.min_clip == -__builtin_inff() && ep.max_clip == __builtin_inff());
            using F0 = std::integral_constant<int, 0>;
            const bool fast = !clip && !ep.add_to;
            const int form = !fast ? 0 : 1 + (ep.bias_fp != nullptr ? 1 : 0) + (relu ? 2 : 0);
            auto run = [&](auto esz_c) {
                if (form == 1) {
                    slab(esz_c, FalseC{}, std::integral_constant<int, 1>{});
                } else if (form == 2) {
                    slab(esz_c, FalseC{}, std::integral_constant<int, 2>{});
                } else if (form == 3) {
                    slab(esz_c, FalseC{}, std::integral_constant<int, 3>{});
                } else if (form == 4) {
                    slab(esz_c, FalseC{}, std::integral_constant<int, 4>{});
                } else if (clip) {
                    slab(esz_c, TrueC{}, F0{});
                } else {
                    slab(esz_c, FalseC{}, F0{});
                }
            };
            if (f16) {
                run(std::integral_constant<int, 2>{});
            } else {
                run(std::integral_constant<int, 4>{});
            }
        } else {
#pragma unroll
            for (int j = 0; j < FN; ++j) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const int n = n0 + wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
                    const ColFp cp = col_fp(j, g);
#pragma unroll
                    for (int i = 0; i < FM; ++i) {
                        const int m = m0 + wm0 + i * 32 + (lane & 31);
                        if (m >= p.m || n >= p.n) {
                            continue;
                        }
                        const v4f o = values(i, j, g, cp, sa_i[i], std::integral_constant<bool, true>{},
                                             std::integral_constant<int, 0>{});
                        char* cptr = static_cast<char*>(p.c) + (int64_t)m * p.ldc_bytes + (int64_t)n * (f16 ? 2 : 4);
                        if (f16) {
                            _Float16 h[4] = {(_Float16)o[0], (_Float16)o[1], (_Float16)o[2], (_Float16)o[3]};
                            uint2 w;
                            __builtin_memcpy(&w, h, 8);
                            *reinterpret_cast<uint2*>(cptr) = w;
                        } else {
                            *reinterpret_cast<v4f*>(cptr) = o;
                        }
                    }
                }
            }
        }
    } else {
        // int32 groups (16-byte-aligned rows: host-checked for C, N % 4 == 0;
        // a last group past N stays within the partials' pitch),
        // staged through the ring so every store is a 16-byte piece of a
        // whole tile row: 32 lanes write one row's BN * 4 bytes. Straight
        // from the accumulator layout a store instruction would touch 32 rows
        // with 32 bytes each, which writes at a fraction of the HBM rate
        // (config 5's 22 MB of partials: 9.6 us against 3 us for the same
        // bytes in row pieces). Passes of PI fragment rows per wave row keep
        // the staged slab within the ring.
        const int32_t floor_v = (MODE == RING_S32 && ep.act == NNOPS_ACT_RELU) ? 0 : INT32_MIN;
        char* cbase;
        int64_t ld;
        if constexpr (MODE == RING_S32) {
            cbase = static_cast<char*>(p.c);
            ld = p.ldc_bytes;
        } else {
            cbase = reinterpret_cast<char*>(sk.part + (int64_t)sp * p.m * sk.ldp);
            ld = (int64_t)sk.ldp * 4;
        }
        constexpr int kRowB = BN * 4 + 16;            // staged row pitch: rows 16 bytes apart in the banks
        constexpr int PI = (WM * FM * 32 * kRowB <= NS * kStage) ? FM
                           : (FM % 2 == 0 && WM * (FM / 2) * 32 * kRowB <= NS * kStage) ? FM / 2 : 1;
        static_assert(WM * PI * 32 * kRowB <= NS * kStage, "int32 staging fits the ring");
        constexpr int kCPR = BN / 4;                  // 16-byte chunks per tile row
        constexpr int kRows = WM * PI * 32;           // staged rows per pass
        static_assert((kRows * kCPR) % (W * 64) == 0, "whole chunks per thread");
        const int wmi = wave / WN;
#pragma unroll
        for (int pass = 0; pass < FM / PI; ++pass) {
#pragma unroll
            for (int ii = 0; ii < PI; ++ii) {
                const int i = pass * PI + ii;
                const int sr = (wmi * PI + ii) * 32 + (lane & 31);
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    v16i a;
                    if constexpr (F16) {
                        a = __builtin_bit_cast(v16i, acc[i][j]);
                    } else {
                        a = acc[i][j];
                    }
#pragma unroll
                    for (int g = 0; g < 4; ++g) {
                        v4i v;
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            v[e] = F16 ? a[4 * g + e] : max(a[4 * g + e], floor_v);
                        }
                        const int col = wn0 + j * 32 + 8 * g + 4 * (lane >> 5);
                        *reinterpret_cast<v4i*>(ring + sr * kRowB + col * 4) = v;
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int q = 0; q < kRows * kCPR / (W * 64); ++q) {
                const int idx = (q * W + wave) * 64 + lane;
                const int sr = idx / kCPR, cc = idx % kCPR;
                const int m = m0 + (sr / (PI * 32)) * TM + (pass * PI + (sr / 32) % PI) * 32 + (sr & 31);
                const int n = n0 + cc * 4;
                const v4i v = *reinterpret_cast<const v4i*>(ring + sr * kRowB + cc * 16);
                if (m < p.m && n < p.n) {
                    // the int32 destination is written once; the partials are
                    // read back by the reduce, so they keep the default policy
                    if constexpr (MODE == RING_S32) {
                        __builtin_nontemporal_store(v, reinterpret_cast<v4i*>(cbase + (int64_t)m * ld + (int64_t)n * 4));
                    } else {
                        *reinterpret_cast<v4i*>(cbase + (int64_t)m * ld + (int64_t)n * 4) = v;
                    }
                }
            }
            if (pass + 1 < FM / PI) {
                __syncthreads();
            }
        }
    }
}

template <int BM, int BN, int WM, int WN, int NS, bool F16, bool TRB, bool TAIL>
void launch_ring_mode(const GemmI8Kern& k, const RingSplit& sk, int mode, bool flip, hipStream_t s)
{
    const unsigned blocks = (unsigned)(((k.m + BM - 1) / BM) * ((k.n + BN - 1) / BN) * sk.splits);
    const dim3 block(WM * WN * 64);
    if constexpr (TRB) {
        // [K,N] B in place; plain A (no u8 flip: its column sums need the copy)
        (void)flip;
        if (mode == RING_S8) {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_S8, false, false, true, TAIL>), dim3(blocks), block, 0, s,
                         k, sk);
        } else if (mode == RING_S32) {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_S32, false, false, true, TAIL>), dim3(blocks), block, 0,
                         s, k, sk);
        } else if (mode == RING_FP) {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_FP, false, false, true, TAIL>), dim3(blocks), block, 0, s,
                         k, sk);
        } else {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_PART, false, false, true, TAIL>), dim3(blocks), block, 0,
                         s, k, sk);
        }
    } else if constexpr (F16) {
        (void)flip;
        if (mode == RING_FP) {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_FP, false, true, false, TAIL>), dim3(blocks), block, 0,
                               s, k, sk);
        } else {
            NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_PART, false, true, false, TAIL>), dim3(blocks), block,
                               0, s, k, sk);
        }
    } else if (flip) {
        NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_PART, true, false, false, TAIL>), dim3(blocks), block, 0, s, k, sk);
    } else if (mode == RING_S8) {
        NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_S8, false, false, false, TAIL>), dim3(blocks), block, 0, s, k, sk);
    } else if (mode == RING_S32) {
        NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_S32, false, false, false, TAIL>), dim3(blocks), block, 0, s, k, sk);
    } else if (mode == RING_FP) {
        NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_FP, false, false, false, TAIL>), dim3(blocks), block, 0, s, k, sk);
    } else {
        NNOPS_LAUNCH((gemm_i8_ring<BM, BN, WM, WN, NS, RING_PART, false, false, false, TAIL>), dim3(blocks), block, 0, s, k, sk);
    }
}

// 128-byte staged rows (whole cache lines: twice the bytes per L2 request of
// 64-byte rows, which is what limits a CU's load rate). Three stage slots
// where the LDS holds them (192x128 tiles: 33.7 -> 32.9 us against two), two
// for the 256x256 and 256x192 tiles, four for the tiles of 128 columns and rows or fewer;
// the 64 x 64 tiles of small grids keep 8 stages in flight (their latency is
// the call's).
template <int BM, int BN, int WM, int WN, bool F16, bool TRB>
void launch_ring_cfg(const GemmI8Kern& k, const RingSplit& sk, int mode, bool flip, hipStream_t s)
{
    constexpr int NS = BM + BN <= 128 ? 8 : BM + BN <= 256 ? 4 : BM + BN <= 384 ? 3 : 2;
    if (k.k % 128 == 0) {
        launch_ring_mode<BM, BN, WM, WN, NS, F16, TRB, false>(k, sk, mode, flip, s);
    } else {
        launch_ring_mode<BM, BN, WM, WN, NS, F16, TRB, true>(k, sk, mode, flip, s);
    }
}

// The tile shapes a plan can name.
template <bool F16, bool TRB>
void launch_ring_tiles(const GemmI8Kern& k, const RingPlan& r, const RingSplit& sk, hipStream_t s)
{
    const bool flip = k.a_xor != 0u;
    auto is = [&](int bm, int bn) { return r.bm == bm && r.bn == bn; };
    if (is(64, 64)) {
        launch_ring_cfg<64, 64, 2, 2, F16, TRB>(k, sk, r.mode, flip, s);
    } else if (is(128, 64)) {
        launch_ring_cfg<128, 64, 2, 2, F16, TRB>(k, sk, r.mode, flip, s);
    } else if (is(128, 128)) {
        launch_ring_cfg<128, 128, 2, 4, F16, TRB>(k, sk, r.mode, flip, s);
    } else if (is(192, 128)) {
        launch_ring_cfg<192, 128, 2, 4, F16, TRB>(k, sk, r.mode, flip, s);
    } else if (is(128, 192) && !TRB) {
        if constexpr (!TRB) {          // (a TRB stage row is a power of two)
            launch_ring_cfg<128, 192, 4, 2, F16, TRB>(k, sk, r.mode, flip, s);
        }
    } else if (is(256, 192) && !TRB) {
        if constexpr (!TRB) {
            launch_ring_cfg<256, 192, 4, 2, F16, TRB>(k, sk, r.mode, flip, s);
        }
    } else if (is(256, 128)) {
        launch_ring_cfg<256, 128, 4, 2, F16, TRB>(k, sk, r.mode, flip, s);
    } else if (is(128, 256)) {
        launch_ring_cfg<128, 256, 2, 4, F16, TRB>(k, sk, r.mode, flip, s);
    } else {
        launch_ring_cfg<256, 256, 2, 4, F16, TRB>(k, sk, r.mode, flip, s);
    }
}

inline RingSplit ring_split(const GemmI8Kern& k, const RingPlan& r, int32_t* part)
{
    RingSplit sk{};
    sk.splits = r.splits;
    sk.kt_per = ((k.k + 127) / 128) / r.splits;
    sk.part = part;
    sk.ldp = (k.n + 3) / 4 * 4;
    return sk;
}

}  // namespace
}  // namespace nnops_amd
