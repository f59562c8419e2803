// Output pass of the fp x q4_1 routes (nnops_hip_fp_output_pass): the Q4_1
// GEMM writes f32 results into the caller's workspace and this pass adds the
// bias, the residual and the epilogue, or runs the gated combine of Linear's
// gated form, writing the f32 / f16 destination.
//
// Kernel
//   fp_out_pass   one thread per 4 consecutive output columns of a row
//                 (16-byte loads of the f32 results when the row allows),
//                 every float operation a separately rounded one, in the
//                 reference's order. Bound: HBM (rows x n x (4 + 4 or 2)
//                 bytes, twice the source columns when gated).
#include "fp_out.hpp"

#include <cmath>

namespace nnops_amd {
namespace {

// 4 consecutive values of the destination's type from q (16 or 8 bytes in one
// load when `vec`), widened.
__device__ __forceinline__ void load4_out(float (&x)[4], const char* q, bool f16, bool vec, int cn)
{
    if (vec && f16) {
        const uint2 w = *reinterpret_cast<const uint2*>(q);
        _Float16 t[4];
        __builtin_memcpy(t, &w, 8);
        x[0] = (float)t[0], x[1] = (float)t[1], x[2] = (float)t[2], x[3] = (float)t[3];
    } else if (vec) {
        const v4f t = *reinterpret_cast<const v4f*>(q);
        x[0] = t[0], x[1] = t[1], x[2] = t[2], x[3] = t[3];
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e < cn) {
                x[e] = f16 ? (float)reinterpret_cast<const _Float16*>(q)[e] : reinterpret_cast<const float*>(q)[e];
            }
        }
    }
}

__global__ __launch_bounds__(256) void fp_out_pass(FpOut p, int cblocks)
{
    const int64_t r = blockIdx.x / cblocks;
    const int c0 = ((blockIdx.x % cblocks) * 256 + threadIdx.x) * 4;
    if (c0 >= p.n) {
        return;
    }
    const bool f16 = p.out_f16 != 0;
    const int es = f16 ? 2 : 4;
    const float* srow = p.src + r * p.ld_src;
    char* orow = static_cast<char*>(p.out) + r * p.ld_out * es;
    const int cn = min(4, p.n - c0);
    // the bias and the destination's values are loaded ahead of the products
    float bg[4] = {0.0f, 0.0f, 0.0f, 0.0f}, bu[4] = {0.0f, 0.0f, 0.0f, 0.0f}, old[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    char* dst = orow + (int64_t)c0 * es;
    const bool dvec = cn == 4 && ((uintptr_t)dst & (4 * es - 1)) == 0;
    if (p.bias != nullptr) {
        const char* b = static_cast<const char*>(p.bias) + (int64_t)c0 * es;
        load4_out(bg, b, f16, cn == 4 && ((uintptr_t)b & (4 * es - 1)) == 0, cn);
        if (p.gated) {
            const char* b2 = b + (int64_t)p.n * es;
            load4_out(bu, b2, f16, cn == 4 && ((uintptr_t)b2 & (4 * es - 1)) == 0, cn);
        }
    }
    if (fp_out_reads_old(p)) {
        load4_out(old, dst, f16, dvec, cn);
    }
    // 16-byte loads of the f32 results where the row segment allows (every
    // split's: slab % 4 == 0 when it is), the K splits' partials summed in
    // split order with four loads in flight
    const bool vec = cn == 4 && (((uintptr_t)(srow + c0)) & 15) == 0 && (p.splits == 1 || p.slab % 4 == 0) &&
                     (!p.gated || (((uintptr_t)(srow + p.n + c0)) & 15) == 0);
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f}, v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (vec) {
        auto sum = [&](const float* s) {
            v4f t = *reinterpret_cast<const v4f*>(s);
            int i = 1;
            for (; i + 3 < p.splits; i += 4) {
                const v4f x0 = *reinterpret_cast<const v4f*>(s + i * p.slab);
                const v4f x1 = *reinterpret_cast<const v4f*>(s + (i + 1) * p.slab);
                const v4f x2 = *reinterpret_cast<const v4f*>(s + (i + 2) * p.slab);
                const v4f x3 = *reinterpret_cast<const v4f*>(s + (i + 3) * p.slab);
                t = (((t + x0) + x1) + x2) + x3;
            }
            for (; i < p.splits; ++i) {
                t += *reinterpret_cast<const v4f*>(s + i * p.slab);
            }
            return t;
        };
        const v4f x = sum(srow + c0);
        a[0] = x[0], a[1] = x[1], a[2] = x[2], a[3] = x[3];
        if (p.gated) {
            const v4f y = sum(srow + p.n + c0);
            v[0] = y[0], v[1] = y[1], v[2] = y[2], v[3] = y[3];
        }
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e < cn) {
                a[e] = srow[c0 + e];
                v[e] = p.gated ? srow[p.n + c0 + e] : 0.0f;
                for (int i = 1; i < p.splits; ++i) {
                    a[e] += srow[i * p.slab + c0 + e];
                    v[e] += p.gated ? srow[i * p.slab + p.n + c0 + e] : 0.0f;
                }
            }
        }
    }
    float y[4];
    if (p.silu) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            y[e] = fp_out_silu(p, a[e], v[e], bg[e], bu[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (e < cn && !p.silu) {
            y[e] = fp_out_value(p, a[e], v[e], old[e], bg[e], bu[e]);
        }
    }
    if (dvec && f16) {
        const _Float16 h[4] = {(_Float16)y[0], (_Float16)y[1], (_Float16)y[2], (_Float16)y[3]};
        uint2 w;
        __builtin_memcpy(&w, h, 8);
        *reinterpret_cast<uint2*>(dst) = w;
    } else if (dvec) {
        *reinterpret_cast<v4f*>(dst) = v4f{y[0], y[1], y[2], y[3]};
    } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (e < cn) {
                fp_out_store(p, orow, c0 + e, y[e]);
            }
        }
    }
}

bool gate_act_ok(int a)
{
    return a == NNOPS_ACT_NONE || a == NNOPS_ACT_RELU || a == NNOPS_ACT_GELU || a == NNOPS_ACT_SIGMOID ||
           a == NNOPS_ACT_TANH || a == NNOPS_ACT_SILU;
}

}  // namespace

int make_fp_out(const NnopsFpOutArgs* a, FpOut& p)
{
    if (a == nullptr || a->rows < 0 || a->n < 0 || a->n > INT32_MAX) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (a->out == nullptr || a->ld_out < a->n) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (a->act < NNOPS_ACT_NONE || a->act > NNOPS_ACT_RELU6 || (a->gated && !gate_act_ok(a->gate_act)) ||
        (a->gated && a->add_to && a->residual_pre) || (a->gated && a->matmul_order)) {
        return NNOPS_UNSUPPORTED;
    }
    p = FpOut{};
    p.src = a->src;
    p.ld_src = a->ld_src;
    p.out = a->out;
    p.ld_out = a->ld_out;
    p.rows = a->rows;
    p.n = (int)a->n;
    p.out_f16 = a->out_f16 != 0;
    p.bias = a->bias;
    p.ep.act = a->act;
    p.ep.act_alpha = a->act_alpha;
    p.ep.act_beta = a->act_beta;
    p.ep.min_clip = a->min_clip;
    p.ep.max_clip = a->max_clip;
    p.ep.out_kind = p.out_f16 ? NNOPS_OUT_F16 : NNOPS_OUT_F32;
    p.add_to = a->add_to != 0;
    p.residual_pre = a->residual_pre != 0;
    p.gated = a->gated != 0;
    p.gate_act = a->gate_act;
    p.gate_alpha = a->gate_alpha;
    p.gate_beta = a->gate_beta;
    p.gate_limit = a->gate_limit;
    p.splits = 1;
    p.mm = a->matmul_order != 0;
    p.alpha = a->alpha;
    p.beta = a->beta;
    p.silu = p.gated && p.gate_act == NNOPS_ACT_SILU && std::isinf(p.gate_limit) && p.ep.act == NNOPS_ACT_NONE &&
             p.ep.min_clip == -INFINITY && p.ep.max_clip == INFINITY && !p.add_to;
    return NNOPS_OK;
}

void launch_fp_out_pass(const FpOut& p, hipStream_t s)
{
    const int64_t cblocks = ((int64_t)p.n + 1023) / 1024;
    NNOPS_LAUNCH(fp_out_pass, dim3((unsigned)(cblocks * p.rows)), dim3(256), 0, s, p, (int)cblocks);
}

}  // namespace nnops_amd

using namespace nnops_amd;

extern "C" int nnops_hip_fp_output_pass(const NnopsFpOutArgs* a, void* stream)
{
    const TimingDisarm disarm;
    if (a == nullptr || a->rows < 0 || a->n < 0 || a->n > INT32_MAX) {
        return NNOPS_INVALID_ARGUMENT;
    }
    if (a->rows == 0 || a->n == 0) {
        return NNOPS_OK;
    }
    if (a->src == nullptr || a->ld_src < (a->gated ? 2 : 1) * a->n) {
        return NNOPS_INVALID_ARGUMENT;
    }
    FpOut p;
    if (const int rc = make_fp_out(a, p); rc != NNOPS_OK) {
        return rc;
    }
    if ((a->n + 1023) / 1024 * a->rows > INT32_MAX) {
        return NNOPS_UNSUPPORTED;
    }
    launch_fp_out_pass(p, static_cast<hipStream_t>(stream));
    return hipGetLastError() == hipSuccess ? NNOPS_OK : NNOPS_INTERNAL;
}
