// Kernels of the mixers beyond grouped-query attention, and of blocks with norms on both
// sides of a branch: the gated close of a branch, a clamped gated activation, the blends of
// a token with the one before it, two recurrences with a matrix state per head (decay per key
// channel; scalar decay), a short causal convolution, a gated group norm, the common close of
// two branches that run side by side, and what attention over a cached latent needs around its
// kernel (norms, rotation and page write, rotation of the queries, one small product per head).
//
// Statistics, gates, decays, exponentials, angles and states are float32 whatever the compute
// dtype; a value is rounded once, where it is stored in the compute dtype.
//
// Sequences: kernels that carry state walk the tokens of each sequence of the step in order.
// seq_qstart [S + 1] gives each sequence's tokens among the step's, seq_rows [S] its row of
// the state tensor [rows, stride] (float32).
#include "common.h"
#include "mfma.h"
#include "recurrent.h"

__device__ __forceinline__ float soc_sigmoid(float x) { return 1.f / (1.f + expf(-x)); }

__device__ __forceinline__ void store8(float* p, const float (&x)[8]) {
    *reinterpret_cast<float4*>(p) = make_float4(x[0], x[1], x[2], x[3]);
    *reinterpret_cast<float4*>(p + 4) = make_float4(x[4], x[5], x[6], x[7]);
}
__device__ __forceinline__ void store8(bf16* p, const float (&x)[8]) {
    *reinterpret_cast<uint4*>(p) = make_uint4(pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(x[4], x[5]),
                                              pack_bf16x2(x[6], x[7]));
}


// ---- the close of a branch ---------------------------------------------------------------------
// residual += mult * gain * g / rms(g) with g = y * sigmoid(logits + bias) (no gate: g = y); the logits are the
// first d elements of rows of ldg elements (they may be columns of a wider product);
// then, if next_gain is given, out = residual / rms(residual) * next_gain. y is in the compute dtype, or float32 if
// y_f32; y_bias (float32 [d], or null) is added to it first.
template <typename T>
__device__ __forceinline__ float branch_result(const void* y, int y_f32, const float* y_bias, size_t at, int c) {
    const float v = y_f32 ? ((const float*)y)[at] : to_float(((const T*)y)[at]);
    return y_bias ? v + y_bias[c] : v;
}

template <typename T>
__global__ void __launch_bounds__(256)
gated_norm_add_kernel(float* __restrict__ residual, const void* __restrict__ y, int y_f32, const float* __restrict__ y_bias,
                      const T* __restrict__ logits, int ldg,
                      const float* __restrict__ bias, const float* __restrict__ gain, float eps, float mult,
                      const float* __restrict__ next_gain, float next_eps, T* __restrict__ out, int d) {
    __shared__ float scratch[16];
    const size_t base = (size_t)blockIdx.x * d, gbase = (size_t)blockIdx.x * ldg;
    float ss = 0.f;
    for (int c = threadIdx.x; c < d; c += blockDim.x) {
        float g = branch_result<T>(y, y_f32, y_bias, base + c, c);
        if (logits) g *= soc_sigmoid(to_float(logits[gbase + c]) + bias[c]);
        ss += g * g;
    }
    ss = block_sum(ss, scratch);
    const float scale = mult / sqrtf(ss / (float)d + eps);
    float rr = 0.f;
    for (int c = threadIdx.x; c < d; c += blockDim.x) {
        float g = branch_result<T>(y, y_f32, y_bias, base + c, c);
        if (logits) g *= soc_sigmoid(to_float(logits[gbase + c]) + bias[c]);
        const float r = residual[base + c] + scale * gain[c] * g;
        residual[base + c] = r;
        rr += r * r;
    }
    if (!next_gain) return;
    rr = block_sum(rr, scratch);
    const float inv = 1.f / sqrtf(rr / (float)d + next_eps);
    for (int c = threadIdx.x; c < d; c += blockDim.x)
        out[base + c] = from_float<T>(residual[base + c] * inv * next_gain[c]);
}

// The same with the row in registers (PER elements per thread, d <= 256 * PER): every element is
// read once, all loads are issued before the first is used.
template <typename T, int PER>
__global__ void __launch_bounds__(256)
gated_norm_add_regs_kernel(float* __restrict__ residual, const void* __restrict__ y, int y_f32, const float* __restrict__ y_bias,
                           const T* __restrict__ logits, int ldg,
                           const float* __restrict__ bias, const float* __restrict__ gain, float eps, float mult,
                           const float* __restrict__ next_gain, float next_eps, T* __restrict__ out, int d) {
    __shared__ float scratch[16];
    const size_t base = (size_t)blockIdx.x * d, gbase = (size_t)blockIdx.x * ldg;
    float g[PER], res[PER], gate[PER], gn[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        const bool in = c < d;
        g[i] = in ? branch_result<T>(y, y_f32, y_bias, base + c, c) : 0.f;
        gate[i] = (in && logits) ? to_float(logits[gbase + c]) + bias[c] : 0.f;
        res[i] = in ? residual[base + c] : 0.f;
        gn[i] = in ? gain[c] : 0.f;
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        if (logits) g[i] *= soc_sigmoid(gate[i]);
        ss += g[i] * g[i];
    }
    ss = block_sum(ss, scratch);
    const float scale = mult / sqrtf(ss / (float)d + eps);
    float rr = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        res[i] += scale * gn[i] * g[i];
        if (c < d) residual[base + c] = res[i];
        rr += res[i] * res[i];
    }
    if (!next_gain) return;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        gn[i] = c < d ? next_gain[c] : 0.f;
    }
    rr = block_sum(rr, scratch);
    const float inv = 1.f / sqrtf(rr / (float)d + next_eps);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        if (c < d) out[base + c] = from_float<T>(res[i] * inv * gn[i]);
    }
}

// The same again for widths that are multiples of 8, eight consecutive elements per load (16 bytes of
// bfloat16, 32 of float32), CH such pieces per thread (d <= 2048 * CH); the next norm's gain comes with
// the first loads, so the kernel waits for memory once.
template <typename T, int CH>
__global__ void __launch_bounds__(256)
gated_norm_add_vec8_kernel(float* __restrict__ residual, const void* __restrict__ y, int y_f32, const float* __restrict__ y_bias,
                           const T* __restrict__ logits, int ldg,
                           const float* __restrict__ bias, const float* __restrict__ gain, float eps, float mult,
                           const float* __restrict__ next_gain, float next_eps, T* __restrict__ out, int d) {
    __shared__ float scratch[16];
    const size_t base = (size_t)blockIdx.x * d, gbase = (size_t)blockIdx.x * ldg;
    float g[CH][8], res[CH][8], gate[CH][8], gn[CH][8], nx[CH][8];
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = (threadIdx.x + i * 256) * 8;
        if (c < d) {
            if (y_f32) VecLoad<float, 8>::load((const float*)y + base + c, g[i]);
            else VecLoad<T, 8>::load((const T*)y + base + c, g[i]);
            if (y_bias) {
                float yb[8];
                VecLoad<float, 8>::load(y_bias + c, yb);
#pragma unroll
                for (int e = 0; e < 8; ++e) g[i][e] += yb[e];
            }
            VecLoad<float, 8>::load(residual + base + c, res[i]);
            VecLoad<float, 8>::load(gain + c, gn[i]);
            if (logits) {
                float b[8];
                VecLoad<T, 8>::load(logits + gbase + c, gate[i]);
                VecLoad<float, 8>::load(bias + c, b);
#pragma unroll
                for (int e = 0; e < 8; ++e) gate[i][e] += b[e];
            }
            if (next_gain) VecLoad<float, 8>::load(next_gain + c, nx[i]);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) g[i][e] = res[i][e] = gn[i][e] = gate[i][e] = nx[i][e] = 0.f;
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (logits) g[i][e] *= soc_sigmoid(gate[i][e]);
            ss += g[i][e] * g[i][e];
        }
    ss = block_sum(ss, scratch);
    const float scale = mult / sqrtf(ss / (float)d + eps);
    float rr = 0.f;
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = (threadIdx.x + i * 256) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            res[i][e] += scale * gn[i][e] * g[i][e];
            rr += res[i][e] * res[i][e];
        }
        if (c < d) store8(residual + base + c, res[i]);
    }
    if (!next_gain) return;
    rr = block_sum(rr, scratch);
    const float inv = 1.f / sqrtf(rr / (float)d + next_eps);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
        const int c = (threadIdx.x + i * 256) * 8;
#pragma unroll
        for (int e = 0; e < 8; ++e) res[i][e] *= inv * nx[i][e];
        if (c < d) store8(out + base + c, res[i]);
    }
}

template <typename T>
static void launch_gated_norm_add(float* residual, const void* y, int y_f32, const float* y_bias, const void* logits, int ldg, const float* bias, const float* gain,
                                  float eps, float mult, const float* next_gain, float next_eps, void* out, int N, int d,
                                  hipStream_t stream) {
#define SOC_GNA(PER)                                                                                                    \
    hipLaunchKernelGGL((gated_norm_add_regs_kernel<T, PER>), dim3(N), dim3(256), 0, stream, residual, y, y_f32, y_bias, \
                       (const T*)logits, ldg, bias, gain, eps, mult, next_gain, next_eps, (T*)out, d)
#define SOC_GNA8(CH)                                                                                                    \
    hipLaunchKernelGGL((gated_norm_add_vec8_kernel<T, CH>), dim3(N), dim3(256), 0, stream, residual, y, y_f32, y_bias,  \
                       (const T*)logits, ldg, bias, gain, eps, mult, next_gain, next_eps, (T*)out, d)
    // (pieces of eight elements: the width, the logits' rows and their first element all sit at multiples of 8)
    const bool by8 = d % 8 == 0 && ldg % 8 == 0 && ((uintptr_t)logits % (8 * sizeof(T))) == 0 &&
                     ((uintptr_t)y % (y_f32 ? 32 : 8 * sizeof(T))) == 0;
    if (by8 && d <= 2048) SOC_GNA8(1);
    else if (by8 && d <= 4096) SOC_GNA8(2);
    else if (by8 && d <= 8192) SOC_GNA8(4);
    else if (d <= 1024) SOC_GNA(4);
    else if (d <= 2048) SOC_GNA(8);
    else if (d <= 4096) SOC_GNA(16);
    else if (d <= 8192) SOC_GNA(32);
    else
        hipLaunchKernelGGL(gated_norm_add_kernel<T>, dim3(N), dim3(256), 0, stream, residual, y, y_f32, y_bias, (const T*)logits,
                           ldg, bias, gain, eps, mult, next_gain, next_eps, (T*)out, d);
}

SOC_EXPORT int soc_gated_norm_add(float* residual, const void* y, int y_f32, const float* y_bias, const void* logits, int ldg, const float* bias,
                                  const float* gain, float eps, float mult, const float* next_gain, float next_eps,
                                  void* out, int N, int d, int dtype, hipStream_t stream) {
    if (N <= 0) return 0;
    if (dtype == 0) launch_gated_norm_add<float>(residual, y, y_f32, y_bias, logits, ldg, bias, gain, eps, mult, next_gain, next_eps, out, N, d, stream);
    else launch_gated_norm_add<bf16>(residual, y, y_f32, y_bias, logits, ldg, bias, gain, eps, mult, next_gain, next_eps, out, N, d, stream);
    return soc_last_error();
}

// ---- two branches into the stream at once -----------------------------------------------------------
// residual += scale1 * branch1 + scale2 * branch2 (a scale of null multiplies by one; a branch of null is none),
// then, if next_gain is given, out = residual / rms(residual) * next_gain. A branch is [N, d] in the compute dtype
// (parts 0), float32 partial sums [parts, N, d] added in order, or (top > 0) the weighted sum of a token's experts:
// weight[n, r] times row place[n top + r] of y (float32, by place), r < top. One workgroup per row.
struct BranchIn {
    const void* y;
    int parts;
    const int* place;
    const float* weight;
    int top;
    const float* scale;
};

template <typename T, int V>
__device__ __forceinline__ void branch_load(const BranchIn& b, int n, size_t total, int d, int c, float (&x)[V]) {
    if (b.top > 0) {
#pragma unroll
        for (int e = 0; e < V; ++e) x[e] = 0.f;
        for (int r = 0; r < b.top; ++r) {
            float t[V];
            const float w = b.weight[(size_t)n * b.top + r];
            VecLoad<float, V>::load((const float*)b.y + (size_t)b.place[(size_t)n * b.top + r] * d + c, t);
#pragma unroll
            for (int e = 0; e < V; ++e) x[e] = fmaf(w, t[e], x[e]);
        }
    } else if (b.parts > 0) {
        VecLoad<float, V>::load((const float*)b.y + (size_t)n * d + c, x);
        for (int s = 1; s < b.parts; ++s) {
            float t[V];
            VecLoad<float, V>::load((const float*)b.y + (size_t)s * total + (size_t)n * d + c, t);
#pragma unroll
            for (int e = 0; e < V; ++e) x[e] += t[e];
        }
    } else {
        VecLoad<T, V>::load((const T*)b.y + (size_t)n * d + c, x);
    }
    if (b.scale) {
        float g[V];
        VecLoad<float, V>::load(b.scale + c, g);
#pragma unroll
        for (int e = 0; e < V; ++e) x[e] *= g[e];
    }
}

// PER pieces of V elements per thread: the row stays in registers (d <= 256 * V * PER, d a multiple of V).
template <typename T, int V, int PER>
__global__ void __launch_bounds__(256)
branches_add_kernel(float* __restrict__ residual, BranchIn first, BranchIn second, const float* __restrict__ next_gain,
                    float next_eps, T* __restrict__ out, int N, int d) {
    __shared__ float scratch[16];
    const int n = blockIdx.x;
    const size_t base = (size_t)n * d, total = (size_t)N * d;
    float res[PER][V], nx[PER][V], rr = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = (threadIdx.x + i * 256) * V;
        if (c < d) {
            float a[V], b[V];
            VecLoad<float, V>::load(residual + base + c, res[i]);
            branch_load<T, V>(first, n, total, d, c, a);
            if (second.y) branch_load<T, V>(second, n, total, d, c, b);
            if (next_gain) VecLoad<float, V>::load(next_gain + c, nx[i]);
#pragma unroll
            for (int e = 0; e < V; ++e) {
                res[i][e] += second.y ? a[e] + b[e] : a[e];
                rr += res[i][e] * res[i][e];
            }
            if constexpr (V == 8) store8(residual + base + c, res[i]);
            else {
#pragma unroll
                for (int e = 0; e < V; ++e) residual[base + c + e] = res[i][e];
            }
        }
    }
    if (!next_gain) return;
    rr = block_sum(rr, scratch);
    const float inv = 1.f / sqrtf(rr / (float)d + next_eps);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = (threadIdx.x + i * 256) * V;
        if (c < d) {
#pragma unroll
            for (int e = 0; e < V; ++e) res[i][e] *= inv * nx[i][e];
            if constexpr (V == 8) store8(out + base + c, res[i]);
            else {
#pragma unroll
                for (int e = 0; e < V; ++e) out[base + c + e] = from_float<T>(res[i][e]);
            }
        }
    }
}

template <typename T>
static int launch_branches_add(float* residual, const BranchIn& a, const BranchIn& b, const float* next_gain, float next_eps, void* out,
                               int N, int d, hipStream_t stream) {
#define SOC_BA(V, PER) hipLaunchKernelGGL((branches_add_kernel<T, V, PER>), dim3(N), dim3(256), 0, stream, residual, a, b, next_gain, next_eps, (T*)out, N, d)
    if (d % 8 == 0 && d <= 2048) SOC_BA(8, 1);
    else if (d % 8 == 0 && d <= 4096) SOC_BA(8, 2);
    else if (d % 8 == 0 && d <= 8192) SOC_BA(8, 4);
    else if (d % 8 == 0 && d <= 16384) SOC_BA(8, 8);
    else if (d <= 1024) SOC_BA(1, 4);
    else if (d <= 4096) SOC_BA(1, 16);
    else if (d <= 16384) SOC_BA(1, 64);
    else return (int)hipErrorInvalidValue;
#undef SOC_BA
    return soc_last_error();
}

SOC_EXPORT int soc_branches_add(float* residual, const void* y1, int parts1, const int* place1, const float* weight1, int top1,
                                const float* scale1, const void* y2, int parts2, const int* place2, const float* weight2, int top2,
                                const float* scale2, const float* next_gain, float next_eps, void* out, int N, int d, int dtype,
                                hipStream_t stream) {
    if (N <= 0) return 0;
    if (!y1 || parts1 < 0 || parts2 < 0 || (top1 > 0 && (!place1 || !weight1)) || (top2 > 0 && (!place2 || !weight2)) || (next_gain && !out))
        return (int)hipErrorInvalidValue;
    const BranchIn a{y1, parts1, place1, weight1, top1, scale1}, b{y2, parts2, place2, weight2, top2, scale2};
    if (dtype == 0) return launch_branches_add<float>(residual, a, b, next_gain, next_eps, out, N, d, stream);
    return launch_branches_add<bf16>(residual, a, b, next_gain, next_eps, out, N, d, stream);
}

// ---- g * sigmoid(slope g) * (u + 1), g = min(gate, limit), u = clamp(up, -limit, limit) ---------
// gate and up are the first 2 ff elements of rows of ld elements.
template <typename T>
__global__ void glu_clamped_kernel(const T* __restrict__ gate_up, T* __restrict__ out, size_t total, int ff, int ld,
                                   float limit, float slope) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const size_t n = i / ff, c = i % ff;
    const float g = fminf(to_float(gate_up[n * ld + c]), limit);
    const float u = fminf(fmaxf(to_float(gate_up[n * ld + ff + c]), -limit), limit);
    out[i] = from_float<T>(g * soc_sigmoid(slope * g) * (u + 1.f));
}

// (eight consecutive elements per lane where ff is a multiple of 8)
template <typename T>
__global__ void glu_clamped_vec8_kernel(const T* __restrict__ gate_up, T* __restrict__ out, size_t groups, int ff, int ld,
                                        float limit, float slope) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= groups) return;
    const int per_row = ff / 8;
    const size_t n = i / per_row, c = (i % per_row) * 8;
    float g[8], u[8], y[8];
    VecLoad<T, 8>::load(gate_up + n * ld + c, g);
    VecLoad<T, 8>::load(gate_up + n * ld + ff + c, u);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const float gg = fminf(g[e], limit), uu = fminf(fmaxf(u[e], -limit), limit);
        y[e] = gg * soc_sigmoid(slope * gg) * (uu + 1.f);
    }
    store8(out + n * ff + c, y);
}

SOC_EXPORT int soc_glu_clamped(const void* gate_up, void* out, int N, int ff, int ld, float limit, float slope, int dtype,
                               hipStream_t stream) {
    const size_t total = (size_t)N * ff;
    if (total == 0) return 0;
    if (ld < 2 * ff) return (int)hipErrorInvalidValue;
    if (ff % 8 == 0 && ld % 8 == 0) {
        const size_t groups = total / 8;
        const dim3 grid((unsigned)((groups + 255) / 256));
        if (dtype == 0)
            hipLaunchKernelGGL(glu_clamped_vec8_kernel<float>, grid, dim3(256), 0, stream, (const float*)gate_up, (float*)out,
                               groups, ff, ld, limit, slope);
        else
            hipLaunchKernelGGL(glu_clamped_vec8_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)gate_up, (bf16*)out,
                               groups, ff, ld, limit, slope);
        return soc_last_error();
    }
    const dim3 grid((unsigned)((total + 255) / 256));
    if (dtype == 0)
        hipLaunchKernelGGL(glu_clamped_kernel<float>, grid, dim3(256), 0, stream, (const float*)gate_up, (float*)out,
                           total, ff, ld, limit, slope);
    else
        hipLaunchKernelGGL(glu_clamped_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)gate_up, (bf16*)out,
                           total, ff, ld, limit, slope);
    return soc_last_error();
}

// ---- blends of a token's input with the one before it ---------------------------------------------
// out[s, n, c] = h[n, c] + (prev[n, c] - h[n, c]) * mu[s, c]; prev of a sequence's first token of
// the step is what the row's state holds, which then becomes the input of its last token. Grid
// (chunks of SHIFT_CHUNK tokens, sequences, blocks of 256 columns): the workgroups of a sequence's
// first chunk are the only ones that touch the state, each thread its own column, reading before writing.
constexpr int SHIFT_CHUNK = 8;

template <typename T>
__global__ void __launch_bounds__(256)
token_shift_kernel(const T* __restrict__ h, const float* __restrict__ mu, int n_streams, float* __restrict__ state,
                   size_t stride, int offset, const int* __restrict__ seq_qstart, const int* __restrict__ seq_rows,
                   T* __restrict__ out, int N, int d) {
    const int seq = blockIdx.y;
    const int lo = seq_qstart[seq], hi = seq_qstart[seq + 1];
    const int first = lo + blockIdx.x * SHIFT_CHUNK;
    if (first >= hi) return;
    const int last = min(first + SHIFT_CHUNK, hi);
    float* kept = state + (size_t)seq_rows[seq] * stride + offset;
    const int c = blockIdx.z * blockDim.x + threadIdx.x;
    if (c < d) {
        float prev = first == lo ? kept[c] : to_float(h[(size_t)(first - 1) * d + c]);
        for (int n = first; n < last; ++n) {
            const float cur = to_float(h[(size_t)n * d + c]);
            const float diff = prev - cur;
            for (int s = 0; s < n_streams; ++s)
                out[((size_t)s * N + n) * d + c] = from_float<T>(cur + diff * mu[(size_t)s * d + c]);
            prev = cur;
        }
        if (first == lo) kept[c] = to_float(h[(size_t)(hi - 1) * d + c]);
    }
}

SOC_EXPORT int soc_token_shift(const void* h, const float* mu, int n_streams, float* state, long long stride, int offset,
                               const int* seq_qstart, const int* seq_rows, void* out, int N, int d, int n_seqs,
                               int max_q_len, int dtype, hipStream_t stream) {
    if (N <= 0 || n_seqs <= 0) return 0;
    if (n_seqs > 65535 || (d + 255) / 256 > 65535) return (int)hipErrorInvalidValue;
    const dim3 grid((max_q_len + SHIFT_CHUNK - 1) / SHIFT_CHUNK, n_seqs, (d + 255) / 256);
    if (dtype == 0)
        hipLaunchKernelGGL(token_shift_kernel<float>, grid, dim3(256), 0, stream, (const float*)h, mu, n_streams, state,
                           (size_t)stride, offset, seq_qstart, seq_rows, (float*)out, N, d);
    else
        hipLaunchKernelGGL(token_shift_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)h, mu, n_streams, state,
                           (size_t)stride, offset, seq_qstart, seq_rows, (bf16*)out, N, d);
    return soc_last_error();
}

// ---- decay = exp(-exp(tanh(t) W2^T + w0)) --------------------------------------------------------
// t [N, rank] float32; W2 transposed, [rank, C] (consecutive threads read consecutive elements); grid (blocks
// of 256 channels, tokens), a thread per channel, tanh(t) of the token in LDS.
// TOK tokens to a workgroup share what it reads of W2: with one token the kernel reads all of W2 per token out of
// L2 (2,048 tokens, rank 64, 2,560 channels, bf16: 61 us; with eight, 29). Eight where that still leaves every
// compute unit a workgroup. Same additions in the same order.
template <typename T, int TOK>
__global__ void __launch_bounds__(256)
wkv_decay_kernel(const float* __restrict__ t, const T* __restrict__ w2, const float* __restrict__ w0,
                 float* __restrict__ out, int N, int C, int rank) {
    extern __shared__ float th[];                       // [rank][TOK]
    const int n0 = blockIdx.y * TOK;
    for (int i = threadIdx.x; i < rank * TOK; i += blockDim.x)
        th[i] = tanhf(t[(size_t)min(n0 + i % TOK, N - 1) * rank + i / TOK]);
    __syncthreads();
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c < C) {
        float z[TOK];
#pragma unroll
        for (int q = 0; q < TOK; ++q) z[q] = 0.f;
#pragma unroll 8
        for (int j = 0; j < rank; ++j) {
            const float wj = to_float(w2[(size_t)j * C + c]);
#pragma unroll
            for (int q = 0; q < TOK; ++q) z[q] = fmaf(th[j * TOK + q], wj, z[q]);
        }
        const float base = w0[c];
#pragma unroll
        for (int q = 0; q < TOK; ++q)
            if (n0 + q < N) out[(size_t)(n0 + q) * C + c] = expf(-expf(z[q] + base));
    }
}

SOC_EXPORT int soc_wkv_decay(const float* t, const void* w2, const float* w0, float* out, int N, int C, int rank,
                             int dtype, hipStream_t stream) {
    if (N <= 0) return 0;
    if (N > 65535) return (int)hipErrorInvalidValue;
    const int blocks = (C + 255) / 256;
    const bool many = (long)blocks * ((N + 7) / 8) >= 256 && rank <= 1024;
#define SOC_DECAY(T, TOK)                                                                                               \
    hipLaunchKernelGGL((wkv_decay_kernel<T, TOK>), dim3(blocks, (N + TOK - 1) / TOK), dim3(256), (size_t)rank * TOK * 4, \
                       stream, t, (const T*)w2, w0, out, N, C, rank)
    if (dtype == 0) { if (many) SOC_DECAY(float, 8); else SOC_DECAY(float, 1); }
    else { if (many) SOC_DECAY(bf16, 8); else SOC_DECAY(bf16, 1); }
#undef SOC_DECAY
    return soc_last_error();
}

// ---- the two recurrences with a matrix state per head ---------------------------------------------------
// A workgroup of 256 threads owns CW columns of one head's state S [keys, columns] for one sequence, in
// registers: thread (part, column) holds keys part * KPT .. (part + 1) * KPT - 1 of its column (PARTS * CW =
// 256; consecutive lanes are consecutive columns). Columns never meet in the recurrence, so a head is
// spread over as many workgroups as fill the GPU (CW = 16 when sequences and heads alone give too few,
// else 64). Tokens go in batches: what all threads need of a batch (per key: r, k, decay; or B,
// C) is staged through LDS; the next batch's global loads are issued before the current batch is computed
// and land in LDS after it; the partial sums of a column's PARTS threads meet in LDS once per batch.
// Decay per key channel: o_t[j] = sum_i r_t[i] (S[i, j] + u[i] k_t[i] v_t[j]); S[i, j] <- w_t[i] S[i, j] +
// k_t[i] v_t[j]. o goes out in float32; its norm over the head is another kernel's.
template <typename T, int DK, int CW>
__global__ void __launch_bounds__(256)
wkv_kernel(const T* __restrict__ r, const T* __restrict__ k, const T* __restrict__ v, const float* __restrict__ decay,
           const float* __restrict__ bonus, int H, int D, float* __restrict__ state, size_t stride, int offset,
           const int* __restrict__ seq_qstart, const int* __restrict__ seq_rows, int below, float* __restrict__ out) {
    constexpr int REC_TB = rec_batch(DK), PARTS = 256 / CW, KPT = DK / PARTS, STAGE = (REC_TB * DK + 255) / 256;
    __shared__ float sr[2][REC_TB][DK], sk[2][REC_TB][DK], sw[2][REC_TB][DK];
    __shared__ float red[REC_TB][PARTS][CW], su[DK];
    const int blocks = (D + CW - 1) / CW;
    const int head = blockIdx.x / blocks, seq = blockIdx.y, tid = threadIdx.x;
    const int lo = seq_qstart[seq], hi = seq_qstart[seq + 1];
    if (lo >= hi || hi - lo >= below) return;
    const int col0 = (blockIdx.x % blocks) * CW;
    const int col = col0 + tid % CW, part = tid / CW, i0 = part * KPT;
    const bool live = col < D;
    float* S = state + (size_t)seq_rows[seq] * stride + offset + (size_t)head * D * D;
    const size_t C = (size_t)H * D, hoff = (size_t)head * D;
    float s[KPT];
#pragma unroll
    for (int ii = 0; ii < KPT; ++ii) s[ii] = (live && i0 + ii < D) ? S[(size_t)(i0 + ii) * D + col] : 0.f;
    for (int i = tid; i < DK; i += 256) su[i] = i < D ? bonus[head * D + i] : 0.f;

    float fr[STAGE], fk[STAGE], fw[STAGE], fv[REC_TB];
    auto fetch = [&](int n0) {
#pragma unroll
        for (int q = 0; q < STAGE; ++q) {
            const int e = tid + q * 256, t = e / DK, i = e % DK;
            const bool in = t < REC_TB && n0 + t < hi && i < D;
            const size_t at = (size_t)(n0 + t) * C + hoff + i;
            fr[q] = in ? to_float(r[at]) : 0.f;
            fk[q] = in ? to_float(k[at]) : 0.f;
            fw[q] = in ? decay[at] : 0.f;
        }
#pragma unroll
        for (int t = 0; t < REC_TB; ++t)
            fv[t] = (live && n0 + t < hi) ? to_float(v[(size_t)(n0 + t) * C + hoff + col]) : 0.f;
    };
    auto land = [&](int buf) {
#pragma unroll
        for (int q = 0; q < STAGE; ++q) {
            const int e = tid + q * 256, t = e / DK, i = e % DK;
            if (t < REC_TB) { sr[buf][t][i] = fr[q]; sk[buf][t][i] = fk[q]; sw[buf][t][i] = fw[q]; }
        }
    };
    fetch(lo);
    land(0);
    lds_barrier();
    int buf = 0;
    for (int n0 = lo; n0 < hi; n0 += REC_TB, buf ^= 1) {
        const int nb = min(REC_TB, hi - n0);
        const bool more = n0 + REC_TB < hi;
        float vj[REC_TB];
#pragma unroll
        for (int t = 0; t < REC_TB; ++t) vj[t] = fv[t];
        if (more) fetch(n0 + REC_TB);
#pragma unroll
        for (int t = 0; t < REC_TB; ++t) {
            if (t < nb) {
                float acc = 0.f;
#pragma unroll
                for (int ii = 0; ii < KPT; ++ii) {
                    const float kv = sk[buf][t][i0 + ii] * vj[t];
                    acc = fmaf(sr[buf][t][i0 + ii], fmaf(su[i0 + ii], kv, s[ii]), acc);
                    s[ii] = fmaf(sw[buf][t][i0 + ii], s[ii], kv);
                }
                red[t][part][tid % CW] = acc;
            }
        }
        lds_barrier();
        for (int f = tid; f < REC_TB * CW; f += 256) {
            const int t = f / CW, cl = f % CW;
            if (t < nb && col0 + cl < D) {
                float o = 0.f;
#pragma unroll
                for (int pp = 0; pp < PARTS; ++pp) o += red[t][pp][cl];
                out[(size_t)(n0 + t) * C + hoff + col0 + cl] = o;
            }
        }
        if (more) land(buf ^ 1);
        lds_barrier();
    }
    if (live) {
#pragma unroll
        for (int ii = 0; ii < KPT; ++ii)
            if (i0 + ii < D) S[(size_t)(i0 + ii) * D + col] = s[ii];
    }
}

template <typename T, int DK>
static void launch_wkv(const void* r, const void* k, const void* v, const float* decay, const float* bonus, int H, int D,
                       float* state, long long stride, int offset, const int* seq_qstart, const int* seq_rows, int below, float* out,
                       int n_seqs, int cw, hipStream_t stream) {
#define SOC_WKV_LAUNCH(CW)                                                                                                  \
    hipLaunchKernelGGL((wkv_kernel<T, DK, CW>), dim3(H * ((D + CW - 1) / CW), n_seqs), dim3(256), 0, stream, (const T*)r, \
                       (const T*)k, (const T*)v, decay, bonus, H, D, state, (size_t)stride, offset, seq_qstart, seq_rows, below, out)
    if (cw == 16) SOC_WKV_LAUNCH(16); else SOC_WKV_LAUNCH(64);
}

SOC_EXPORT int soc_wkv(const void* r, const void* k, const void* v, const float* decay, const float* bonus, int H, int D,
                       float* state, long long stride, int offset, const int* seq_qstart, const int* seq_rows, int below, float* out,
                       int n_seqs, int max_q_len, int dtype, hipStream_t stream) {
    if (n_seqs <= 0 || H <= 0) return 0;
    if (D < 1 || D > 256 || n_seqs > 65535) return (int)hipErrorInvalidValue;
    const int cw = columns_per_workgroup(H, D, n_seqs, max_q_len, below);
#define SOC_WKV_F32(DK) launch_wkv<float, DK>(r, k, v, decay, bonus, H, D, state, stride, offset, seq_qstart, seq_rows, below, out, n_seqs, cw, stream)
#define SOC_WKV_BF16(DK) launch_wkv<bf16, DK>(r, k, v, decay, bonus, H, D, state, stride, offset, seq_qstart, seq_rows, below, out, n_seqs, cw, stream)
    if (dtype == 0) { SOC_BY_STATE_SIZE(D, SOC_WKV_F32) } else { SOC_BY_STATE_SIZE(D, SOC_WKV_BF16) }
    return soc_last_error();
}

// Scalar decay per head: xbc [N, x (H P) | B (G Ns) | C (G Ns)]; dt = softplus(dt_raw + bias);
// S[i, p] <- exp(-exp(a_log) dt) S[i, p] + dt B[i] x[p]; y[p] = sum_i C[i] S[i, p] + skip x[p], float32.
template <typename T, int NK, int CW>
__global__ void __launch_bounds__(256)
ssd_kernel(const T* __restrict__ xbc, const float* __restrict__ dt_raw, const float* __restrict__ dt_bias,
           const float* __restrict__ a_log, const float* __restrict__ skip, int H, int P, int Ns, int G,
           float* __restrict__ state, size_t stride, int offset, const int* __restrict__ seq_qstart,
           const int* __restrict__ seq_rows, int below, float* __restrict__ out) {
    constexpr int REC_TB = rec_batch(NK), PARTS = 256 / CW, KPT = NK / PARTS, STAGE = (REC_TB * NK + 255) / 256;
    __shared__ float sb[2][REC_TB][NK], sc[2][REC_TB][NK], skeep[2][REC_TB], sdt[2][REC_TB];
    __shared__ float red[REC_TB][PARTS][CW];
    const int blocks = (P + CW - 1) / CW;
    const int head = blockIdx.x / blocks, seq = blockIdx.y, tid = threadIdx.x;
    const int lo = seq_qstart[seq], hi = seq_qstart[seq + 1];
    if (lo >= hi || hi - lo >= below) return;
    const int col0 = (blockIdx.x % blocks) * CW;
    const int col = col0 + tid % CW, part = tid / CW, i0 = part * KPT;
    const bool live = col < P;
    const int group = head / (H / G);
    const int inner = H * P, ld = inner + 2 * G * Ns;
    const int boff = inner + group * Ns, coff = inner + G * Ns + group * Ns;
    float* S = state + (size_t)seq_rows[seq] * stride + offset + (size_t)head * Ns * P;
    float s[KPT];
#pragma unroll
    for (int ii = 0; ii < KPT; ++ii) s[ii] = (live && i0 + ii < Ns) ? S[(size_t)(i0 + ii) * P + col] : 0.f;
    const float rate = expf(a_log[head]), through = skip[head], shift = dt_bias[head];
    auto step_size = [&](int n) {
        const float z = dt_raw[(size_t)n * H + head] + shift;
        return z > 20.f ? z : log1pf(expf(z));
    };

    // (a token's step size and decay are computed once, by one thread, and go through LDS with B and C)
    float fb[STAGE], fc[STAGE], fx[REC_TB], fdt = 0.f, fkeep = 1.f;
    auto fetch = [&](int n0) {
#pragma unroll
        for (int t = 0; t < REC_TB; ++t)
            fx[t] = (live && n0 + t < hi) ? to_float(xbc[(size_t)(n0 + t) * ld + head * P + col]) : 0.f;
#pragma unroll
        for (int q = 0; q < STAGE; ++q) {
            const int e = tid + q * 256, t = e / NK, i = e % NK;
            const bool in = t < REC_TB && n0 + t < hi && i < Ns;
            const T* row = xbc + (size_t)(n0 + t) * ld;
            fb[q] = in ? to_float(row[boff + i]) : 0.f;
            fc[q] = in ? to_float(row[coff + i]) : 0.f;
        }
        if (tid < REC_TB) {
            fdt = n0 + tid < hi ? step_size(n0 + tid) : 0.f;
            fkeep = expf(-rate * fdt);
        }
    };
    auto land = [&](int buf) {
#pragma unroll
        for (int q = 0; q < STAGE; ++q) {
            const int e = tid + q * 256, t = e / NK, i = e % NK;
            if (t < REC_TB) { sb[buf][t][i] = fb[q]; sc[buf][t][i] = fc[q]; }
        }
        if (tid < REC_TB) { sdt[buf][tid] = fdt; skeep[buf][tid] = fkeep; }
    };
    fetch(lo);
    land(0);
    lds_barrier();
    int buf = 0;
    for (int n0 = lo; n0 < hi; n0 += REC_TB, buf ^= 1) {
        const int nb = min(REC_TB, hi - n0);
        const bool more = n0 + REC_TB < hi;
        float xj[REC_TB];
#pragma unroll
        for (int t = 0; t < REC_TB; ++t) xj[t] = fx[t];
        if (more) fetch(n0 + REC_TB);
#pragma unroll
        for (int t = 0; t < REC_TB; ++t) {
            if (t < nb) {
                const float keep = skeep[buf][t], dx = sdt[buf][t] * xj[t];
                float acc = part == 0 ? through * xj[t] : 0.f;
#pragma unroll
                for (int ii = 0; ii < KPT; ++ii) {
                    s[ii] = fmaf(keep, s[ii], sb[buf][t][i0 + ii] * dx);
                    acc = fmaf(sc[buf][t][i0 + ii], s[ii], acc);
                }
                red[t][part][tid % CW] = acc;
            }
        }
        lds_barrier();
        for (int f = tid; f < REC_TB * CW; f += 256) {
            const int t = f / CW, cl = f % CW;
            if (t < nb && col0 + cl < P) {
                float y = 0.f;
#pragma unroll
                for (int pp = 0; pp < PARTS; ++pp) y += red[t][pp][cl];
                out[(size_t)(n0 + t) * inner + head * P + col0 + cl] = y;
            }
        }
        if (more) land(buf ^ 1);
        lds_barrier();
    }
    if (live) {
#pragma unroll
        for (int ii = 0; ii < KPT; ++ii)
            if (i0 + ii < Ns) S[(size_t)(i0 + ii) * P + col] = s[ii];
    }
}

template <typename T, int NK>
static void launch_ssd(const void* xbc, const float* dt_raw, const float* dt_bias, const float* a_log, const float* skip,
                       int H, int P, int Ns, int G, float* state, long long stride, int offset, const int* seq_qstart,
                       const int* seq_rows, int below, float* out, int n_seqs, int cw, hipStream_t stream) {
#define SOC_SSD_LAUNCH(CW)                                                                                                   \
    hipLaunchKernelGGL((ssd_kernel<T, NK, CW>), dim3(H * ((P + CW - 1) / CW), n_seqs), dim3(256), 0, stream, (const T*)xbc, \
                       dt_raw, dt_bias, a_log, skip, H, P, Ns, G, state, (size_t)stride, offset, seq_qstart, seq_rows, below, out)
    if (cw == 16) SOC_SSD_LAUNCH(16); else SOC_SSD_LAUNCH(64);
}

SOC_EXPORT int soc_ssd(const void* xbc, const float* dt_raw, const float* dt_bias, const float* a_log, const float* skip,
                       int H, int P, int Ns, int G, float* state, long long stride, int offset, const int* seq_qstart,
                       const int* seq_rows, int below, float* out, int n_seqs, int max_q_len, int dtype, hipStream_t stream) {
    if (n_seqs <= 0 || H <= 0) return 0;
    if (Ns < 1 || Ns > 256 || P < 1 || G < 1 || H % G || n_seqs > 65535) return (int)hipErrorInvalidValue;
    const int cw = columns_per_workgroup(H, P, n_seqs, max_q_len, below);
#define SOC_SSD_F32(NK) launch_ssd<float, NK>(xbc, dt_raw, dt_bias, a_log, skip, H, P, Ns, G, state, stride, offset, seq_qstart, seq_rows, below, out, n_seqs, cw, stream)
#define SOC_SSD_BF16(NK) launch_ssd<bf16, NK>(xbc, dt_raw, dt_bias, a_log, skip, H, P, Ns, G, state, stride, offset, seq_qstart, seq_rows, below, out, n_seqs, cw, stream)
    if (dtype == 0) { SOC_BY_STATE_SIZE(Ns, SOC_SSD_F32) } else { SOC_BY_STATE_SIZE(Ns, SOC_SSD_BF16) }
    return soc_last_error();
}

// ---- causal convolution per channel, then silu -------------------------------------------------------
// y[n, c] = silu(bias[c] + sum_j w[c, j] in(n - (taps - 1) + j)); inputs before the step's first token
// come from the row's state [taps - 1, C], which then becomes the step's last taps - 1 inputs.
// Grid (channel blocks, chunks of CONV_CHUNK tokens, sequences); only a sequence's first chunk
// touches the state (taps - 1 <= CONV_CHUNK), each thread its own channel, reading before writing.
constexpr int CONV_CHUNK = 32;

template <typename T>
__global__ void __launch_bounds__(256)
causal_conv_silu_kernel(const T* __restrict__ x, int ldx, int col, int C, const float* __restrict__ w,
                        const float* __restrict__ bias, int taps, float* __restrict__ state, size_t stride, int offset,
                        const int* __restrict__ seq_qstart, const int* __restrict__ seq_rows, T* __restrict__ out) {
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int seq = blockIdx.z;
    const int lo = seq_qstart[seq], hi = seq_qstart[seq + 1];
    const int first = lo + blockIdx.y * CONV_CHUNK;
    if (c >= C || first >= hi) return;
    const int last = min(first + CONV_CHUNK, hi);
    float* kept = state + (size_t)seq_rows[seq] * stride + offset;
    const int back = taps - 1;
    for (int n = first; n < last; ++n) {
        float y = bias[c];
        for (int j = 0; j < taps; ++j) {
            const int idx = n - lo - back + j;          // among the step's tokens of this sequence
            const float in = idx >= 0 ? to_float(x[(size_t)(lo + idx) * ldx + col + c])
                                      : kept[(size_t)(back + idx) * C + c];
            y = fmaf(w[(size_t)c * taps + j], in, y);
        }
        out[(size_t)n * C + c] = from_float<T>(y * soc_sigmoid(y));
    }
    if (first == lo) {
        const int len = hi - lo;
        for (int j = 0; j < back; ++j) {                // ascending: entry j + len is read before it is written
            const int idx = len - back + j;
            kept[(size_t)j * C + c] = idx >= 0 ? to_float(x[(size_t)(lo + idx) * ldx + col + c])
                                               : kept[(size_t)(j + len) * C + c];
        }
    }
}

// The same for two to four taps and chunks that are mostly full: a thread has its channel's taps and all inputs
// of its chunk on their way before it adds the first (the kernel above waits for every input, TAPS times over:
// 2,048 tokens of 5,376 channels, 4 taps, bf16 took it 103 us, this one 19). Tokens past the sequence's end are loaded as its
// last and not written. Same additions in the same order.
template <typename T, int TAPS>
__global__ void __launch_bounds__(256)
causal_conv_silu_chunk_kernel(const T* __restrict__ x, int ldx, int col, int C, const float* __restrict__ w,
                              const float* __restrict__ bias, float* __restrict__ state, size_t stride, int offset,
                              const int* __restrict__ seq_qstart, const int* __restrict__ seq_rows, T* __restrict__ out) {
    constexpr int BACK = TAPS - 1;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int seq = blockIdx.z;
    const int lo = seq_qstart[seq], hi = seq_qstart[seq + 1];
    const int first = lo + blockIdx.y * CONV_CHUNK;
    if (c >= C || first >= hi) return;
    float* kept = state + (size_t)seq_rows[seq] * stride + offset + c;
    const T* xc = x + col + c;
    T raw[CONV_CHUNK];
#pragma unroll
    for (int i = 0; i < CONV_CHUNK; ++i) raw[i] = xc[(size_t)min(first + i, hi - 1) * ldx];
    float wr[TAPS], in[TAPS];
#pragma unroll
    for (int j = 0; j < TAPS; ++j) wr[j] = w[(size_t)c * TAPS + j];
    const float b = bias[c];
#pragma unroll
    for (int j = 0; j < BACK; ++j)                      // inputs first - BACK + j
        in[j] = first == lo ? kept[(size_t)j * C] : to_float(xc[(size_t)(first - BACK + j) * ldx]);
#pragma unroll
    for (int i = 0; i < CONV_CHUNK; ++i) {
        in[BACK] = to_float(raw[i]);
        float y = b;
#pragma unroll
        for (int j = 0; j < TAPS; ++j) y = fmaf(wr[j], in[j], y);
        if (first + i < hi) out[(size_t)(first + i) * C + c] = from_float<T>(y * soc_sigmoid(y));
#pragma unroll
        for (int j = 0; j < BACK; ++j) in[j] = in[j + 1];
    }
    if (first == lo) {
        const int len = hi - lo;
        for (int j = 0; j < BACK; ++j) {                // ascending: entry j + len is read before it is written
            const int idx = len - BACK + j;
            kept[(size_t)j * C] = idx >= 0 ? to_float(xc[(size_t)(lo + idx) * ldx]) : kept[(size_t)(j + len) * C];
        }
    }
}

SOC_EXPORT int soc_causal_conv_silu(const void* x, int ldx, int col, int C, const float* w, const float* bias, int taps,
                                    float* state, long long stride, int offset, const int* seq_qstart,
                                    const int* seq_rows, void* out, int n_seqs, int max_q_len, int dtype,
                                    hipStream_t stream) {
    if (n_seqs <= 0 || C <= 0) return 0;
    if (taps < 1 || taps - 1 > CONV_CHUNK) return (int)hipErrorInvalidValue;
    const dim3 grid((C + 255) / 256, (max_q_len + CONV_CHUNK - 1) / CONV_CHUNK, n_seqs);
#define SOC_CONV(T, TAPS)                                                                                                     \
    hipLaunchKernelGGL((causal_conv_silu_chunk_kernel<T, TAPS>), grid, dim3(256), 0, stream, (const T*)x, ldx, col, C, w, bias, \
                       state, (size_t)stride, offset, seq_qstart, seq_rows, (T*)out)
#define SOC_CONV_T(T) { if (taps == 2) SOC_CONV(T, 2); else if (taps == 3) SOC_CONV(T, 3); else SOC_CONV(T, 4); }
    // a chunk is loaded whole, so from half a chunk on (a decode step's single token keeps the plain kernel)
    if (taps >= 2 && taps <= 4 && max_q_len >= CONV_CHUNK / 2) {
        if (dtype == 0) SOC_CONV_T(float) else SOC_CONV_T(bf16)
        return soc_last_error();
    }
#undef SOC_CONV_T
#undef SOC_CONV
    if (dtype == 0)
        hipLaunchKernelGGL(causal_conv_silu_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, ldx, col, C, w, bias,
                           taps, state, (size_t)stride, offset, seq_qstart, seq_rows, (float*)out);
    else
        hipLaunchKernelGGL(causal_conv_silu_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)x, ldx, col, C, w, bias,
                           taps, state, (size_t)stride, offset, seq_qstart, seq_rows, (bf16*)out);
    return soc_last_error();
}

// ---- RMS norm in equal parts with a gate silu(z), in front of the norm or behind it ------------------------
// y float32 [N, inner]; z the first `inner` columns of rows of ldz elements. Gate first: norm(y silu(z)) gain;
// gate last: norm(y) gain silu(z). sigmoid_gate: the gate is sigmoid(z) in place of silu(z). An item (part, token) is one wave's (four items to a workgroup), or, for
// parts of 512 elements and more, a whole workgroup's.
template <typename T, bool GATE_FIRST, int WAVES>
__global__ void __launch_bounds__(256)
gated_group_norm_kernel(const float* __restrict__ y, const T* __restrict__ z, int ldz, const float* __restrict__ gain,
                        int inner, int part, int n_items, float eps, int sigmoid_gate, T* __restrict__ out) {
    __shared__ float scratch[16];
    constexpr int THREADS = WAVES * SOC_WAVE;
    const int item = WAVES == 1 ? blockIdx.x * (256 / SOC_WAVE) + threadIdx.x / SOC_WAVE : blockIdx.x;
    const int lane = threadIdx.x % THREADS;
    if (item >= n_items) return;
    const int parts = inner / part;
    const int n = item / parts, c0 = (item % parts) * part;
    float ss = 0.f;
    for (int c = c0 + lane; c < c0 + part; c += THREADS) {
        float v = y[(size_t)n * inner + c];
        if (GATE_FIRST) { const float zz = to_float(z[(size_t)n * ldz + c]); v *= sigmoid_gate ? soc_sigmoid(zz) : zz * soc_sigmoid(zz); }
        ss += v * v;
    }
    ss = WAVES == 1 ? wave_sum(ss) : block_sum(ss, scratch);
    const float inv = 1.f / sqrtf(ss / (float)part + eps);
    for (int c = c0 + lane; c < c0 + part; c += THREADS) {
        const float zz = to_float(z[(size_t)n * ldz + c]);
        const float v = y[(size_t)n * inner + c] * (sigmoid_gate ? soc_sigmoid(zz) : zz * soc_sigmoid(zz));
        out[(size_t)n * inner + c] = from_float<T>(v * inv * gain[c]);
    }
}

SOC_EXPORT int soc_gated_group_norm(const float* y, const void* z, int ldz, const float* gain, int N, int inner, int parts,
                                    float eps, int gate_first, int sigmoid_gate, void* out, int dtype, hipStream_t stream) {
    if (N <= 0) return 0;
    if (parts < 1 || inner % parts || (long long)N * parts > 0x7fffffffLL) return (int)hipErrorInvalidValue;
    const int items = N * parts;
    const bool wide = inner / parts >= 512;
    const dim3 grid(wide ? items : (items + 3) / 4);
#define SOC_GGN(T, FIRST, WAVES)                                                                                              \
    hipLaunchKernelGGL((gated_group_norm_kernel<T, FIRST, WAVES>), grid, dim3(256), 0, stream, y, (const T*)z, ldz, gain, inner, \
                       inner / parts, items, eps, sigmoid_gate, (T*)out)
#define SOC_GGN_T(T)                                                                                   \
    if (gate_first) { if (wide) SOC_GGN(T, true, 4); else SOC_GGN(T, true, 1); }                       \
    else { if (wide) SOC_GGN(T, false, 4); else SOC_GGN(T, false, 1); }
    if (dtype == 0) { SOC_GGN_T(float) } else { SOC_GGN_T(bf16) }
    return soc_last_error();
}

// ---- everything that attention over a cached latent does with its first product's row -----------------------------
// x: rows of ld elements. Workgroups (token, role): the latent, R elements from col_kv on, RMS-normed with kv_gain, and
// the key part behind it (Dr elements) turned pair by pair (pairs 2i, 2i + 1 of the first 2 * half by position * inv_freq[i]),
// into the token's place of the pool [pages, 1, block, width], zeros up to width behind them (pool null: no such role); the query latent, the first q_rank elements, RMS-normed into q_out [N, q_rank] (q_rank 0:
// no such role); or, where the row starts with H heads of D + Dr, their last Dr elements turned into folded
// [N, H, width] behind the first R, zeros behind them (folded null: no such role).
template <typename T, int PER>
__device__ __forceinline__ void wg_rms_row(const T* __restrict__ row, const float* __restrict__ gain, T* __restrict__ dst, int dim, float eps,
                                           float* scratch) {
    float v[PER], ss = 0.f;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        v[i] = c < dim ? to_float(row[c]) : 0.f;
        ss += v[i] * v[i];
    }
    const float inv = 1.f / sqrtf(block_sum(ss, scratch) / (float)dim + eps);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int c = threadIdx.x + i * 256;
        if (c < dim) dst[c] = from_float<T>(v[i] * inv * gain[c]);
    }
}

template <typename T>
__global__ void __launch_bounds__(256)
latent_prepare_kernel(const T* __restrict__ x, int ld, int q_rank, const float* __restrict__ q_gain, T* __restrict__ q_out, int H, int D,
                      T* __restrict__ folded, int R, int Dr, const float* __restrict__ kv_gain, float eps, const float* __restrict__ inv_freq,
                      int half, const int* __restrict__ positions, const int* __restrict__ token_rows, const int* __restrict__ table,
                      int table_width, T* __restrict__ pool, int block, int width, int col_kv, int role0) {
    __shared__ float scratch[16];
    __shared__ float cs[320], sn[320];
    const int n = blockIdx.x, tid = threadIdx.x, role = blockIdx.y == 0 ? role0 : (int)blockIdx.y + role0;
    const T* row = x + (size_t)n * ld;
    if (role == 1) {                                       // the queries: a latent to be normed, or rotated parts
        if (q_rank > 0) {
            if (q_rank <= 512) wg_rms_row<T, 2>(row, q_gain, q_out + (size_t)n * q_rank, q_rank, eps, scratch);
            else if (q_rank <= 2048) wg_rms_row<T, 8>(row, q_gain, q_out + (size_t)n * q_rank, q_rank, eps, scratch);
            else wg_rms_row<T, 32>(row, q_gain, q_out + (size_t)n * q_rank, q_rank, eps, scratch);
            return;
        }
        const float pos = (float)positions[n];
        for (int i = tid; i < half; i += 256) sincosf(pos * inv_freq[i], &sn[i], &cs[i]);
        __syncthreads();
        const int per = width - R;
        for (int i = tid; i < H * per; i += 256) {
            const int h = i / per, e = i % per, pair = e / 2;
            const T* src = row + (size_t)h * (D + Dr) + D;
            T* dst = folded + ((size_t)n * H + h) * width + R;
            if (e >= Dr) dst[e] = from_float<T>(0.f);
            else if (pair >= half) dst[e] = src[e];
            else {
                const float a = to_float(src[2 * pair]), b = to_float(src[2 * pair + 1]);
                dst[e] = from_float<T>((e & 1) ? b * cs[pair] + a * sn[pair] : a * cs[pair] - b * sn[pair]);
            }
        }
        return;
    }
    const int pos = positions[n];
    const int page = table[(size_t)token_rows[n] * table_width + pos / block];
    T* dst = pool + ((size_t)page * block + pos % block) * width;
    row += col_kv;
    wg_rms_row<T, 3>(row, kv_gain, dst, R, eps, scratch);
    for (int e = tid; e < width - R; e += 256) {
        const int pair = e / 2;
        if (e >= Dr) dst[R + e] = from_float<T>(0.f);
        else if (pair >= half) dst[R + e] = row[R + e];
        else {
            float s, c;
            sincosf((float)pos * inv_freq[pair], &s, &c);
            const float a = to_float(row[R + 2 * pair]), b = to_float(row[R + 2 * pair + 1]);
            dst[R + e] = from_float<T>((e & 1) ? b * c + a * s : a * c - b * s);
        }
    }
}

SOC_EXPORT int soc_latent_prepare(const void* x, int ld, int q_rank, const float* q_gain, void* q_out, int H, int D, void* folded, int R, int Dr,
                                  const float* kv_gain, float eps, const float* inv_freq, int half, const int* positions,
                                  const int* token_rows, const int* table, int table_width, void* pool, int block, int width, int col_kv,
                                  int N, int with_q, int dtype, hipStream_t stream) {
    if (N <= 0) return 0;
    const int roles = (pool ? 1 : 0) + (with_q ? 1 : 0);
    if (!roles) return 0;
    if (R < 1 || R > 768 || 2 * half > Dr || half > 320 || R + Dr > width || q_rank > 8192 || (with_q && q_rank > 0 && (!q_gain || !q_out)) ||
        (with_q && q_rank <= 0 && (!folded || (long long)H * (D + Dr) > ld)) || (pool && (col_kv < 0 || col_kv + R + Dr > ld || block < 1)))
        return (int)hipErrorInvalidValue;
    const dim3 grid(N, roles);
#define SOC_LP(T)                                                                                                                     \
    hipLaunchKernelGGL(latent_prepare_kernel<T>, grid, dim3(256), 0, stream, (const T*)x, ld, q_rank, q_gain, (T*)q_out, H, D, (T*)folded, R, \
                       Dr, kv_gain, eps, inv_freq, half, positions, token_rows, table, table_width, (T*)pool, block, width, col_kv, pool ? 0 : 1)
    if (dtype == 0) SOC_LP(float); else SOC_LP(bf16);
#undef SOC_LP
    return soc_last_error();
}

// ---- the rotated part of every head's query, beside the folded plain part ---------------------------------------
// q: rows ldq apart that start with H heads of D + Dr -> out [N, H, width]: out[.., R : R + Dr] = turned q[.., D :], zeros behind it.
// (out[.., : R] is written by the product per head.) One thread per (token, head, pair or padding element).
template <typename T>
__global__ void latent_query_turn_kernel(const T* __restrict__ q, int ldq, int H, int D, int Dr, int R, int width,
                                         const float* __restrict__ inv_freq, int half, const int* __restrict__ positions,
                                         T* __restrict__ out, size_t total) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int per = width - R;                      // elements behind the folded part
    const int e = (int)(i % per);
    const size_t nh = i / per;
    const int n = (int)(nh / H);
    const T* src = q + (size_t)n * ldq + (size_t)(nh % H) * (D + Dr) + D;
    T* dst = out + nh * width + R;
    if (e >= Dr) { dst[e] = from_float<T>(0.f); return; }
    const int pair = e / 2;
    if (pair >= half || (e | 1) >= Dr) { dst[e] = src[e]; return; }
    float sn, cs;
    sincosf((float)positions[n] * inv_freq[pair], &sn, &cs);
    const float a = to_float(src[2 * pair]), b = to_float(src[2 * pair + 1]);
    dst[e] = from_float<T>((e & 1) ? b * cs + a * sn : a * cs - b * sn);
}

SOC_EXPORT int soc_latent_query_turn(const void* q, int ldq, int N, int H, int D, int Dr, int R, int width, const float* inv_freq,
                                     int half, const int* positions, void* out, int dtype, hipStream_t stream) {
    const size_t total = (size_t)N * H * (width - R);
    if (total == 0) return 0;
    if (2 * half > Dr || R + Dr > width || ldq < H * (D + Dr)) return (int)hipErrorInvalidValue;
    const dim3 grid((unsigned)((total + 255) / 256));
    if (dtype == 0)
        hipLaunchKernelGGL(latent_query_turn_kernel<float>, grid, dim3(256), 0, stream, (const float*)q, ldq, H, D, Dr, R, width,
                           inv_freq, half, positions, (float*)out, total);
    else
        hipLaunchKernelGGL(latent_query_turn_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)q, ldq, H, D, Dr, R, width,
                           inv_freq, half, positions, (bf16*)out, total);
    return soc_last_error();
}

// ---- one small product per head ------------------------------------------------------------------------------------
// out[n, h, o] = sum_k x[n, h, k] w[h, o, k], k < K, o < n_out; tokens of x lie ldn elements apart (they may be columns
// of a wider product), heads ldx (its first K are read), out rows of ldo elements per head (its first n_out are written). Tiles of 16 tokens x 64 outputs,
// 32 k at a time through LDS; float32 sums, k in order.
template <typename T>
__global__ void __launch_bounds__(256)
head_linear_kernel(const T* __restrict__ x, int ldn, int ldx, const T* __restrict__ w, T* __restrict__ out, int ldo,
                   int N, int H, int n_out, int K) {
    __shared__ float xs[16][33], ws[64][33];
    const int head = blockIdx.z, n0 = blockIdx.y * 16, o0 = blockIdx.x * 64;
    const int to = threadIdx.x % 64, tn = threadIdx.x / 64;          // output column; token group of 4
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 32) {
        for (int e = threadIdx.x; e < 16 * 32; e += 256) {
            const int rn = e / 32, rk = e % 32;
            xs[rn][rk] = (n0 + rn < N && k0 + rk < K) ? to_float(x[(size_t)(n0 + rn) * ldn + (size_t)head * ldx + k0 + rk]) : 0.f;
        }
        for (int e = threadIdx.x; e < 64 * 32; e += 256) {
            const int ro = e / 32, rk = e % 32;
            ws[ro][rk] = (o0 + ro < n_out && k0 + rk < K) ? to_float(w[((size_t)head * n_out + o0 + ro) * K + k0 + rk]) : 0.f;
        }
        __syncthreads();
#pragma unroll
        for (int kk = 0; kk < 32; ++kk) {
            const float wv = ws[to][kk];
#pragma unroll
            for (int t = 0; t < 4; ++t) acc[t] = fmaf(xs[tn * 4 + t][kk], wv, acc[t]);
        }
        __syncthreads();
    }
    if (o0 + to < n_out)
        for (int t = 0; t < 4; ++t)
            if (n0 + tn * 4 + t < N)
                out[((size_t)(n0 + tn * 4 + t) * H + head) * ldo + o0 + to] = from_float<T>(acc[t]);
}

// The same product for steps of at most 16 tokens, where the tiles above would wait for memory once per 32 k:
// a wave per (head, output), its lanes over k, all loads issued at once, one sum over the wave per token.
template <typename T>
__global__ void __launch_bounds__(256)
head_linear_rows_kernel(const T* __restrict__ x, int ldn, int ldx, const T* __restrict__ w, T* __restrict__ out, int ldo,
                        int N, int H, int n_out, int K) {
    const int head = blockIdx.y, o = blockIdx.x * 4 + threadIdx.x / SOC_WAVE, lane = threadIdx.x % SOC_WAVE;
    if (o >= n_out) return;
    float acc[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) acc[n] = 0.f;
    const T* wrow = w + ((size_t)head * n_out + o) * K;
    for (int k = lane; k < K; k += SOC_WAVE) {
        const float wv = to_float(wrow[k]);
#pragma unroll
        for (int n = 0; n < 16; ++n)
            if (n < N) acc[n] = fmaf(to_float(x[(size_t)n * ldn + (size_t)head * ldx + k]), wv, acc[n]);
    }
#pragma unroll
    for (int n = 0; n < 16; ++n) {
        if (n < N) {
            const float sum = wave_sum(acc[n]);
            if (lane == 0) out[((size_t)n * H + head) * ldo + o] = from_float<T>(sum);
        }
    }
}

SOC_EXPORT int soc_head_linear(const void* x, int ldn, int ldx, const void* w, void* out, int ldo, int N, int H, int n_out, int K,
                               int dtype, hipStream_t stream) {
    if (N <= 0 || H <= 0 || n_out <= 0) return 0;
    if (K < 1 || K > ldx || (long long)ldn < (long long)(H - 1) * ldx + K || n_out > ldo || H > 65535 || (N + 15) / 16 > 65535) return (int)hipErrorInvalidValue;
    if (N <= 16) {
        const dim3 rows_grid((n_out + 3) / 4, H);
        if (dtype == 0)
            hipLaunchKernelGGL(head_linear_rows_kernel<float>, rows_grid, dim3(256), 0, stream, (const float*)x, ldn, ldx,
                               (const float*)w, (float*)out, ldo, N, H, n_out, K);
        else
            hipLaunchKernelGGL(head_linear_rows_kernel<bf16>, rows_grid, dim3(256), 0, stream, (const bf16*)x, ldn, ldx,
                               (const bf16*)w, (bf16*)out, ldo, N, H, n_out, K);
        return soc_last_error();
    }
    const dim3 grid((n_out + 63) / 64, (N + 15) / 16, H);
    if (dtype == 0)
        hipLaunchKernelGGL(head_linear_kernel<float>, grid, dim3(256), 0, stream, (const float*)x, ldn, ldx, (const float*)w,
                           (float*)out, ldo, N, H, n_out, K);
    else
        hipLaunchKernelGGL(head_linear_kernel<bf16>, grid, dim3(256), 0, stream, (const bf16*)x, ldn, ldx, (const bf16*)w,
                           (bf16*)out, ldo, N, H, n_out, K);
    return soc_last_error();
}

// The same product in bfloat16 on the matrix cores (K, ldn, ldx and ldo multiples of 8; x and out on 16 bytes). Weights are
// operand A, tokens operand B, so a lane ends with four consecutive outputs of one token.
//
// Few tokens: a workgroup takes one head, 16 tokens (grid z) and 64 outputs, a wave 16 of them over the whole of K; or
// (SPLIT, long K) 16 outputs, each wave a quarter of K, the four sums meeting in LDS. Operands come straight from
// memory in the products' layout.
template <bool SPLIT>
__global__ void __launch_bounds__(256)
head_mfma_rows_kernel(const bf16* __restrict__ x, int ldn, int ldx, const bf16* __restrict__ w, bf16* __restrict__ out, int ldo, int N, int H,
                      int n_out, int K) {
    __shared__ f32x4_t part[SPLIT ? 4 : 1][64];
    const int wave = threadIdx.x / SOC_WAVE, lane = threadIdx.x % SOC_WAVE, li = lane % 16, kb = lane / 16;
    const int head = blockIdx.y, n = blockIdx.z * 16 + li;
    const int o0 = SPLIT ? blockIdx.x * 16 : (blockIdx.x * 4 + wave) * 16;
    if (!SPLIT && o0 >= n_out) return;
    const int per = SPLIT ? (K + 127) / 128 * 32 : K, k_lo = SPLIT ? wave * per : 0, k_hi = min(K, k_lo + per);
    const bf16* wrow = w + ((size_t)head * n_out + min(o0 + li, n_out - 1)) * K;
    const bf16* xrow = x + (size_t)min(n, N - 1) * ldn + (size_t)head * ldx;
    f32x4_t acc = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int k0 = k_lo; k0 < k_hi; k0 += 32) {
        const int k = k0 + kb * 8;
        uint4 a = make_uint4(0u, 0u, 0u, 0u), b = a;
        if (k < k_hi) {
            a = *reinterpret_cast<const uint4*>(wrow + k);
            b = *reinterpret_cast<const uint4*>(xrow + k);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8_t*>(&a), *reinterpret_cast<const bf16x8_t*>(&b), acc, 0, 0, 0);
    }
    if constexpr (SPLIT) {
        part[wave][lane] = acc;
        __syncthreads();
        if (wave > 0) return;
        acc = part[0][lane] + part[1][lane] + part[2][lane] + part[3][lane];
    }
    if (n >= N) return;
    bf16* dst = out + ((size_t)n * H + head) * ldo + o0 + 4 * kb;
    if (o0 + 4 * kb + 3 < n_out) {
        *reinterpret_cast<uint2*>(dst) = make_uint2(pack_bf16x2(acc[0], acc[1]), pack_bf16x2(acc[2], acc[3]));
    } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (o0 + 4 * kb + r < n_out) dst[r] = from_float<bf16>(acc[r]);
    }
}

// Many tokens: tiles of 128 tokens x 128 outputs of one head, 64 k at a time through two LDS buffers, four waves of
// 64 x 64.
__global__ void __launch_bounds__(256)
head_mfma_tiles_kernel(const bf16* __restrict__ x, int ldn, int ldx, const bf16* __restrict__ w, bf16* __restrict__ out, int ldo, int N, int H,
                       int n_out, int K) {
    constexpr int BK = 64, STRIDE = BK + 8, PER = 128 * 8 / 256;
    __shared__ __attribute__((aligned(16))) uint16_t Xs[2][128 * STRIDE], Ws[2][128 * STRIDE];
    const int tid = threadIdx.x, wave = tid / SOC_WAVE, lane = tid % SOC_WAVE, li = lane % 16, kb = lane / 16;
    const int wn = wave / 2, wo = wave % 2;
    const int head = blockIdx.z, n0 = blockIdx.y * 128, o0 = blockIdx.x * 128;
    const bf16* xs_src[PER];
    const bf16* ws_src[PER];
    const int kc = (tid % 8) * 8;
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int r = tid / 8 + 32 * i;
        xs_src[i] = x + (size_t)min(n0 + r, N - 1) * ldn + (size_t)head * ldx + kc;
        ws_src[i] = w + ((size_t)head * n_out + min(o0 + r, n_out - 1)) * K + kc;
    }
    uint4 xr[PER], wr[PER];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const bool in = k0 + kc < K;
            xr[i] = in ? *reinterpret_cast<const uint4*>(xs_src[i] + k0) : make_uint4(0u, 0u, 0u, 0u);
            wr[i] = in ? *reinterpret_cast<const uint4*>(ws_src[i] + k0) : make_uint4(0u, 0u, 0u, 0u);
        }
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            *reinterpret_cast<uint4*>(&Xs[buf][(tid / 8 + 32 * i) * STRIDE + kc]) = xr[i];
            *reinterpret_cast<uint4*>(&Ws[buf][(tid / 8 + 32 * i) * STRIDE + kc]) = wr[i];
        }
    };
    f32x4_t acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
    fetch(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += BK, buf ^= 1) {
        const bool more = k0 + BK < K;
        if (more) fetch(k0 + BK);
#pragma unroll
        for (int ks = 0; ks < BK; ks += 32) {
            bf16x8_t b[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) b[j] = *reinterpret_cast<const bf16x8_t*>(&Xs[buf][(wn * 64 + j * 16 + li) * STRIDE + ks + kb * 8]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bf16x8_t a = *reinterpret_cast<const bf16x8_t*>(&Ws[buf][(wo * 64 + i * 16 + li) * STRIDE + ks + kb * 8]);
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[j], acc[i][j], 0, 0, 0);
            }
        }
        if (more) stash(buf ^ 1);
        __syncthreads();
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int n = n0 + wn * 64 + j * 16 + li;
        if (n >= N) continue;
        bf16* row = out + ((size_t)n * H + head) * ldo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int o = o0 + wo * 64 + i * 16 + 4 * kb;
            if (o + 3 < n_out) {
                *reinterpret_cast<uint2*>(row + o) = make_uint2(pack_bf16x2(acc[i][j][0], acc[i][j][1]), pack_bf16x2(acc[i][j][2], acc[i][j][3]));
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (o + r < n_out) row[o + r] = from_float<bf16>(acc[i][j][r]);
            }
        }
    }
}

SOC_EXPORT int soc_head_linear_mfma(const void* x, int ldn, int ldx, const void* w, void* out, int ldo, int N, int H, int n_out, int K,
                                    hipStream_t stream) {
    if (N <= 0 || H <= 0 || n_out <= 0) return 0;
    if (K < 8 || K % 8 || ldn % 8 || ldx % 8 || ldo % 4 || K > ldx || n_out > ldo || H > 65535 || (N + 15) / 16 > 65535 ||
        (long long)ldn < (long long)(H - 1) * ldx + K)
        return (int)hipErrorInvalidValue;
    if (N > 64) {
        hipLaunchKernelGGL(head_mfma_tiles_kernel, dim3((n_out + 127) / 128, (N + 127) / 128, H), dim3(256), 0, stream, (const bf16*)x, ldn, ldx,
                           (const bf16*)w, (bf16*)out, ldo, N, H, n_out, K);
    } else if (K >= 256) {
        hipLaunchKernelGGL(head_mfma_rows_kernel<true>, dim3((n_out + 15) / 16, H, (N + 15) / 16), dim3(256), 0, stream, (const bf16*)x, ldn, ldx,
                           (const bf16*)w, (bf16*)out, ldo, N, H, n_out, K);
    } else {
        hipLaunchKernelGGL(head_mfma_rows_kernel<false>, dim3((n_out + 63) / 64, H, (N + 15) / 16), dim3(256), 0, stream, (const bf16*)x, ldn, ldx,
                           (const bf16*)w, (bf16*)out, ldo, N, H, n_out, K);
    }
    return soc_last_error();
}
