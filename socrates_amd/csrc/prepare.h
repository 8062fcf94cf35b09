// What a prompt's attention layers do with a token's projected heads before the attention itself, for heads of 64 or 128 elements
// in bfloat16: bias, norm, rotation, the values' blend or turn, and the writes to queries and pages. One workgroup per token:
// its angles are taken once, in LDS, and 16 (8) lanes own a head, eight neighbouring elements each, so that a load or store is 16
// bytes a lane and a norm crosses lanes in registers. Bound by memory and, per token, the trip to its position and page.
// The general kernels (attn_prepare, window_prepare) take an angle per element, or walk heads in pieces of two elements. Us, 32 +
// 2 x 8 heads of 128: 2,339 tokens with norms, 64 elements turned and blended values 48 to 54, now 19; 2,048 tokens with biases,
// norms and turned values 45, now 17; 3,000 tokens as they are 31 to 41, now 17 (their 74 MB take 15 at a copy's rate).
#pragma once

#include "common.h"

struct PrepareArgs {
    const bf16* x;                                           // rows of ld elements
    int ld, col_q, col_k, col_v;
    const float* bias;                                       // [ld] or null
    const bf16* first;                                       // rows of ldf elements that values are blended with by lam[0], or null
    int ldf;
    const float* lam;
    bf16 *q_out, *k_pool, *v_pool;                           // [N, Hq, D]; [pages, Hkv, BS, D]
    const int* table;
    int table_width;
    const int *token_rows, *positions;
    const float *q_gain, *k_gain;                            // per head [D], or over all heads (WHOLE) [Hq D] and [Hkv D]; or null
    int norm;                                                // 0: none, 1: per head, 2: over the whole of q and of k
    float eps;
    const float* inv_freq;                                   // [half]: angles of the first 2 half elements of q and k
    int half;
    float magnitude;                                         // of their cosines and sines
    const float* value_freq;                                 // [D / 2]: angles of the values' pairs, or null
    int Hq, Hkv, BS;
};

// lanes 8 or 16 apart from each other's group: the sum over a group, in all its lanes
template <int LANES> __device__ __forceinline__ float prepare_sum(float v) {
    v += soc_dpp<SOC_DPP_XOR1>(v);
    v += soc_dpp<SOC_DPP_XOR2>(v);
    v += soc_dpp<SOC_DPP_HALF_MIRROR>(v);
    if (LANES == 16) v += soc_dpp<SOC_DPP_ROW_MIRROR>(v);
    return v;
}

// PAIRS: elements 2 i and 2 i + 1 turn together, else i and i + half (half a multiple of 8).
template <int D, bool PAIRS>
__global__ void __launch_bounds__(256)
heads_prepare_kernel(PrepareArgs a) {
    constexpr int LANES = D / 8, HEADS = 256 / LANES;        // lanes of a head, heads of a pass
    __shared__ float cs[D / 2], sn[D / 2], vcs[D / 2], vsn[D / 2], scratch[16];
    const int n = blockIdx.x, tid = threadIdx.x, part = tid % LANES, at = part * 8;
    const int pos = a.positions[n];
    const bf16* row = a.x + (size_t)n * a.ld;
    const size_t page = a.Hkv ? (size_t)a.table[(size_t)a.token_rows[n] * a.table_width + pos / a.BS] : 0;
    if (tid < a.half) {
        float s, c;
        sincosf((float)pos * a.inv_freq[tid], &s, &c);
        cs[tid] = c * a.magnitude;
        sn[tid] = s * a.magnitude;
    }
    if (a.value_freq && tid >= 128 && tid < 128 + D / 2) {
        float s, c;
        sincosf((float)pos * a.value_freq[tid - 128], &s, &c);
        vcs[tid - 128] = c;
        vsn[tid - 128] = s;
    }
    auto load = [&](int col, float (&v)[8]) {
        VecLoad<bf16, 8>::load(row + col, v);
        if (a.bias) {
            float b[8];
            VecLoad<float, 8>::load(a.bias + col, b);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] += b[e];
        }
    };
    float iq = 1.f, ik = 1.f;
    if (a.norm == 2) {
        float sq = 0.f, sk = 0.f;
        for (int h = tid / LANES; h < a.Hq + a.Hkv; h += HEADS) {
            float v[8], ss = 0.f;
            load((h < a.Hq ? a.col_q + h * D : a.col_k + (h - a.Hq) * D) + at, v);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
            if (h < a.Hq) sq += ss;
            else sk += ss;
        }
        sq = block_sum(sq, scratch);
        sk = block_sum(sk, scratch);
        iq = 1.f / sqrtf(sq / (float)(a.Hq * D) + a.eps);
        ik = 1.f / sqrtf(sk / (float)(a.Hkv * D) + a.eps);
    }
    __syncthreads();                                         // the angles
    const float lam = a.first ? a.lam[0] : 0.f;
    // (every lane of a group of heads takes part in the crossings, those past the last head with the last one's elements)
    const int heads = a.Hq + 2 * a.Hkv;
    for (int h0 = 0; h0 < heads; h0 += HEADS) {
        const bool own = h0 + tid / LANES < heads;
        const int h = own ? h0 + tid / LANES : heads - 1;
        const bool is_q = h < a.Hq, is_v = h >= a.Hq + a.Hkv;
        const int kvh = is_q ? 0 : is_v ? h - a.Hq - a.Hkv : h - a.Hq;
        float v[8];
        load((is_q ? a.col_q + h * D : (is_v ? a.col_v : a.col_k) + kvh * D) + at, v);
        if (a.norm == 1) {
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(v[e], v[e], ss);
            ss = prepare_sum<LANES>(ss);
            const float* gain = is_q ? a.q_gain : a.k_gain;
            if (!is_v && gain) {
                const float inv = 1.f / sqrtf(ss / (float)D + a.eps);
                float g[8];
                VecLoad<float, 8>::load(gain + at, g);
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = v[e] * inv * g[e];
            }
        } else if (a.norm == 2 && !is_v) {
            float g[8];
            VecLoad<float, 8>::load((is_q ? a.q_gain + h * D : a.k_gain + kvh * D) + at, g);
            const float inv = is_q ? iq : ik;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = v[e] * inv * g[e];
        }
        if constexpr (PAIRS) {
            const float *c = is_v ? vcs : cs, *s = is_v ? vsn : sn;
            const int turned = is_v ? (a.value_freq ? D / 2 : 0) : a.half;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const int i = (at + e) / 2;
                if (i < turned) {
                    const float p = v[e], q = v[e + 1];
                    v[e] = p * c[i] - q * s[i];
                    v[e + 1] = q * c[i] + p * s[i];
                }
            }
        } else {
            const int step = a.half / 8;
            const bool low = at < a.half, turned = !is_v && at < 2 * a.half;
            const int other = (tid % 64) + (turned ? (low ? step : -step) : 0), i = low ? at : at - a.half;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float p = __shfl(v[e], other, 64);
                if (turned) v[e] = low ? v[e] * cs[i + e] - p * sn[i + e] : v[e] * cs[i + e] + p * sn[i + e];
            }
        }
        if (is_v && a.first) {
            float f[8];
            VecLoad<bf16, 8>::load(a.first + (size_t)n * a.ldf + kvh * D + at, f);
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = (1.f - lam) * v[e] + lam * f[e];
        }
        bf16* to = (is_q ? a.q_out + ((size_t)n * a.Hq + h) * D
                         : (is_v ? a.v_pool : a.k_pool) + ((page * a.Hkv + kvh) * a.BS + pos % a.BS) * D) + at;
        if (own)
            *reinterpret_cast<uint4*>(to) = make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7]));
    }
}

// Whether the kernel above takes these heads: their size, rows and columns on 16 bytes, and tokens enough for a workgroup each
// (fewer tokens than compute units are better served by the general kernels' several workgroups a token).
static inline bool heads_prepare_fits(const PrepareArgs& a, int N, int D, int Dv, int P, bool pairs) {
    const uintptr_t sixteen = (uintptr_t)a.x | (uintptr_t)a.bias | (uintptr_t)a.first | (uintptr_t)a.q_out | (uintptr_t)a.k_pool | (uintptr_t)a.v_pool
                              | (uintptr_t)a.q_gain | (uintptr_t)a.k_gain;
    return N >= 256 && (D == 64 || D == 128) && Dv == D && P == D && a.ld % 8 == 0 && a.ldf % 8 == 0 && a.col_q % 8 == 0 && a.col_k % 8 == 0
           && a.col_v % 8 == 0 && a.norm <= 2 && (pairs || a.half % 8 == 0) && sixteen % 16 == 0;
}
