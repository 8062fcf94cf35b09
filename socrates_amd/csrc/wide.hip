// Products of many rows: out[M, N] = x[M, K] w[N, K]^T in bfloat16 with float32 sums (the loop is in wide.h), with a gated
// activation in the epilogue where the weights are a feed-forward's gate and up rows: the rounded
// products that another kernel would read back never go to memory.

#include "wide.h"

// x [M, K], w [N, K], K a multiple of 64; out [M, N] (N a multiple of 8), or with an activation over pairs [M, N / 2] (N a
// multiple of 32) of gate and up rows that alternate by 16 (ff 0) or lie one half behind the other (ff = N / 2). With parts,
// out holds float32 [parts, M, N]: the sums over each part of K, added up by whoever reads them.
// Workgroups go round-robin over the eight XCDs: each gets a run of tiles, in blocks of eight tiles of rows, so that the 32 that
// an XCD works on at a time share rows and weights in its L2. An XCD's last tiles, where they leave half of its compute units
// without work, are halved (TAIL): 608 tiles of 256 x 256 are 2.4 rounds, which otherwise cost 3.
template <int MI, int NJ, int ACT, typename TO>
__device__ __forceinline__ void wide_linear_tile(uint16_t* lds, const bf16* x, const bf16* w, TO* out, int M, int N, int K, int m0, int n0,
                                                 int k0, int steps, int ff, WideGate gate) {
    constexpr bool PAIRS = wide_pairs(ACT);
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    uint32_t xo[MI], wo[NJ];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int row = (wave * MI + i) * 8 + lane / 8;
        xo[i] = (uint32_t)min(m0 + row, M - 1) * (uint32_t)K * 2 + ((lane % 8) ^ wide_swap(row)) * 16;
    }
#pragma unroll
    for (int i = 0; i < NJ; ++i) {
        const int row = (wave * NJ + i) * 8 + lane / 8;
        int at = min(n0 + row, N - 1);
        if (PAIRS && ff) at = at / 32 * 16 + at % 16 + (at / 16 % 2 ? ff : 0);
        wo[i] = (uint32_t)at * (uint32_t)K * 2 + ((lane % 8) ^ wide_swap(row)) * 16;
    }
    f32x4_t acc[MI][NJ];
    wide_walk<MI, NJ>(reinterpret_cast<const char*>(x + k0), reinterpret_cast<const char*>(w + k0), xo, wo, steps, lds, acc);
    wide_results<MI, NJ, ACT, TO>(acc, out, m0, M, PAIRS ? n0 / 2 : n0, PAIRS ? N / 2 : N, gate, false);
}

template <int MI, int NJ, bool TAIL, int ACT, typename TO>
__global__ void __launch_bounds__(256, 1)
wide_linear_kernel(const bf16* __restrict__ x, const bf16* __restrict__ w, TO* __restrict__ out, int M, int N, int K, int m_tiles,
                   int n_tiles, int parts, int ff, WideGate gate) {
    using Rings = WideRings<MI, NJ>;
    constexpr int LDS = Rings::RX * MI + Rings::RW * NJ, HALF = TAIL ? WideRings<MI, NJ / 2>::RX * MI + WideRings<MI, NJ / 2>::RW * (NJ / 2) : 0;
    __shared__ __attribute__((aligned(1024))) uint16_t lds[(LDS > HALF ? LDS : HALF) * 2048];
    const int total = m_tiles * n_tiles * parts, chunk = (total + 7) / 8;
    const int full = TAIL ? chunk / 32 * 32 : chunk;          // whole tiles of an XCD
    int at = (int)(blockIdx.x / 8), right = -1;
    if (TAIL && at >= full) {
        right = (at - full) % 2;
        at = full + (at - full) / 2;
    }
    int item = (int)(blockIdx.x % 8) * chunk + at;
    if (at >= chunk || item >= total) return;
    const int part = item / (m_tiles * n_tiles);
    item %= m_tiles * n_tiles;
    const int block = item / (8 * n_tiles), in_block = item % (8 * n_tiles), high = min(8, m_tiles - 8 * block);
    const int m0 = (8 * block + in_block % high) * 32 * MI, n0 = in_block / high * 32 * NJ;
    const int steps = K / 64, s0 = (int)((long long)steps * part / parts), s1 = (int)((long long)steps * (part + 1) / parts);
    out += (size_t)part * M * N;
    if (TAIL && right >= 0) {
        if constexpr (TAIL) {
            if (n0 + right * 16 * NJ < N)
                wide_linear_tile<MI, NJ / 2, ACT, TO>(lds, x, w, out, M, N, K, m0, n0 + right * 16 * NJ, s0 * 64, s1 - s0, ff, gate);
        }
    } else {
        wide_linear_tile<MI, NJ, ACT, TO>(lds, x, w, out, M, N, K, m0, n0, s0 * 64, s1 - s0, ff, gate);
    }
}

template <int MI, int NJ, bool TAIL, int ACT, typename TO>
static void wide_launch(const void* x, const void* w, void* out, int M, int N, int K, int parts, int ff, WideGate gate, hipStream_t s) {
    const int mt = (M + 32 * MI - 1) / (32 * MI), nt = (N + 32 * NJ - 1) / (32 * NJ);
    const int chunk = (mt * nt * parts + 7) / 8, full = TAIL ? chunk / 32 * 32 : chunk;
    hipLaunchKernelGGL((wide_linear_kernel<MI, NJ, TAIL, ACT, TO>), dim3(8 * (full + 2 * (chunk - full))), dim3(256), 0, s, (const bf16*)x,
                       (const bf16*)w, (TO*)out, M, N, K, mt, nt, parts, ff, gate);
}

// The forms: blocks of 32 rows of x and of weight rows, us per step of 64 k and beside the steps per tile, and whether an XCD's last
// tiles may be halved. The figures were measured with every compute unit at work and weights from memory; between them the plan
// is within 10 % of the best form of a sweep over 64 to 2,048 rows at the widths of 4B- and 8B-sized layers.
struct WideForm { int mi, nj, tail; float step, beside; };
static const WideForm WIDE_FORMS[] = {
    {8, 8, 0, 1.34f, 7.f},   {8, 8, 1, 1.34f, 7.f},  {6, 8, 0, 1.02f, 6.5f}, {6, 8, 1, 1.02f, 6.5f}, {5, 8, 0, .94f, 6.f},   {4, 8, 0, .81f, 6.f},
    {4, 8, 1, .81f, 6.f},    {3, 8, 0, .72f, 5.5f},  {2, 8, 0, .60f, 5.f},   {8, 4, 0, .76f, 6.f},   {8, 6, 0, 1.f, 6.5f},   {6, 6, 0, .77f, 6.5f},
    {8, 5, 0, .91f, 6.f},    {4, 6, 0, .67f, 6.f},   {5, 5, 0, .66f, 5.5f},  {4, 5, 0, .55f, 5.f},   {4, 4, 0, .48f, 4.5f},  {3, 5, 0, .47f, 4.5f}};
// of the halves of 8 x 8, 6 x 8 and 4 x 8
static float wide_half_step(int mi) { return mi == 8 ? .76f : mi == 6 ? .62f : .48f; }

// Form and parts of K for a product, by the rounds of workgroups of the XCD that has most and what a part's float32 sums cost
// beside one rounded result (5 TB/s, written and read; a kernel that adds them up where the consumer does not, partial_ok 0).
// 0: not a product for this kernel.
SOC_EXPORT int soc_wide_plan(int M, int N, int K, int act, int partial_ok, int* mi, int* nj, int* tail, int* parts) {
    const bool pairs = wide_pairs(act);
    if (M < 1 || N < (pairs ? 32 : 8) || N % (pairs ? 32 : 8) || K < 64 || K % 64) return 0;
    if ((unsigned long long)M * K >= 1ull << 31 || (unsigned long long)N * K >= 1ull << 31 || (unsigned long long)M * N >= 1ull << 31) return 0;
    double best = 0.0;
    *mi = 0;
    for (const WideForm& f : WIDE_FORMS) {
        if (pairs && f.nj % 4) continue;
        const double mt = (M + 32 * f.mi - 1) / (32 * f.mi), nt = (N + 32 * f.nj - 1) / (32 * f.nj);
        for (int p = 1; p <= (act == WIDE_PLAIN ? 12 : 1) && p * 4 <= K / 64 + 3; ++p) {
            const long long chunk = ((long long)(mt * nt) * p + 7) / 8, rest = chunk % 32;
            const double steps = (K / 64 + p - 1) / p, tile = f.beside + (act ? .035 * f.mi * f.nj : 0.) + steps * f.step;
            double us = 3. + tile * (double)(chunk / 32);
            if (rest && f.tail) us += (rest <= 16 ? 1. : 2.) * (f.beside - 1. + (act ? .018 * f.mi * f.nj : 0.) + steps * wide_half_step(f.mi));
            else if (rest) us += tile;
            if (p > 1) us += (4. * p - 2.) * M * (double)N / 5e6 * 1.5 + (partial_ok ? 0. : 3.);
            if (!*mi || us < best) {
                best = us;
                *mi = f.mi;
                *nj = f.nj;
                *tail = f.tail;
                *parts = p;
            }
        }
    }
    return *mi != 0;
}

// out[i] = the sum of parts[s][i] over s, in order; n a multiple of four.
template <typename TO>
__global__ void __launch_bounds__(256)
wide_sum_kernel(const float* __restrict__ parts, TO* __restrict__ out, size_t n, int S) {
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    float4 t = *reinterpret_cast<const float4*>(parts + i);
    for (int s = 1; s < S; ++s) {
        const float4 v = *reinterpret_cast<const float4*>(parts + (size_t)s * n + i);
        t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
    }
    if constexpr (sizeof(TO) == 4) *reinterpret_cast<float4*>(out + i) = t;
    else *reinterpret_cast<uint2*>(out + i) = make_uint2(pack_bf16x2(t.x, t.y), pack_bf16x2(t.z, t.w));
}

// mi, nj, tail: a form above. act: WIDE_*; out_f32: float32 results (WIDE_PLAIN only). parts > 1: sums holds float32
// [parts, M, N], and out, if given, their sum.
SOC_EXPORT int soc_wide_linear(const void* x, const void* w, void* out, float* sums, int M, int N, int K, int mi, int nj, int tail,
                               int parts, int act, int ff, float limit, float slope, float shift, int out_f32, hipStream_t s) {
    if (M <= 0 || N <= 0) return 0;
    const bool pairs = wide_pairs(act);
    if (K < 64 || K % 64 || N % (pairs ? 32 : 8) || (uintptr_t)x % 16 || (uintptr_t)w % 16 || (uintptr_t)out % 16 || (uintptr_t)sums % 16) return (int)hipErrorInvalidValue;
    if ((unsigned long long)M * K >= 1ull << 31 || (unsigned long long)N * K >= 1ull << 31) return (int)hipErrorInvalidValue;   // 32-bit offsets in bytes
    if (parts < 1 || parts > 64 || parts > K / 64 || (long long)((M + 63) / 64) * ((N + 63) / 64) * parts >= 1 << 26) return (int)hipErrorInvalidValue;
    if (act < WIDE_PLAIN || act > WIDE_SQUARED || (act && (out_f32 || parts > 1)) || (parts > 1 ? !sums : !out) || (ff && (!pairs || 2 * ff != N)))
        return (int)hipErrorInvalidValue;
    const WideGate gate{limit, slope, shift};
#define SOC_WIDE(MI, NJ, TAIL)                                                                                                   \
    if (mi == MI && nj == NJ && (tail != 0) == TAIL) {                                                                           \
        if (parts > 1) wide_launch<MI, NJ, TAIL, WIDE_PLAIN, float>(x, w, sums, M, N, K, parts, 0, gate, s);                      \
        else if (out_f32) wide_launch<MI, NJ, TAIL, WIDE_PLAIN, float>(x, w, out, M, N, K, 1, 0, gate, s);                        \
        else if (act == WIDE_PLAIN) wide_launch<MI, NJ, TAIL, WIDE_PLAIN, bf16>(x, w, out, M, N, K, 1, 0, gate, s);               \
        else if (act == WIDE_SQUARED) wide_launch<MI, NJ, TAIL, WIDE_SQUARED, bf16>(x, w, out, M, N, K, 1, 0, gate, s);           \
        else if constexpr (NJ % 4 == 0) {                                                                                        \
            if (act == WIDE_SILU) wide_launch<MI, NJ, TAIL, WIDE_SILU, bf16>(x, w, out, M, N, K, 1, ff, gate, s);                 \
            else if (act == WIDE_GATED) wide_launch<MI, NJ, TAIL, WIDE_GATED, bf16>(x, w, out, M, N, K, 1, ff, gate, s);          \
            else wide_launch<MI, NJ, TAIL, WIDE_GELU, bf16>(x, w, out, M, N, K, 1, ff, gate, s);                                  \
        } else return (int)hipErrorInvalidValue;                                                                                 \
    } else
    SOC_WIDE(8, 8, false)
    SOC_WIDE(8, 8, true)
    SOC_WIDE(6, 8, false)
    SOC_WIDE(6, 8, true)
    SOC_WIDE(5, 8, false)
    SOC_WIDE(4, 8, false)
    SOC_WIDE(4, 8, true)
    SOC_WIDE(8, 4, false)
    SOC_WIDE(2, 8, false)
    SOC_WIDE(3, 8, false)
    SOC_WIDE(8, 6, false)
    SOC_WIDE(6, 6, false)
    SOC_WIDE(8, 5, false)
    SOC_WIDE(4, 6, false)
    SOC_WIDE(5, 5, false)
    SOC_WIDE(4, 5, false)
    SOC_WIDE(4, 4, false)
    SOC_WIDE(3, 5, false)
        return (int)hipErrorInvalidValue;
#undef SOC_WIDE
    const int err = soc_last_error();
    if (err || parts == 1 || !out) return err;
    const size_t n = (size_t)M * N;
    const dim3 grid((unsigned)((n / 4 + 255) / 256));
    if (out_f32) hipLaunchKernelGGL(wide_sum_kernel<float>, grid, dim3(256), 0, s, sums, (float*)out, n, parts);
    else hipLaunchKernelGGL(wide_sum_kernel<bf16>, grid, dim3(256), 0, s, sums, (bf16*)out, n, parts);
    return soc_last_error();
}
