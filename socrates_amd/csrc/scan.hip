// Linear recurrences with a matrix state per head, S <- decay S + k v^T, over long portions: 64 tokens at a time on
// the matrix cores instead of token by token on the vector units.
//
// Inside a chunk the outputs are (scores of the chunk against itself under the decays) V + (queries decayed back to
// the chunk's start) S, and the state moves once: S <- (the chunk's decay) S + (keys decayed to its end)^T V. Three
// kernels: scan_chunks (every chunk and head by itself: scores, their share of the outputs, the chunk's addend to the
// state), scan_states (the states before every chunk, element by element), scan_apply (the states' share of the
// outputs). All products are v_mfma_f32_16x16x4_f32: float32 in, float32 sums, as the walk has.
//
// Decays only ever multiply: a product over tokens j+1 .. i is formed from its factors, by runs of 16 tokens (start of
// the run to i) * (whole runs between) * (j to its run's end); inside a run pair by pair. Nothing is divided and no
// logarithm taken, so a decay of 0, or a product that underflows, gives what the walk gives. The decay is one number
// per head, one per token and head, or one per token, head and key channel.
//
// Bound by memory: per chunk and head the addend (D x Dv float32) is written, read, written as a state and read
// again, the outputs written, read and written. 64 tokens: with 32 the addends weigh twice as much, with 128 a
// chunk's queries, keys and decays of 128 channels do not fit LDS.
//
// Measured for 2,048 tokens of one prompt, us, the walk -> these kernels with what prepares them: retention (20 heads of
// 128 x 128) 908 -> 110 (chunks 48, states 17, apply 30), gated linear attention (10 of 128 x 256) 1,032 -> 136 (75, 17, 30),
// wkv (40 of 64 x 64) 595 -> 100 with its norm (55, 10, 18), ssd (80 of 128 x 64) 1,166 -> 175 (101, 24, 58).
#include "common.h"

typedef __attribute__((ext_vector_type(4))) float f32x4;

constexpr int SCAN_C = 64;                 // tokens of a chunk
constexpr int SCAN_AS = SCAN_C + 4;        // floats from one row of scores to the next in LDS
constexpr int SCAN_VC = 32, SCAN_VS = SCAN_VC + 4;   // value columns at a time, floats from one row to the next

// What the decays are, and which state an output sees.
enum { SCAN_HEAD = 0,      // decays[h]; the state after the token
       SCAN_STEP = 1,      // exp(-exp(a_log[h]) dt), k times dt, dt = softplus(dt_raw + bias); after the token, plus skip * v
       SCAN_CHANNEL = 2,   // decay[n, h D + i]; after the token
       SCAN_BONUS = 3 };   // decay[n, h D + i]; before the token, plus bonus[h, i] k_i v of the token itself

struct ScanArgs {
    const void *q, *k, *v;
    const float *decay, *p1, *p2, *p3;     // STEP: dt_raw, dt_bias, a_log, skip; BONUS: decay, bonus
    long long ldq, ldk, ldv, lda;          // elements from one token to the next
    int hq, hk, hv, group;                 // elements from one head to the next; heads that share q and k
    int H, D, Dv, held, v_act, vec;        // held: value columns in v, the others read 1; vec: rows may be read by fours
    int first, count, compact;             // chunks of every sequence: first .. first + count - 1; how slots are numbered
    const int* qstart;
    const int* rows;
    float* state;
    long long stride;
    int offset;
    // [N, H Dv]; per slot and head: addend, later state [D, Dv]; queries decayed to the chunk's start [64, DK] (a decay
    // per channel) or those decays [64]; the chunk's whole decay [DK]
    float *out, *adds, *queries, *factors;
};

// Scratch of a sequence's chunk: with one launch over all tokens the chunks lie one behind the other.
__device__ __forceinline__ size_t scan_slot(const ScanArgs& a, int seq, int c) {
    return a.compact ? (size_t)(a.qstart[seq] / SCAN_C + seq + c) : (size_t)seq * a.count + c;
}

template <typename T> __device__ __forceinline__ float4 scan_quad(const T* __restrict__ p, int n, int vec) {
    float x[4] = {0.f, 0.f, 0.f, 0.f};
    if (vec && n >= 4) VecLoad<T, 4>::load(p, x);
    else
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (e < n) x[e] = to_float(p[e]);
    return make_float4(x[0], x[1], x[2], x[3]);
}

__device__ __forceinline__ float4 mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float4 mul4(float4 a, float b) { return make_float4(a.x * b, a.y * b, a.z * b, a.w * b); }

template <int DK, int MODE, typename TQ, typename TV>
__global__ void __launch_bounds__(512)
scan_chunks_kernel(ScanArgs a) {
    constexpr bool CH = MODE >= SCAN_CHANNEL;
    constexpr int LS = DK + 4, Q4 = DK / 4;
    constexpr bool V_IN_Q = SCAN_C * LS >= SCAN_C * (SCAN_AS + SCAN_VS);
    __shared__ __align__(16) float Qs[SCAN_C * LS];                  // later the scores, and behind them the values
    __shared__ __align__(16) float Ks[SCAN_C * LS];
    __shared__ __align__(16) float Ds[CH ? SCAN_C * LS : 4];
    __shared__ __align__(16) float Vx[V_IN_Q ? 4 : SCAN_C * SCAN_VS];
    __shared__ __align__(16) float dg[CH ? 2 : 1][4][16][16];        // decays (CH: scores) inside a run of 16 tokens
    __shared__ __align__(16) float tot[4][CH ? DK : 1];              // a run's whole decay
    __shared__ float sa[SCAN_C], sdt[SCAN_C], pin[SCAN_C], sfx[SCAN_C];
    float* As = Qs;
    float* Vs = V_IN_Q ? Qs + SCAN_C * SCAN_AS : Vx;

    const int head = blockIdx.x, c = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x;
    const int lo = a.qstart[seq] + (a.first + c) * SCAN_C, hi = a.qstart[seq + 1];
    if (lo >= hi) return;
    const int nt = min(SCAN_C, hi - lo);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    const size_t slot = scan_slot(a, seq, c) * a.H + head;
    float skip = 0.f;

    if constexpr (!CH) {
        if (tid < SCAN_C) {
            float d = 1.f, dt = 0.f;
            if (tid < nt) {
                if (MODE == SCAN_HEAD) { d = a.decay[head]; dt = 1.f; }
                else {
                    const float z = a.decay[(size_t)(lo + tid) * a.H + head] + a.p1[head];
                    dt = z > 20.f ? z : log1pf(expf(z));
                    d = expf(-expf(a.p2[head]) * dt);
                }
            }
            sa[tid] = d;
            sdt[tid] = dt;
        }
        if (MODE == SCAN_STEP) skip = a.p3[head];
    }
    const TQ* q = (const TQ*)a.q + (size_t)(head / a.group) * a.hq;
    const TQ* k = (const TQ*)a.k + (size_t)(head / a.group) * a.hk;
#pragma unroll
    for (int it = 0; it < SCAN_C * Q4 / 512; ++it) {
        const int e = it * 512 + tid, t = e / Q4, i = e % Q4 * 4;
        const int n = t < nt ? a.D - i : 0;
        const float4 zero = make_float4(0.f, 0.f, 0.f, 0.f);
        *reinterpret_cast<float4*>(Qs + t * LS + i) = n > 0 ? scan_quad(q + (size_t)(lo + t) * a.ldq + i, n, a.vec) : zero;
        *reinterpret_cast<float4*>(Ks + t * LS + i) = n > 0 ? scan_quad(k + (size_t)(lo + t) * a.ldk + i, n, a.vec) : zero;
        if constexpr (CH)
            *reinterpret_cast<float4*>(Ds + t * LS + i) =
                n > 0 ? scan_quad(a.decay + (size_t)(lo + t) * a.lda + head * a.D + i, n, a.vec) : make_float4(1.f, 1.f, 1.f, 1.f);
    }
    __syncthreads();

    // -- scores: blocks of 16 x 16 (run I of queries, run J <= I of keys)
    f32x4 sc[2];
    int bi[2], bj[2];
    if constexpr (!CH) {
        if (tid < SCAN_C) {                          // down a column of its run: decay from behind token j to token i
            const int I = tid / 16, j = tid % 16;
            float p = sdt[tid];
            for (int i = 0; i < 16; ++i) {
                if (i > j) p *= sa[I * 16 + i];
                dg[0][I][i][j] = i >= j ? p : 0.f;
            }
            sfx[tid] = p;
        } else if (tid < 2 * SCAN_C) {
            const int i = tid - SCAN_C, I = i / 16;
            float p = 1.f;
            for (int t = I * 16; t <= i; ++t) p *= sa[t];
            pin[i] = p;
            if (i % 16 == 15) tot[I][0] = p;
        }
    } else {
        // inside a run pair by pair: wave (run, half of the channels), lane (query r, a quarter of the half's channels)
        constexpr int CPL = DK / 8;
        const int I = wave / 2, c0 = (wave % 2) * (DK / 2) + g * CPL;
        float qv[CPL], w[CPL], u[MODE == SCAN_BONUS ? CPL : 1];
#pragma unroll
        for (int i = 0; i < CPL; ++i) {
            qv[i] = Qs[(I * 16 + r) * LS + c0 + i];
            w[i] = 1.f;
            if constexpr (MODE == SCAN_BONUS) u[i] = c0 + i < a.D ? a.p1[head * a.D + c0 + i] : 0.f;
        }
#pragma unroll 2
        for (int j = 15; j >= 0; --j) {              // (unrolled further, all rows are loaded at once and registers spill)
            const float* kj = Ks + (I * 16 + j) * LS + c0;
            const float* dj = Ds + (I * 16 + min(j + 1, 15)) * LS + c0;
            // the decays between: of tokens j + 1 .. r, or .. r - 1 where the output sees the state before its token
            const bool on = j < (MODE == SCAN_BONUS ? r - 1 : r);
            float s = 0.f;
#pragma unroll
            for (int i = 0; i < CPL; i += 4) {
                float kx[4], dx[4];
                VecLoad<float, 4>::load(kj + i, kx);
                VecLoad<float, 4>::load(dj + i, dx);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    w[i + e] *= on ? dx[e] : 1.f;
                    float f = w[i + e];
                    if constexpr (MODE == SCAN_BONUS) f = j == r ? u[i + e] : f;
                    s = fmaf(qv[i + e] * f, kx[e], s);
                }
            }
            s = sum_xor32(sum_xor16(j <= r ? s : 0.f));
            if (g == 0) dg[wave % 2][I][r][j] = s;
        }
        __syncthreads();
        // queries decayed back to their run's start, keys to its end, in place
        for (int e = tid; e < 4 * DK; e += 512) {
            const int run = e / DK, ch = e % DK;
            float p = 1.f;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int at = (run * 16 + t) * LS + ch;
                if (MODE == SCAN_BONUS) { Qs[at] *= p; p *= Ds[at]; }
                else { p *= Ds[at]; Qs[at] *= p; }
            }
            tot[run][ch] = p;
            p = 1.f;
#pragma unroll
            for (int t = 15; t >= 0; --t) {
                const int at = (run * 16 + t) * LS + ch;
                Ks[at] *= p;
                p *= Ds[at];
            }
        }
        __syncthreads();
    }
    constexpr int BLOCKS = CH ? 6 : 10;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        const int b = wave + 8 * x;
        bi[x] = -1;
        if (b >= BLOCKS) continue;
        int I, J;
        if (CH) { I = b < 1 ? 1 : b < 3 ? 2 : 3; J = b - I * (I - 1) / 2; }
        else { I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3; J = b - I * (I + 1) / 2; }
        bi[x] = I; bj[x] = J;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < DK; m += 16) {
            float4 qf = *reinterpret_cast<const float4*>(Qs + (I * 16 + r) * LS + m + 4 * g);
            const float4 kf = *reinterpret_cast<const float4*>(Ks + (J * 16 + r) * LS + m + 4 * g);
            if constexpr (CH)
                for (int run = J + 1; run < I; ++run) qf = mul4(qf, *reinterpret_cast<const float4*>(&tot[run][m + 4 * g]));
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.x, qf.x, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.y, qf.y, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.z, qf.z, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf.w, qf.w, s, 0, 0, 0);
        }
        sc[x] = s;
    }
    if constexpr (!CH) __syncthreads();             // the factors of the runs

    // -- queries decayed back to the chunk's start, for scan_apply (one decay for all channels: that alone); the whole decay
    if constexpr (CH) {
#pragma unroll
        for (int it = 0; it < SCAN_C * Q4 / 512; ++it) {
            const int e = it * 512 + tid, t = e / Q4, i = e % Q4 * 4, I = t / 16;
            float4 x = *reinterpret_cast<const float4*>(Qs + t * LS + i);
            for (int run = 0; run < I; ++run) x = mul4(x, *reinterpret_cast<const float4*>(&tot[run][i]));
            *reinterpret_cast<float4*>(a.queries + (slot * SCAN_C + t) * DK + i) = x;
        }
    } else if (tid < SCAN_C) {
        float p = pin[tid];
        for (int run = 0; run < tid / 16; ++run) p *= tot[run][0];
        a.queries[slot * SCAN_C + tid] = p;
    }
    if (tid < DK) {
        const int ch = CH ? tid : 0;
        a.factors[slot * DK + tid] = tot[0][ch] * tot[1][ch] * tot[2][ch] * tot[3][ch];
    }
    __syncthreads();

    // -- the scores over the queries' place; keys decayed on to the chunk's end, in place
#pragma unroll
    for (int x = 0; x < 2; ++x) {
        if (bi[x] < 0) continue;
        const int I = bi[x], J = bj[x], i = I * 16 + r;
        float f[4] = {1.f, 1.f, 1.f, 1.f};
        if constexpr (!CH) {
            float p = pin[i];
            for (int run = J + 1; run < I; ++run) p *= tot[run][0];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = I == J ? dg[0][I][r][4 * g + e] : p * sfx[J * 16 + 4 * g + e];
        }
        float4 s = make_float4(sc[x][0] * f[0], sc[x][1] * f[1], sc[x][2] * f[2], sc[x][3] * f[3]);
        if (MODE == SCAN_STEP && I == J) {
            if (r == 4 * g) s.x += skip;
            if (r == 4 * g + 1) s.y += skip;
            if (r == 4 * g + 2) s.z += skip;
            if (r == 4 * g + 3) s.w += skip;
        }
        *reinterpret_cast<float4*>(As + i * SCAN_AS + J * 16 + 4 * g) = s;
    }
    if constexpr (CH) {
        for (int e = tid; e < 4 * 16 * 16; e += 512) {
            const int I = e / 256, i = e / 16 % 16, j = e % 16;
            As[(I * 16 + i) * SCAN_AS + I * 16 + j] = dg[0][I][i][j] + dg[1][I][i][j];
        }
    }
#pragma unroll
    for (int it = 0; it < SCAN_C * Q4 / 512; ++it) {
        const int e = it * 512 + tid, t = e / Q4, i = e % Q4 * 4, I = t / 16;
        float4 x = *reinterpret_cast<const float4*>(Ks + t * LS + i);
        if constexpr (CH) {
            for (int run = 3; run > I; --run) x = mul4(x, *reinterpret_cast<const float4*>(&tot[run][i]));
        } else {
            float p = sfx[t];
            for (int run = I + 1; run < 4; ++run) p *= tot[run][0];
            x = mul4(x, p);
        }
        *reinterpret_cast<float4*>(Ks + t * LS + i) = x;
    }

    // -- values, 32 columns at a time: the scores' share of the outputs, and the addend to the state
    const TV* v = (const TV*)a.v + (size_t)head * a.hv;
    const int vt = tid / 8, vc = tid % 8 * 4;
    auto fetch = [&](int col) {
        float x[4] = {0.f, 0.f, 0.f, 0.f};
        if (vt < nt) {
            const TV* row = v + (size_t)(lo + vt) * a.ldv + col;
            if (a.vec && col + 4 <= a.held) VecLoad<TV, 4>::load(row, x);
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < a.Dv) x[e] = col + e < a.held ? to_float(row[e]) : 1.f;
            if (a.v_act)
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = x[e] / (1.f + expf(-x[e]));
        }
        return make_float4(x[0], x[1], x[2], x[3]);
    };
    auto put = [&](float* p, int n, const f32x4& y, bool whole) {    // n columns are left
        if (whole && n >= 4) *reinterpret_cast<float4*>(p) = make_float4(y[0], y[1], y[2], y[3]);
        else
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (e < n) p[e] = y[e];
    };
    const bool by4 = a.Dv % 4 == 0;
    float4 next = fetch(vc);
    for (int col0 = 0; col0 < a.Dv; col0 += SCAN_VC) {
        __syncthreads();                            // the scores are there; the values before these have been read
        *reinterpret_cast<float4*>(Vs + vt * SCAN_VS + vc) = next;
        __syncthreads();
        if (col0 + SCAN_VC < a.Dv) next = fetch(col0 + SCAN_VC + vc);
        {
            const int I = wave / 2, p = wave % 2;
            f32x4 o = {0.f, 0.f, 0.f, 0.f};
            for (int s = 0; s <= I; ++s) {
                const float4 x = *reinterpret_cast<const float4*>(As + (I * 16 + r) * SCAN_AS + 16 * s + 4 * g);
                const float* y = Vs + (16 * s + 4 * g) * SCAN_VS + p * 16 + r;
                o = __builtin_amdgcn_mfma_f32_16x16x4f32(y[0], x.x, o, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x4f32(y[SCAN_VS], x.y, o, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x4f32(y[2 * SCAN_VS], x.z, o, 0, 0, 0);
                o = __builtin_amdgcn_mfma_f32_16x16x4f32(y[3 * SCAN_VS], x.w, o, 0, 0, 0);
            }
            const int t = I * 16 + r, col = col0 + p * 16 + 4 * g;
            if (t < nt && col < a.Dv) put(a.out + ((size_t)(lo + t) * a.H + head) * a.Dv + col, a.Dv - col, o, by4);
        }
        {
            // 16 channels by 32 columns a wave, or with 64 channels by 16
            constexpr int TILES = DK / 64;
            const int ct = DK == 128 ? wave : wave / 2, p0 = DK == 128 ? 0 : wave % 2;
            f32x4 s[TILES];
#pragma unroll
            for (int p = 0; p < TILES; ++p) s[p] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int m = 0; m < SCAN_C; m += 16)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = m + 4 * g + e;
                    const float x = Ks[t * LS + ct * 16 + r];
#pragma unroll
                    for (int p = 0; p < TILES; ++p)
                        s[p] = __builtin_amdgcn_mfma_f32_16x16x4f32(Vs[t * SCAN_VS + (p0 + p) * 16 + r], x, s[p], 0, 0, 0);
                }
            const int ch = ct * 16 + r;
#pragma unroll
            for (int p = 0; p < TILES; ++p) {
                const int col = col0 + (p0 + p) * 16 + 4 * g;
                if (ch < a.D && col < a.Dv) put(a.adds + (slot * a.D + ch) * a.Dv + col, a.Dv - col, s[p], by4);
            }
        }
    }
}

// In place: every chunk's addend becomes the state before that chunk, and the row's state moves on to the end of the
// last one. A thread owns V elements of a head's state; the addends of eight chunks are on their way at a time.
template <int V>
__global__ void __launch_bounds__(256)
scan_states_kernel(ScanArgs a, int dk) {
    const int head = blockIdx.y, seq = blockIdx.z;
    const int size = a.D * a.Dv, at = ((int)blockIdx.x * 256 + (int)threadIdx.x) * V;
    const int left = a.qstart[seq + 1] - a.qstart[seq] - a.first * SCAN_C;
    if (at >= size || left <= 0) return;
    const int n = min(a.count, (left + SCAN_C - 1) / SCAN_C);
    float* S = a.state + (size_t)a.rows[seq] * a.stride + a.offset + (size_t)head * size + at;
    const size_t slot0 = scan_slot(a, seq, 0) * a.H + head;
    float* add = a.adds + slot0 * size + at;
    const float* f = a.factors + slot0 * dk + at / a.Dv;
    const size_t step = (size_t)a.H * size, fstep = (size_t)a.H * dk;
    float s[V], x[8][V], y[8];
    VecLoad<float, V>::load(S, s);
    for (int c = 0; c < n; c += 8) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (c + i < n) { VecLoad<float, V>::load(add + (c + i) * step, x[i]); y[i] = f[(c + i) * fstep]; }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (c + i < n) {
                float* p = add + (c + i) * step;
                if constexpr (V == 4) *reinterpret_cast<float4*>(p) = make_float4(s[0], s[1], s[2], s[3]);
                else p[0] = s[0];
#pragma unroll
                for (int e = 0; e < V; ++e) s[e] = fmaf(y[i], s[e], x[i][e]);
            }
    }
    if constexpr (V == 4) *reinterpret_cast<float4*>(S) = make_float4(s[0], s[1], s[2], s[3]);
    else S[0] = s[0];
}

// out += queries S, 64 tokens by 32 CG columns a workgroup: CG waves side by side with 32 columns of S in registers,
// 4 / CG of those one above the other.
// CH: the queries lie decayed in scratch; else they come as they came to scan_chunks, with a decay per token.
template <int DK, int CG, bool CH, typename TQ>
__global__ void __launch_bounds__(256)
scan_apply_kernel(ScanArgs a) {
    constexpr int LS = DK + 4, Q4 = DK / 4;
    __shared__ __align__(16) float Qs[SCAN_C * LS];
    const int blocks = (a.Dv + 32 * CG - 1) / (32 * CG);
    const int head = blockIdx.x / blocks, c = blockIdx.y, seq = blockIdx.z, tid = threadIdx.x;
    const int lo = a.qstart[seq] + (a.first + c) * SCAN_C, hi = a.qstart[seq + 1];
    if (lo >= hi) return;
    const int nt = min(SCAN_C, hi - lo);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    const size_t slot = scan_slot(a, seq, c) * a.H + head;
    const int col0 = (blockIdx.x % blocks) * 32 * CG + (wave % CG) * 32, row0 = (wave / CG) * 16 * CG;
    const float* S = a.adds + slot * a.D * a.Dv + col0 + 2 * r;
    const int n = a.Dv - col0 - 2 * r;
    const bool by2 = a.Dv % 2 == 0;
    float sx[DK / 4], sy[DK / 4];                    // columns 2 r and 2 r + 1 of channels 16 s + 4 g + e
#pragma unroll
    for (int i = 0; i < DK / 4; ++i) {
        const int ch = i / 4 * 16 + 4 * g + i % 4;
        sx[i] = sy[i] = 0.f;
        if (ch < a.D && n > 0) {
            const float* p = S + (size_t)ch * a.Dv;
            if (by2) { const float2 t = *reinterpret_cast<const float2*>(p); sx[i] = t.x; sy[i] = t.y; }
            else { sx[i] = p[0]; if (n > 1) sy[i] = p[1]; }
        }
    }
#pragma unroll
    for (int it = 0; it < SCAN_C * Q4 / 256; ++it) {
        const int e = it * 256 + tid, t = e / Q4, i = e % Q4 * 4;
        float4 x;
        if constexpr (CH) x = *reinterpret_cast<const float4*>(a.queries + (slot * SCAN_C + t) * DK + i);
        else {
            const TQ* q = (const TQ*)a.q + (size_t)(head / a.group) * a.hq + (size_t)(lo + t) * a.ldq + i;
            x = t < nt && i < a.D ? mul4(scan_quad(q, a.D - i, a.vec), a.queries[slot * SCAN_C + t]) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        *reinterpret_cast<float4*>(Qs + t * LS + i) = x;
    }
    __syncthreads();
    f32x4 x[CG], y[CG];
#pragma unroll
    for (int i = 0; i < CG; ++i) x[i] = y[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < DK / 16; ++s) {
        float q[CG][4];
#pragma unroll
        for (int i = 0; i < CG; ++i) VecLoad<float, 4>::load(Qs + (row0 + i * 16 + r) * LS + 16 * s + 4 * g, q[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < CG; ++i) {
                x[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[s * 4 + e], q[i][e], x[i], 0, 0, 0);
                y[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(sy[s * 4 + e], q[i][e], y[i], 0, 0, 0);
            }
    }
    // a lane has columns col0 + 8 g .. + 7 of token row0 + 16 i + r
#pragma unroll
    for (int i = 0; i < CG; ++i) {
        const int t = row0 + i * 16 + r, col = col0 + 8 * g;
        if (t >= nt || col >= a.Dv) continue;
        float* p = a.out + ((size_t)(lo + t) * a.H + head) * a.Dv + col;
        if (a.Dv % 4 == 0 && col + 8 <= a.Dv) {
            float4 u = *reinterpret_cast<const float4*>(p), w = *reinterpret_cast<const float4*>(p + 4);
            u.x += x[i][0]; u.y += y[i][0]; u.z += x[i][1]; u.w += y[i][1];
            w.x += x[i][2]; w.y += y[i][2]; w.z += x[i][3]; w.w += y[i][3];
            *reinterpret_cast<float4*>(p) = u;
            *reinterpret_cast<float4*>(p + 4) = w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < a.Dv) p[e] += e % 2 ? y[i][e / 2] : x[i][e / 2];
        }
    }
}

template <int DK, int MODE, typename TQ, typename TV>
static void launch_scan(const ScanArgs& a, int n_seqs, bool vec_state, hipStream_t s) {
    hipLaunchKernelGGL((scan_chunks_kernel<DK, MODE, TQ, TV>), dim3(a.H, a.count, n_seqs), dim3(512), 0, s, a);
    const int size = a.D * a.Dv;
    if (vec_state) hipLaunchKernelGGL((scan_states_kernel<4>), dim3((size / 4 + 255) / 256, a.H, n_seqs), dim3(256), 0, s, a, DK);
    else hipLaunchKernelGGL((scan_states_kernel<1>), dim3((size + 255) / 256, a.H, n_seqs), dim3(256), 0, s, a, DK);
    constexpr bool CH = MODE >= SCAN_CHANNEL;
    if (a.Dv <= 32) hipLaunchKernelGGL((scan_apply_kernel<DK, 1, CH, TQ>), dim3(a.H, a.count, n_seqs), dim3(256), 0, s, a);
    else if (a.Dv <= 64) hipLaunchKernelGGL((scan_apply_kernel<DK, 2, CH, TQ>), dim3(a.H, a.count, n_seqs), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((scan_apply_kernel<DK, 4, CH, TQ>), dim3(a.H * ((a.Dv + 127) / 128), a.count, n_seqs), dim3(256), 0, s, a);
}

// One of the recurrences above over chunks first .. first + count - 1 of every sequence (64 tokens each; a sequence
// may have fewer), from and into the rows' states. D <= 128. adds, queries and factors: scratch of `slots` chunks,
// n_tokens / 64 + n_seqs of them with compact (first 0 and count for the longest sequence), n_seqs * count without.
// q and k are float32 with q_f32, else in dtype like v. dtype 0 float32, 1 bfloat16.
SOC_EXPORT int soc_scan(int mode, const void* q, long long ldq, int hq, const void* k, long long ldk, int hk, int group, int q_f32,
                        const void* v, long long ldv, int hv, int v_act, int ones, const float* decay, long long lda,
                        const float* p1, const float* p2, const float* p3, int H, int D, int Dv, float* state, long long stride,
                        int offset, const int* seq_qstart, const int* seq_rows, int n_seqs, int first, int count, int compact,
                        float* out, float* adds, float* queries, float* factors, int dtype, hipStream_t stream) {
    if (n_seqs <= 0 || H <= 0 || count <= 0) return 0;
    if (D < 1 || D > 128 || Dv < 1 || ones < 0 || ones >= Dv || group < 1 || H % group || n_seqs > 65535 || count > 65535 || first < 0 ||
        (compact && first) || !adds || !queries || !factors || !decay) return (int)hipErrorInvalidValue;
    ScanArgs a;
    a.q = q; a.k = k; a.v = v; a.decay = decay; a.p1 = p1; a.p2 = p2; a.p3 = p3;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.lda = lda; a.hq = hq; a.hk = hk; a.hv = hv; a.group = group;
    a.H = H; a.D = D; a.Dv = Dv; a.held = Dv - ones; a.v_act = v_act;
    a.first = first; a.count = count; a.compact = compact; a.qstart = seq_qstart; a.rows = seq_rows;
    a.state = state; a.stride = stride; a.offset = offset; a.out = out; a.adds = adds; a.queries = queries; a.factors = factors;
    const int qe = q_f32 || dtype == 0 ? 16 : 8, ve = dtype == 0 ? 16 : 8;       // bytes of four elements
    a.vec = D % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && lda % 4 == 0 && hq % 4 == 0 && hk % 4 == 0 && hv % 4 == 0 &&
            (uintptr_t)q % qe == 0 && (uintptr_t)k % qe == 0 && (uintptr_t)v % ve == 0 && (uintptr_t)decay % 16 == 0;
    const bool vec_state = Dv % 4 == 0 && stride % 4 == 0 && offset % 4 == 0 && (uintptr_t)state % 16 == 0;
#define SOC_SCAN(MODE_, TQ_, TV_) \
    do { if (D <= 64) launch_scan<64, MODE_, TQ_, TV_>(a, n_seqs, vec_state, stream); else launch_scan<128, MODE_, TQ_, TV_>(a, n_seqs, vec_state, stream); } while (0)
    if (mode == SCAN_HEAD && q_f32) { if (dtype == 0) SOC_SCAN(SCAN_HEAD, float, float); else SOC_SCAN(SCAN_HEAD, float, bf16); }
    else if (mode == SCAN_CHANNEL && q_f32) { if (dtype == 0) SOC_SCAN(SCAN_CHANNEL, float, float); else SOC_SCAN(SCAN_CHANNEL, float, bf16); }
    else if (mode == SCAN_STEP && !q_f32 && p1 && p2 && p3) { if (dtype == 0) SOC_SCAN(SCAN_STEP, float, float); else SOC_SCAN(SCAN_STEP, bf16, bf16); }
    else if (mode == SCAN_BONUS && !q_f32 && p1) { if (dtype == 0) SOC_SCAN(SCAN_BONUS, float, float); else SOC_SCAN(SCAN_BONUS, bf16, bf16); }
    else return (int)hipErrorInvalidValue;
#undef SOC_SCAN
    return soc_last_error();
}
