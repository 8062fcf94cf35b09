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
// No further off float64 than the walk: products of decays are formed in float64 and rounded once (a head's decay is the same
// in every chunk, and so would its rounding be: its whole chunk's goes to scan_states in two parts), contractions are summed
// in blocks, and the scores of the delta rule, whose chunk inverts a matrix of them, are float64 matrix instructions. Error of
// results / states against the walk's, 2,048 tokens, 1e-7: retention 1.5 / 1.2 against 3.0 / 2.9, linear attention with
// activations 1.1 / 0.9 against 1.6 / 3.0, with a decay per channel 11 / 15 against 12 / 15, wkv 1.4 / 1.1 against 2.5 / 2.5,
// ssd 1.4 / 1.7 against 1.6 / 1.8, delta rule 0.8 to 4 / 0.7 to 7 against 0.8 to 9 / 0.6 to 16 (unlike to nearly repeating
// keys). With one chain per sum and float32 throughout it was 11 / 11 for retention, 15 / 16 with activations, 1.9 to 10 / 2
// to 14 for the delta rule, 2 to 9 times the walk's; the difference costs up to 5 % of the time.
//
// Bound by memory: per chunk and head the addend (D x Dv float32) is written, read, written as a state and read
// again, the outputs written, read and written. 64 tokens: with 32 the addends weigh twice as much, with 128 a
// chunk's queries, keys and decays of 128 channels do not fit LDS.
//
// Measured for 2,048 tokens of one prompt, us, the walk -> these kernels with what prepares them: retention (20 heads of
// 128 x 128) 908 -> 109 (chunks 47, states 17, apply 30), gated linear attention (10 of 128 x 256) 1,030 -> 130 (66, 17, 28),
// wkv (40 of 64 x 64) 595 -> 99 with its norm (52, 10, 17), ssd (80 of 128 x 64) 1,166 -> 168 (91, 22, 56); the gated
// delta rule (20 of 128 x 128), 3,000 tokens, 700 -> 284 with its convolutions (2,048 tokens: chunks 104, states 65, apply 28). scan_chunks is
// bound by its reads of LDS, a 4-byte read per operand and product where an operand lies across the tokens.
#include "common.h"
#include "recurrent.h"          // lds_barrier: loads and stores on their way are not waited for

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) double f64x4;

constexpr int SCAN_C = 64;                 // tokens of a chunk
constexpr int SCAN_AS = SCAN_C + 4;        // floats from one row of scores to the next in LDS
constexpr int SCAN_VC = 32, SCAN_VS = SCAN_VC + 4;   // value columns at a time, floats from one row to the next

// Waves of a workgroup that takes a chunk: 16 where LDS leaves room for one workgroup on a compute unit only.
constexpr int scan_waves(int DK, bool one) { return DK == 128 && one ? 16 : 8; }

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
    int n_seqs, least;                     // sequences of fewer than `least` tokens are not these kernels'
    const int* qstart;
    const int* rows;
    float* state;
    long long stride;
    int offset;
    // [N, H Dv]; per slot and head: addend, later state, in tiles; queries decayed to the chunk's start [64, DK] (a decay
    // per channel) or those decays [64]; the chunk's whole decay [DK]
    float *out, *adds, *queries, *factors;
};

// Addends and states lie in tiles of 16 channels x 16 columns as a lane of the matrix products has them, so that a
// wave's store or load is 1 KB in one piece and no size needs a mask: [channel tile][column tile][lane][4], lane
// (r, g) = (lane % 16, lane / 16) holding channels 4 g .. 4 g + 3 of one column. The columns of two neighbouring tiles
// take turns by fours, so that the outputs of a lane of scan_apply are eight neighbours.
__device__ __forceinline__ int scan_col(int p, int r) { return r / 4 * 8 + p * 4 + r % 4; }     // within 32 columns
__host__ __device__ __forceinline__ int scan_tiles(int Dv) { return (Dv + 31) / 32 * 2; }

// Chunks are numbered for the grid and for scratch. With one launch over all tokens (compact) those of the l-th sequence of
// `least` tokens and more begin at number qstart / 64 + l, so that they lie nearly one behind the other whatever the
// lengths; else at l * count. A wave looks at 64 sequences at a time. A step's decoding rows are not among these sequences: each
// would fill one token of a chunk, and a chunk costs the same however few of its tokens there are.
struct ScanPlace { int seq, c, slot; };
template <typename Args, typename Is>
__device__ __forceinline__ bool scan_search(const Args& a, ScanPlace& at, Is is) {
    const int lane = threadIdx.x % 64;
    for (int seq0 = 0, found = 0; seq0 < a.n_seqs; seq0 += 64) {
        const int seq = min(seq0 + lane, a.n_seqs - 1), start = a.qstart[seq], len = a.qstart[seq + 1] - start;
        const unsigned long long own = __ballot(seq0 + lane < a.n_seqs && len >= a.least);
        const int l = found + __popcll(own & ((1ull << lane) - 1));
        const int slot = a.compact ? start / SCAN_C + l : l * a.count;
        const unsigned long long hit = __ballot((own >> lane & 1) && is(l, slot, a.compact ? (len + SCAN_C - 1) / SCAN_C : a.count));
        if (hit) {
            const int src = __builtin_ctzll(hit);
            at.seq = seq0 + src;
            at.slot = __builtin_amdgcn_readlane(slot, src);
            return true;
        }
        found += __popcll(own);
    }
    return false;
}
// the sequence and the chunk of number b; or, of the l-th such sequence, the first chunk's number
// (one sequence alone is not searched for: its chunks' numbers are their own)
template <typename Args> __device__ __forceinline__ bool scan_chunk(const Args& a, int b, ScanPlace& at) {
    if (a.n_seqs == 1) {
        at.seq = 0; at.c = at.slot = b;
        return true;
    }
    if (!scan_search(a, at, [&](int, int slot, int n) { return slot <= b && b < slot + n; })) return false;
    at.c = b - at.slot;
    at.slot = b;
    return true;
}
template <typename Args> __device__ __forceinline__ bool scan_sequence(const Args& a, int which, ScanPlace& at) {
    if (a.n_seqs == 1) {
        at.seq = at.slot = 0;
        return true;
    }
    return scan_search(a, at, [&](int l, int, int) { return l == which; });
}

// Four elements of a row of which the first n exist (n <= 0: none; then p is not read where vec). With vec the load
// stands on its own, at an address that exists whatever n: a branch around it would make the wave wait for it there.
template <typename T> __device__ __forceinline__ float4 scan_quad(const T* __restrict__ p, const T* __restrict__ any, int n, int vec) {
    float x[4] = {0.f, 0.f, 0.f, 0.f};
    if (vec) {
        VecLoad<T, 4>::load(n > 0 ? p : any, x);
        return n > 0 ? make_float4(x[0], x[1], x[2], x[3]) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (e < n) x[e] = to_float(p[e]);
    return make_float4(x[0], x[1], x[2], x[3]);
}

__device__ __forceinline__ float4 mul4(float4 a, float4 b) { return make_float4(a.x * b.x, a.y * b.y, a.z * b.z, a.w * b.w); }
__device__ __forceinline__ float4 mul4(float4 a, float b) { return make_float4(a.x * b, a.y * b, a.z * b, a.w * b); }

__device__ __forceinline__ f32x4 mfma4(float a0, float a1, float a2, float a3, float4 b, f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a0, b.x, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a1, b.y, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x4f32(a2, b.z, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a3, b.w, c, 0, 0, 0);
}
// f(I0) + .. + f(I0 + N - 1), pairwise: blocks of 16 of a contraction have sums of their own, because one chain of 64 or 128
// additions into the same float32 sum is off by several times what the walk's short ones are.
template <int N, int I0 = 0, typename F> __device__ __forceinline__ f32x4 sum_pairs(F f) {
    if constexpr (N == 1) return f(I0);
    else return sum_pairs<N / 2, I0>(f) + sum_pairs<N - N / 2, I0 + N / 2>(f);
}
// sum over k of 16 of col[k][m] row[n][k]: col points at [4 g][m of the lane] with ld floats between the k, row at [n of the lane][4 g]
__device__ __forceinline__ f32x4 mfma_col_row(const float* col, int ld, const float* row, f32x4 c) {
    return mfma4(col[0], col[ld], col[2 * ld], col[3 * ld], *reinterpret_cast<const float4*>(row), c);
}

// 32 columns of values (Vs [64][SCAN_VS]): out = X V of the chunk's tokens (X [64][SCAN_AS], lower triangle), and the
// addend Z^T V to the state in tiles (Z [64][DK + 4]). NW waves, eight or more.
template <int DK, int NW>
__device__ __forceinline__ void scan_values(float* __restrict__ out, int H, int Dv, bool by4, int lo, int nt, int head, int col0, int tiles,
                                            const float* Z, const float* Vs, const float* X, float* __restrict__ adds, int ch_tiles,
                                            int wave, int r, int g) {
    constexpr int LS = DK + 4, PER = NW * 16 / DK, TILES = 2 / PER;      // PER: waves that share 16 channels
    if (NW == 8 || wave < 8) {
        const int I = wave / 2, p = wave % 2;
        const float* row = X + (I * 16 + r) * SCAN_AS + 4 * g;
        const float* col_v = Vs + 4 * g * SCAN_VS + p * 16 + r;
        float v0 = col_v[16 * I * SCAN_VS], v1 = col_v[(16 * I + 1) * SCAN_VS], v2 = col_v[(16 * I + 2) * SCAN_VS], v3 = col_v[(16 * I + 3) * SCAN_VS];
        f32x4 own = {0.f, 0.f, 0.f, 0.f};
        // The tokens' own run: X is 0 above its diagonal, and 0 times a later token's value that is not finite is not 0. Such a
        // run (any lane's four of the 16 x 16 values) is added up token by token, its products below are of zeros.
        if (__any(!(v0 * 0.f + v1 * 0.f + v2 * 0.f + v3 * 0.f == 0.f))) {
            for (int j = 0; j <= r; ++j) {
                const float x = X[(I * 16 + r) * SCAN_AS + I * 16 + j];
                const float* v = Vs + (I * 16 + j) * SCAN_VS + p * 16 + 4 * g;
#pragma unroll
                for (int e = 0; e < 4; ++e) own[e] = fmaf(x, v[e], own[e]);
            }
            v0 = v1 = v2 = v3 = 0.f;
        }
        f32x4 o = {0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < I; ++s) o += mfma_col_row(col_v + 16 * s * SCAN_VS, SCAN_VS, row + 16 * s, (f32x4){0.f, 0.f, 0.f, 0.f});
        o += mfma4(v0, v1, v2, v3, *reinterpret_cast<const float4*>(row + 16 * I), (f32x4){0.f, 0.f, 0.f, 0.f});
        o += own;
        const int t = I * 16 + r, col = col0 + p * 16 + 4 * g;
        if (t < nt) {
            float* to = out + ((size_t)(lo + t) * H + head) * Dv + col;
            if (by4 && col + 4 <= Dv) *reinterpret_cast<float4*>(to) = make_float4(o[0], o[1], o[2], o[3]);
            else
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (col + e < Dv) to[e] = o[e];
        }
    }
    const int ct = wave / PER, p0 = wave % PER;      // 16 channels by both tiles of columns, or by one
    f32x4 s[TILES][4];                               // (each sum from the first token on: under decays the terms grow along it)
#pragma unroll
    for (int p = 0; p < TILES; ++p)
#pragma unroll
        for (int e = 0; e < 4; ++e) s[p][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int m = 0; m < SCAN_C; m += 16)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = m + 4 * g + e;
            const float x = Z[t * LS + ct * 16 + r];
#pragma unroll
            for (int p = 0; p < TILES; ++p) s[p][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(x, Vs[t * SCAN_VS + scan_col(p0 + p, r)], s[p][e], 0, 0, 0);
        }
    if (ct < ch_tiles) {
#pragma unroll
        for (int p = 0; p < TILES; ++p) {
            const f32x4 y = (s[p][0] + s[p][1]) + (s[p][2] + s[p][3]);
            *reinterpret_cast<float4*>(adds + ((size_t)(ct * tiles + col0 / 16 + p0 + p) * 64 + 16 * g + r) * 4) = make_float4(y[0], y[1], y[2], y[3]);
        }
    }
}

template <int DK, int MODE, typename TQ, typename TV>
__global__ void __launch_bounds__(64 * scan_waves(DK, MODE >= SCAN_CHANNEL))
scan_chunks_kernel(ScanArgs a) {
    constexpr bool CH = MODE >= SCAN_CHANNEL;
    constexpr int LS = DK + 4, Q4 = DK / 4, NW = scan_waves(DK, CH), NT = 64 * NW;
    constexpr bool V_IN_Q = SCAN_C * LS >= SCAN_C * (SCAN_AS + SCAN_VS);
    __shared__ __align__(16) float Qs[SCAN_C * LS];                  // later the scores, and behind them the values
    __shared__ __align__(16) float Ks[SCAN_C * LS];
    __shared__ __align__(16) float Ds[CH ? SCAN_C * LS : 4];
    __shared__ __align__(16) float Vx[V_IN_Q ? 4 : SCAN_C * SCAN_VS];
    __shared__ __align__(16) float dg[CH ? NW / 4 : 1][4][16][16];   // decays (CH: scores) inside a run of 16 tokens
    __shared__ __align__(16) float tot[4][CH ? DK : 1];              // a run's whole decay
    __shared__ float sa[SCAN_C], sdt[SCAN_C], pin[SCAN_C], sfx[SCAN_C];
    __shared__ double run_decay[4];
    float* As = Qs;
    float* Vs = V_IN_Q ? Qs + SCAN_C * SCAN_AS : Vx;

    const int head = blockIdx.x, tid = threadIdx.x;
    ScanPlace at;
    if (!scan_chunk(a, blockIdx.y, at)) return;
    const int lo = a.qstart[at.seq] + (a.first + at.c) * SCAN_C, hi = a.qstart[at.seq + 1];
    if (lo >= hi) return;
    const int nt = min(SCAN_C, hi - lo);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    const size_t slot = (size_t)at.slot * a.H + head;
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
    const TQ* q = (const TQ*)a.q + (size_t)(head / a.group) * a.hq + (size_t)lo * a.ldq;
    const TQ* k = (const TQ*)a.k + (size_t)(head / a.group) * a.hk + (size_t)lo * a.ldk;
    const float* dec = CH ? a.decay + (size_t)lo * a.lda + head * a.D : nullptr;
    constexpr int ROUNDS = SCAN_C * Q4 / NT;
    float4 fq[ROUNDS], fk[ROUNDS], fd[CH ? ROUNDS : 1];
#pragma unroll
    for (int it = 0; it < ROUNDS; ++it) {            // all loads before the first use
        const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4, n = t < nt ? a.D - i : 0;
        fq[it] = scan_quad(q + (size_t)t * a.ldq + i, q, n, a.vec);
        fk[it] = scan_quad(k + (size_t)t * a.ldk + i, k, n, a.vec);
        if constexpr (CH) {
            fd[it] = scan_quad(dec + (size_t)t * a.lda + i, dec, n, a.vec);
            if (n < 1) fd[it].x = 1.f;
            if (n < 2) fd[it].y = 1.f;
            if (n < 3) fd[it].z = 1.f;
            if (n < 4) fd[it].w = 1.f;
        }
    }
#pragma unroll
    for (int it = 0; it < ROUNDS; ++it) {
        const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4;
        *reinterpret_cast<float4*>(Qs + t * LS + i) = fq[it];
        *reinterpret_cast<float4*>(Ks + t * LS + i) = fk[it];
        if constexpr (CH) *reinterpret_cast<float4*>(Ds + t * LS + i) = fd[it];
    }
    __syncthreads();

    // -- scores: blocks of 16 x 16 (run I of queries, run J <= I of keys)
    constexpr int BLOCKS = CH ? 6 : 10, MINE = (BLOCKS + NW - 1) / NW;
    f32x4 sc[MINE];
    int bi[MINE], bj[MINE];
    if constexpr (!CH) {
        if (tid < SCAN_C) {                          // down a column of its run: decay from behind token j to token i
            const int I = tid / 16, j = tid % 16;
            double p = sdt[tid];
            for (int i = 0; i < 16; ++i) {
                if (i > j) p *= sa[I * 16 + i];
                dg[0][I][i][j] = i >= j ? (float)p : 0.f;
            }
            sfx[tid] = (float)p;
        } else if (tid < 2 * SCAN_C) {
            const int i = tid - SCAN_C, I = i / 16;
            double p = 1.0;
            for (int t = I * 16; t <= i; ++t) p *= sa[t];
            pin[i] = (float)p;
            if (i % 16 == 15) { tot[I][0] = (float)p; run_decay[I] = p; }
        }
    } else {
        // inside a run pair by pair: wave (run, share of the channels), lane (query r, a quarter of the share)
        constexpr int PARTS = NW / 4, CPL = DK / 4 / PARTS;
        const int I = wave / PARTS, c0 = (wave % PARTS) * (DK / PARTS) + g * CPL;
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
            if (g == 0) dg[wave % PARTS][I][r][j] = s;
        }
        lds_barrier();
        // queries decayed back to their run's start, keys to its end, in place
        for (int e = tid; e < 4 * DK; e += NT) {
            const int run = e / DK, ch = e % DK;
            double p = 1.0;
#pragma unroll
            for (int t = 0; t < 16; ++t) {
                const int at = (run * 16 + t) * LS + ch;
                if (MODE == SCAN_BONUS) { Qs[at] = (float)(Qs[at] * p); p *= Ds[at]; }
                else { p *= Ds[at]; Qs[at] = (float)(Qs[at] * p); }
            }
            tot[run][ch] = (float)p;
            p = 1.0;
#pragma unroll
            for (int t = 15; t >= 0; --t) {
                const int at = (run * 16 + t) * LS + ch;
                Ks[at] = (float)(Ks[at] * p);
                p *= Ds[at];
            }
        }
        lds_barrier();
    }
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
        const int b = wave + NW * x;
        bi[x] = -1;
        if (b >= BLOCKS) continue;
        int I, J;
        if (CH) { I = b < 1 ? 1 : b < 3 ? 2 : 3; J = b - I * (I - 1) / 2; }
        else { I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3; J = b - I * (I + 1) / 2; }
        bi[x] = I; bj[x] = J;
        float4 between[CH ? DK / 16 : 1];            // the whole runs' decays
        if constexpr (CH) {
#pragma unroll
            for (int m = 0; m < DK / 16; ++m) between[m] = make_float4(1.f, 1.f, 1.f, 1.f);
            for (int run = J + 1; run < I; ++run)
#pragma unroll
                for (int m = 0; m < DK / 16; ++m) between[m] = mul4(between[m], *reinterpret_cast<const float4*>(&tot[run][16 * m + 4 * g]));
        }
        sc[x] = sum_pairs<DK / 16>([&](int m) {
            float4 qf = *reinterpret_cast<const float4*>(Qs + (I * 16 + r) * LS + 16 * m + 4 * g);
            const float4 kf = *reinterpret_cast<const float4*>(Ks + (J * 16 + r) * LS + 16 * m + 4 * g);
            if constexpr (CH) qf = mul4(qf, between[m]);
            return mfma4(kf.x, kf.y, kf.z, kf.w, qf, (f32x4){0.f, 0.f, 0.f, 0.f});
        });
    }
    if constexpr (!CH) lds_barrier();             // the factors of the runs

    // -- queries decayed back to the chunk's start, for scan_apply (one decay for all channels: that alone); the whole decay
    if constexpr (CH) {
#pragma unroll
        for (int it = 0; it < SCAN_C * Q4 / NT; ++it) {
            const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4, I = t / 16;
            float4 x = *reinterpret_cast<const float4*>(Qs + t * LS + i);
            for (int run = 0; run < I; ++run) x = mul4(x, *reinterpret_cast<const float4*>(&tot[run][i]));
            *reinterpret_cast<float4*>(a.queries + (slot * SCAN_C + t) * DK + i) = x;
        }
    } else if (tid < SCAN_C) {
        float p = pin[tid];
        for (int run = 0; run < tid / 16; ++run) p *= tot[run][0];
        a.queries[slot * SCAN_C + tid] = p;
    }
    if constexpr (CH) {
        if (tid < DK) a.factors[slot * DK + tid] = tot[0][tid] * tot[1][tid] * tot[2][tid] * tot[3][tid];
    } else if (tid == 0) {                           // in two parts: a head's decay is the same in every chunk, and so is its rounding
        const double whole = run_decay[0] * run_decay[1] * run_decay[2] * run_decay[3];
        a.factors[slot * DK] = (float)whole;
        a.factors[slot * DK + 1] = (float)(whole - (double)(float)whole);
    }
    lds_barrier();

    // -- the scores over the queries' place; keys decayed on to the chunk's end, in place
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
        if (bi[x] < 0) continue;
        const int I = bi[x], J = bj[x], i = I * 16 + r;
        float f[4] = {1.f, 1.f, 1.f, 1.f};
        if constexpr (!CH) {
            float p = pin[i];
            for (int run = J + 1; run < I; ++run) p *= tot[run][0];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = I == J ? dg[0][I][r][4 * g + e] : p * sfx[J * 16 + 4 * g + e];
        }
        float y[4];                                  // (a later key that is not finite: its score is 0, not 0 times that)
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = I != J || 4 * g + e <= r ? sc[x][e] * f[e] : 0.f;
        float4 s = make_float4(y[0], y[1], y[2], y[3]);
        if (MODE == SCAN_STEP && I == J) {
            if (r == 4 * g) s.x += skip;
            if (r == 4 * g + 1) s.y += skip;
            if (r == 4 * g + 2) s.z += skip;
            if (r == 4 * g + 3) s.w += skip;
        }
        *reinterpret_cast<float4*>(As + i * SCAN_AS + J * 16 + 4 * g) = s;
    }
    if constexpr (CH) {
        for (int e = tid; e < 4 * 16 * 16; e += NT) {
            const int I = e / 256, i = e / 16 % 16, j = e % 16;
            float x = dg[0][I][i][j];
#pragma unroll
            for (int part = 1; part < NW / 4; ++part) x += dg[part][I][i][j];
            As[(I * 16 + i) * SCAN_AS + I * 16 + j] = x;
        }
    }
#pragma unroll
    for (int it = 0; it < SCAN_C * Q4 / NT; ++it) {
        const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4, I = t / 16;
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
    const TV* v = (const TV*)a.v + (size_t)head * a.hv + (size_t)lo * a.ldv;
    const int vt = tid / 8, vc = tid % 8 * 4;
    auto fetch = [&](int col) {
        float4 x = scan_quad(v + (size_t)vt * a.ldv + col, v, vt < nt ? a.held - col : 0, a.vec);      // (threads from 512 on: none)
        if (a.held < a.Dv && vt < nt) {
            if (col >= a.held) x.x = 1.f;
            if (col + 1 >= a.held) x.y = 1.f;
            if (col + 2 >= a.held) x.z = 1.f;
            if (col + 3 >= a.held) x.w = 1.f;
        }
        return x;
    };
    const bool by4 = a.Dv % 4 == 0;
    const int tiles = scan_tiles(a.Dv);
    float* adds = a.adds + slot * ((a.D + 15) / 16) * tiles * 256;
    float4 next = fetch(vc);
    for (int col0 = 0; col0 < a.Dv; col0 += SCAN_VC) {
        if (a.v_act) next = make_float4(next.x / (1.f + expf(-next.x)), next.y / (1.f + expf(-next.y)), next.z / (1.f + expf(-next.z)), next.w / (1.f + expf(-next.w)));
        lds_barrier();                              // the scores are there; the values before these have been read
        if (NT == 512 || tid < 512) *reinterpret_cast<float4*>(Vs + vt * SCAN_VS + vc) = next;
        lds_barrier();
        if (col0 + SCAN_VC < a.Dv) next = fetch(col0 + SCAN_VC + vc);
        scan_values<DK, NW>(a.out, a.H, a.Dv, by4, lo, nt, head, col0, tiles, Ks, Vs, As, adds, (a.D + 15) / 16, wave, r, g);
    }
}

// In place: every chunk's addend becomes the state before that chunk, and the row's state moves on to the end of the
// last one. A thread owns a lane's four elements of a tile; the addends of eight chunks are on their way at a time.
// CH: a factor per channel; else one for all, in two parts.
template <bool CH>
__global__ void __launch_bounds__(256)
scan_states_kernel(ScanArgs a, int dk) {
    ScanPlace in;
    if (!scan_sequence(a, blockIdx.z, in)) return;
    const int head = blockIdx.y, seq = in.seq, tiles = scan_tiles(a.Dv);
    const int size = (a.D + 15) / 16 * tiles * 64, at = (int)blockIdx.x * 256 + (int)threadIdx.x;     // in pieces of four
    const int left = a.qstart[seq + 1] - a.qstart[seq] - a.first * SCAN_C;
    if (at >= size || left <= 0) return;
    const int n = min(a.count, (left + SCAN_C - 1) / SCAN_C);
    const int lane = at % 64, ct = at / 64 % tiles, ch = at / 64 / tiles * 16 + lane / 16 * 4;
    const int col = ct / 2 * 32 + scan_col(ct % 2, lane % 16);
    float* S = a.state + (size_t)a.rows[seq] * a.stride + a.offset + (size_t)head * a.D * a.Dv + (size_t)ch * a.Dv + col;
    const size_t slot0 = (size_t)in.slot * a.H + head;
    float4* add = reinterpret_cast<float4*>(a.adds) + slot0 * size + at;
    const float* f = a.factors + slot0 * dk + (CH ? ch : 0);
    const size_t step = (size_t)a.H * size, fstep = (size_t)a.H * dk;
    float s[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] = col < a.Dv && ch + e < a.D ? S[(size_t)e * a.Dv] : 0.f;
    for (int c = 0; c < n; c += 8) {
        float4 x[8], y[CH ? 8 : 1];
        float2 one[CH ? 1 : 8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int cc = min(c + i, n - 1);
            x[i] = add[cc * step];
            if constexpr (CH) y[i] = *reinterpret_cast<const float4*>(f + cc * fstep);
            else one[i] = *reinterpret_cast<const float2*>(f + cc * fstep);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (c + i < n) {
                add[(c + i) * step] = make_float4(s[0], s[1], s[2], s[3]);
                if constexpr (CH) {
                    s[0] = fmaf(y[i].x, s[0], x[i].x);
                    s[1] = fmaf(y[i].y, s[1], x[i].y);
                    s[2] = fmaf(y[i].z, s[2], x[i].z);
                    s[3] = fmaf(y[i].w, s[3], x[i].w);
                } else {
                    s[0] = fmaf(one[i].x, s[0], fmaf(one[i].y, s[0], x[i].x));
                    s[1] = fmaf(one[i].x, s[1], fmaf(one[i].y, s[1], x[i].y));
                    s[2] = fmaf(one[i].x, s[2], fmaf(one[i].y, s[2], x[i].z));
                    s[3] = fmaf(one[i].x, s[3], fmaf(one[i].y, s[3], x[i].w));
                }
            }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (col < a.Dv && ch + e < a.D) S[(size_t)e * a.Dv] = s[e];
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
    const int head = blockIdx.x / blocks, tid = threadIdx.x;
    ScanPlace at;
    if (!scan_chunk(a, blockIdx.y, at)) return;
    const int lo = a.qstart[at.seq] + (a.first + at.c) * SCAN_C, hi = a.qstart[at.seq + 1];
    if (lo >= hi) return;
    const int nt = min(SCAN_C, hi - lo);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    const size_t slot = (size_t)at.slot * a.H + head;
    const int col0 = (blockIdx.x % blocks) * 32 * CG + (wave % CG) * 32, row0 = (wave / CG) * 16 * CG;
    // two tiles of 16 columns; channels 16 s + 4 g .. + 3 in piece s (tiles beyond the last channel's: the last one, whose
    // queries are zeros; columns beyond the last tile's: read at a place that exists, not used)
    const int tiles = scan_tiles(a.Dv), ch_tiles = (a.D + 15) / 16;
    const float4* S = reinterpret_cast<const float4*>(a.adds) + (slot * ch_tiles * tiles + min(col0 / 16, tiles - 2)) * 64 + lane;
    float4 sx[DK / 16], sy[DK / 16];
#pragma unroll
    for (int i = 0; i < DK / 16; ++i) {
        const float4* p = S + (size_t)min(i, ch_tiles - 1) * tiles * 64;
        sx[i] = p[0];
        sy[i] = p[64];
    }
#pragma unroll
    for (int it = 0; it < SCAN_C * Q4 / 256; ++it) {
        const int e = it * 256 + tid, t = e / Q4, i = e % Q4 * 4;
        float4 x;
        if constexpr (CH) x = *reinterpret_cast<const float4*>(a.queries + (slot * SCAN_C + t) * DK + i);
        else {
            const TQ* q = (const TQ*)a.q + (size_t)(head / a.group) * a.hq + (size_t)lo * a.ldq;
            x = mul4(scan_quad(q + (size_t)t * a.ldq + i, q, t < nt ? a.D - i : 0, a.vec), a.queries[slot * SCAN_C + t]);
        }
        *reinterpret_cast<float4*>(Qs + t * LS + i) = x;
    }
    __syncthreads();
    // a lane has columns col0 + 8 g .. + 7 of token row0 + 16 i + r; a column's sum in parts (see sum_pairs) of 16 channels, or,
    // where the queries come undecayed and the walk's error is twice as large, 32 (fewer registers: 30 against 35 us)
    constexpr int HALF = CH ? 4 : DK / 16;
#pragma unroll 1
    for (int i = 0; i < CG; ++i) {
        f32x4 xs, ys;
#pragma unroll
        for (int s0 = 0; s0 < DK / 16; s0 += HALF) {
            f32x4 x[4], y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = y[e] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = s0; s < s0 + HALF; ++s) {
                const float4 q = *reinterpret_cast<const float4*>(Qs + (row0 + i * 16 + r) * LS + 16 * s + 4 * g);
                x[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[s].x, q.x, x[0], 0, 0, 0);
                y[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(sy[s].x, q.x, y[0], 0, 0, 0);
                x[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[s].y, q.y, x[1], 0, 0, 0);
                y[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(sy[s].y, q.y, y[1], 0, 0, 0);
                x[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[s].z, q.z, x[2], 0, 0, 0);
                y[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(sy[s].z, q.z, y[2], 0, 0, 0);
                x[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(sx[s].w, q.w, x[3], 0, 0, 0);
                y[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(sy[s].w, q.w, y[3], 0, 0, 0);
            }
            const f32x4 xh = (x[0] + x[1]) + (x[2] + x[3]), yh = (y[0] + y[1]) + (y[2] + y[3]);
            xs = s0 ? xs + xh : xh;
            ys = s0 ? ys + yh : yh;
        }
        const int t = row0 + i * 16 + r, col = col0 + 8 * g;
        if (t >= nt || col >= a.Dv) continue;
        float* p = a.out + ((size_t)(lo + t) * a.H + head) * a.Dv + col;
        if (a.Dv % 4 == 0 && col + 8 <= a.Dv) {
            float4 u = *reinterpret_cast<const float4*>(p), w = *reinterpret_cast<const float4*>(p + 4);
            u.x += xs[0]; u.y += xs[1]; u.z += xs[2]; u.w += xs[3];
            w.x += ys[0]; w.y += ys[1]; w.z += ys[2]; w.w += ys[3];
            *reinterpret_cast<float4*>(p) = u;
            *reinterpret_cast<float4*>(p + 4) = w;
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (col + e < a.Dv) p[e] += e < 4 ? xs[e] : ys[e - 4];
        }
    }
}

template <int DK, int MODE, typename TQ, typename TV>
static void launch_scan(const ScanArgs& a, int n_long, int slots, hipStream_t s) {
    hipLaunchKernelGGL((scan_chunks_kernel<DK, MODE, TQ, TV>), dim3(a.H, slots), dim3(64 * scan_waves(DK, MODE >= SCAN_CHANNEL)), 0, s, a);
    const int pieces = (a.D + 15) / 16 * scan_tiles(a.Dv) * 64;
    constexpr bool CH = MODE >= SCAN_CHANNEL;
    hipLaunchKernelGGL(scan_states_kernel<CH>, dim3((pieces + 255) / 256, a.H, n_long), dim3(256), 0, s, a, DK);
    if (a.Dv <= 32) hipLaunchKernelGGL((scan_apply_kernel<DK, 1, CH, TQ>), dim3(a.H, slots), dim3(256), 0, s, a);
    else if (a.Dv <= 64) hipLaunchKernelGGL((scan_apply_kernel<DK, 2, CH, TQ>), dim3(a.H, slots), dim3(256), 0, s, a);
    else hipLaunchKernelGGL((scan_apply_kernel<DK, 4, CH, TQ>), dim3(a.H * ((a.Dv + 127) / 128), slots), dim3(256), 0, s, a);
}

// One of the recurrences above over chunks first .. first + count - 1 (64 tokens each; a sequence may have fewer) of every
// sequence of `least` tokens and more, of which there are at most n_long, from and into the rows' states. D <= 128. adds,
// queries and factors: scratch of `slots` chunks, n_tokens / 64 + n_long of them with compact (first 0 and count for the
// longest sequence), n_long * count without.
// q and k are float32 with q_f32, else in dtype like v. dtype 0 float32, 1 bfloat16.
SOC_EXPORT int soc_scan(int mode, const void* q, long long ldq, int hq, const void* k, long long ldk, int hk, int group, int q_f32,
                        const void* v, long long ldv, int hv, int v_act, int ones, const float* decay, long long lda,
                        const float* p1, const float* p2, const float* p3, int H, int D, int Dv, float* state, long long stride,
                        int offset, const int* seq_qstart, const int* seq_rows, int n_seqs, int least, int n_long, int slots,
                        int first, int count, int compact, float* out, float* adds, float* queries, float* factors, int dtype,
                        hipStream_t stream) {
    if (n_seqs <= 0 || n_long <= 0 || H <= 0 || count <= 0) return 0;
    if (D < 1 || D > 128 || Dv < 1 || ones < 0 || ones >= Dv || group < 1 || H % group || n_long > 65535 || slots < n_long || slots > 65535 ||
        least < 1 || first < 0 || (compact && first) || (!compact && slots != (long long)n_long * count) || !adds || !queries || !factors || !decay) return (int)hipErrorInvalidValue;
    ScanArgs a;
    a.q = q; a.k = k; a.v = v; a.decay = decay; a.p1 = p1; a.p2 = p2; a.p3 = p3;
    a.ldq = ldq; a.ldk = ldk; a.ldv = ldv; a.lda = lda; a.hq = hq; a.hk = hk; a.hv = hv; a.group = group;
    a.H = H; a.D = D; a.Dv = Dv; a.held = Dv - ones; a.v_act = v_act;
    a.first = first; a.count = count; a.compact = compact; a.n_seqs = n_seqs; a.least = least; a.qstart = seq_qstart; a.rows = seq_rows;
    a.state = state; a.stride = stride; a.offset = offset; a.out = out; a.adds = adds; a.queries = queries; a.factors = factors;
    const int qe = q_f32 || dtype == 0 ? 16 : 8, ve = dtype == 0 ? 16 : 8;       // bytes of four elements
    a.vec = D % 4 == 0 && a.held % 4 == 0 && ldq % 4 == 0 && ldk % 4 == 0 && ldv % 4 == 0 && lda % 4 == 0 && hq % 4 == 0 && hk % 4 == 0 && hv % 4 == 0 &&
            (uintptr_t)q % qe == 0 && (uintptr_t)k % qe == 0 && (uintptr_t)v % ve == 0 && (uintptr_t)decay % 16 == 0;
#define SOC_SCAN(MODE_, TQ_, TV_) \
    do { if (D <= 64) launch_scan<64, MODE_, TQ_, TV_>(a, n_long, slots, stream); else launch_scan<128, MODE_, TQ_, TV_>(a, n_long, slots, stream); } while (0)
    if (mode == SCAN_HEAD && q_f32) { if (dtype == 0) SOC_SCAN(SCAN_HEAD, float, float); else SOC_SCAN(SCAN_HEAD, float, bf16); }
    else if (mode == SCAN_CHANNEL && q_f32) { if (dtype == 0) SOC_SCAN(SCAN_CHANNEL, float, float); else SOC_SCAN(SCAN_CHANNEL, float, bf16); }
    else if (mode == SCAN_STEP && !q_f32 && p1 && p2 && p3) { if (dtype == 0) SOC_SCAN(SCAN_STEP, float, float); else SOC_SCAN(SCAN_STEP, bf16, bf16); }
    else if (mode == SCAN_BONUS && !q_f32 && p1) { if (dtype == 0) SOC_SCAN(SCAN_BONUS, float, float); else SOC_SCAN(SCAN_BONUS, bf16, bf16); }
    else return (int)hipErrorInvalidValue;
#undef SOC_SCAN
    return soc_last_error();
}

// ---- the gated delta rule in chunks ---------------------------------------------------------------------------------
// S <- g S; u = beta (v - S^T k); S <- S + k u^T; o = S^T q. With the chunk's start state S0, the decays D_ij from
// behind token j to token i and the decay G_i from the start to i, the u of a chunk solve a triangular system,
//   (I + M) U = diag(beta) (V - diag(G) K S0),   M_ij = beta_i D_ij k_i . k_j for j < i,
// and with T = (I + M)^-1 (by blocks of 16), A_ij = D_ij q_i . k_j for j <= i, X = A T diag(beta) and
// Z = diag(beta) T^T (keys decayed to the chunk's end):
//   O  = X V + (queries decayed to the start - X diag(G) K) S0          the bracket goes where scan_apply reads it
//   S' = (G_end I - Z^T diag(G) K) S0 + Z^T V                           the bracket is the chunk's transition
// so everything but S0's share is the chunk's own, and what is left to do in order is one product per chunk.
// gates float32 [N, H, 2] = (g, beta); the state of a row is [H, Dv, D].
struct DeltaArgs {
    const float *q, *k, *gates;
    const void* v;
    long long ldq, ldv;
    int hq, hv, group, H, D, Dv, vec, first, count, compact, n_seqs, least;
    const int* qstart;
    const int* rows;
    float* state;
    long long stride;
    int offset;
    float *out, *adds, *queries, *moves;      // moves: per slot and head [DK, DK] in tiles
};

template <int DK, typename TV>
__global__ void __launch_bounds__(64 * scan_waves(DK, true))
delta_chunks_kernel(DeltaArgs a) {
    constexpr int LS = DK + 4, Q4 = DK / 4, NW = scan_waves(DK, true), NT = 64 * NW;
    __shared__ __align__(16) float Qs[SCAN_C * LS];                  // later Z
    __shared__ __align__(16) float Ks[SCAN_C * LS];
    __shared__ __align__(16) float As[SCAN_C * SCAN_AS], Ms[SCAN_C * SCAN_AS], Ts[SCAN_C * SCAN_AS];     // Ms later X
    __shared__ __align__(16) float Vs[SCAN_C * SCAN_VS];
    __shared__ __align__(16) float dg[4][16][16];
    __shared__ float sa[SCAN_C], sb[SCAN_C], from[SCAN_C], rest[SCAN_C];
    __shared__ double pin[SCAN_C], sfx[SCAN_C], tot[4];
    __shared__ int broken;                           // the first token whose key, decay or step size is not finite
    const int head = blockIdx.x, tid = threadIdx.x;
    ScanPlace at;
    if (!scan_chunk(a, blockIdx.y, at)) return;
    const int lo = a.qstart[at.seq] + (a.first + at.c) * SCAN_C, hi = a.qstart[at.seq + 1];
    if (lo >= hi) return;
    const int nt = min(SCAN_C, hi - lo);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    const size_t slot = (size_t)at.slot * a.H + head;

    const float* q = a.q + (size_t)(head / a.group) * a.hq + (size_t)lo * a.ldq;
    const float* k = a.k + (size_t)(head / a.group) * a.hq + (size_t)lo * a.ldq;
    if (tid == 0) broken = SCAN_C;
    constexpr int ROUNDS = SCAN_C * Q4 / NT;
    float4 fq[ROUNDS], fk[ROUNDS];
#pragma unroll
    for (int it = 0; it < ROUNDS; ++it) {            // (q and k are padded with zeros to DK; all loads before the first use)
        const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4;
        fq[it] = scan_quad(q + (size_t)t * a.ldq + i, q, t < nt ? 4 : 0, 1);
        fk[it] = scan_quad(k + (size_t)t * a.ldq + i, k, t < nt ? 4 : 0, 1);
    }
    if (tid < SCAN_C) {
        const float2 gb = reinterpret_cast<const float2*>(a.gates)[(size_t)(lo + min(tid, nt - 1)) * a.H + head];
        sa[tid] = tid < nt ? gb.x : 1.f;
        sb[tid] = tid < nt ? gb.y : 0.f;
    }
    lds_barrier();
    if (tid < nt && !(sa[tid] * 0.f + sb[tid] * 0.f == 0.f)) atomicMin(&broken, tid);
#pragma unroll
    for (int it = 0; it < ROUNDS; ++it) {
        const int e = it * NT + tid, t = e / Q4, i = e % Q4 * 4;
        *reinterpret_cast<float4*>(Qs + t * LS + i) = fq[it];
        *reinterpret_cast<float4*>(Ks + t * LS + i) = fk[it];
        if (!(fk[it].x * 0.f + fk[it].y * 0.f + fk[it].z * 0.f + fk[it].w * 0.f == 0.f)) atomicMin(&broken, t);
    }
    __syncthreads();
    // From such a token on nothing of the head is finite, neither results nor state; the tokens before it do not see it. The
    // chunk is computed as if it ended there, and NaN put where the later results and the state are made (its queries' rows
    // and the diagonal of its transition).
    const int sound = broken;
    if (sound < SCAN_C) {
        for (int e = sound * LS + tid; e < SCAN_C * LS; e += NT) Qs[e] = Ks[e] = 0.f;
        if (tid < SCAN_C && tid >= sound) { sa[tid] = 1.f; sb[tid] = 0.f; }
        __syncthreads();
    }
    if (tid < SCAN_C) {
        const int I = tid / 16, j = tid % 16;
        double p = 1.0;
        for (int i = 0; i < 16; ++i) {
            if (i > j) p *= sa[I * 16 + i];
            dg[I][i][j] = i >= j ? (float)p : 0.f;
        }
        sfx[tid] = p;
    } else if (tid < 2 * SCAN_C) {
        const int i = tid - SCAN_C, I = i / 16;
        double p = 1.0;
        for (int t = I * 16; t <= i; ++t) p *= sa[t];
        pin[i] = p;
        if (i % 16 == 15) tot[I] = p;
    }
    // A and M: twenty blocks of 16 x 16
    constexpr int MINE = (20 + NW - 1) / NW;
    f64x4 sc[MINE];
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
        const int b = wave + NW * x, bb = b % 10;
        if (b >= 20) continue;
        const int I = bb < 1 ? 0 : bb < 3 ? 1 : bb < 6 ? 2 : 3, J = bb - I * (I + 1) / 2;
        const float* rows = b < 10 ? Qs : Ks;
        f64x4 s = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int m = 0; m < DK; m += 16) {
            const float4 qf = *reinterpret_cast<const float4*>(rows + (I * 16 + r) * LS + m + 4 * g);
            const float4 kf = *reinterpret_cast<const float4*>(Ks + (J * 16 + r % 4 * 4 + r / 4) * LS + m + 4 * g);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kf.x, (double)qf.x, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kf.y, (double)qf.y, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kf.z, (double)qf.z, s, 0, 0, 0);
            s = __builtin_amdgcn_mfma_f64_16x16x4f64((double)kf.w, (double)qf.w, s, 0, 0, 0);
        }
        sc[x] = s;
    }
    lds_barrier();
    if (tid < SCAN_C) {
        double p = pin[tid], s = sfx[tid];
        for (int run = 0; run < tid / 16; ++run) p *= tot[run];
        for (int run = tid / 16 + 1; run < 4; ++run) s *= tot[run];
        from[tid] = (float)p;
        rest[tid] = (float)s;
    }
#pragma unroll
    for (int x = 0; x < MINE; ++x) {
        const int b = wave + NW * x, bb = b % 10;
        if (b >= 20) continue;
        const int I = bb < 1 ? 0 : bb < 3 ? 1 : bb < 6 ? 2 : 3, J = bb - I * (I + 1) / 2, i = I * 16 + r;
        double f[4], p = pin[i];
        for (int run = J + 1; run < I; ++run) p *= tot[run];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[e] = I == J ? (double)dg[I][r][4 * g + e] : p * sfx[J * 16 + 4 * g + e];
            if (b >= 10) f[e] = I == J && 4 * g + e >= r ? 0.0 : f[e] * sb[i];
        }
        *reinterpret_cast<float4*>((b < 10 ? As : Ms) + i * SCAN_AS + J * 16 + 4 * g) =
            make_float4((float)(sc[x][0] * f[0]), (float)(sc[x][1] * f[1]), (float)(sc[x][2] * f[2]), (float)(sc[x][3] * f[3]));
    }
    lds_barrier();
    // T, the diagonal blocks by substitution, a thread per column
    if (tid < SCAN_C) {
        const int I = tid / 16, col = tid % 16;
        const float* m = Ms + I * 16 * SCAN_AS + I * 16;
        float x[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            float s = i == col ? 1.f : 0.f;
#pragma unroll
            for (int j = 0; j < i; ++j) s = fmaf(-m[i * SCAN_AS + j], x[j], s);
            x[i] = s;
            Ts[(I * 16 + i) * SCAN_AS + I * 16 + col] = s;
        }
    }
    lds_barrier();
    // below them T_IJ = -T_II sum_m M_Im T_mJ, one diagonal after the other
    for (int d = 1; d < 4; ++d) {
        if (wave < 4 - d) {
            const int J = wave, I = wave + d;
            float* mid = Vs + wave * 16 * 20;
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
            for (int m = J; m < I; ++m)
                x = mfma_col_row(Ts + (m * 16 + 4 * g) * SCAN_AS + J * 16 + r, SCAN_AS, Ms + (I * 16 + r) * SCAN_AS + m * 16 + 4 * g, x);
            *reinterpret_cast<float4*>(mid + r * 20 + 4 * g) = make_float4(x[0], x[1], x[2], x[3]);
            __builtin_amdgcn_wave_barrier();
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            x = (f32x4){0.f, 0.f, 0.f, 0.f};
            x = mfma_col_row(mid + 4 * g * 20 + r, 20, Ts + (I * 16 + r) * SCAN_AS + I * 16 + 4 * g, x);
            *reinterpret_cast<float4*>(Ts + (I * 16 + r) * SCAN_AS + J * 16 + 4 * g) = make_float4(-x[0], -x[1], -x[2], -x[3]);
        }
        lds_barrier();
    }
    // X = A T diag(beta), over M
#pragma unroll
    for (int x = 0; x < (10 + NW - 1) / NW; ++x) {
        const int b = wave + NW * x;
        if (b >= 10) continue;
        const int I = b < 1 ? 0 : b < 3 ? 1 : b < 6 ? 2 : 3, J = b - I * (I + 1) / 2;
        f32x4 s = {0.f, 0.f, 0.f, 0.f};
        for (int m = J; m <= I; ++m)
            s = mfma_col_row(Ts + (m * 16 + 4 * g) * SCAN_AS + J * 16 + r, SCAN_AS, As + (I * 16 + r) * SCAN_AS + m * 16 + 4 * g, s);
        const float* be = sb + J * 16 + 4 * g;
        *reinterpret_cast<float4*>(Ms + (I * 16 + r) * SCAN_AS + J * 16 + 4 * g) = make_float4(s[0] * be[0], s[1] * be[1], s[2] * be[2], s[3] * be[3]);
    }
    lds_barrier();
    constexpr int PER = NW * 16 / DK;                // waves that share 16 channels: two
    static_assert(PER == 2, "rows and columns are shared out by halves");
    const int ct = wave / PER, part = wave % PER;
    f32x4 z[4 / PER];
    // queries decayed to the start - X diag(G) K; Z
#pragma unroll
    for (int y = 0; y < 4 / PER; ++y) {
        const int I = 2 * y + part;
        const int i = I * 16 + r;
        const float4 q4 = *reinterpret_cast<const float4*>(Qs + i * LS + ct * 16 + 4 * g);
        f32x4 o = {q4.x * from[i], q4.y * from[i], q4.z * from[i], q4.w * from[i]};
        for (int s = 0; s <= I; ++s) {
            const int j = 16 * s + 4 * g;
            const float* col = Ks + j * LS + ct * 16 + r;
            o += mfma4(-from[j] * col[0], -from[j + 1] * col[LS], -from[j + 2] * col[2 * LS], -from[j + 3] * col[3 * LS],
                       *reinterpret_cast<const float4*>(Ms + i * SCAN_AS + j), (f32x4){0.f, 0.f, 0.f, 0.f});
        }
        if (i >= sound) o[0] = o[1] = o[2] = o[3] = NAN;
        *reinterpret_cast<float4*>(a.queries + (slot * SCAN_C + i) * DK + ct * 16 + 4 * g) = make_float4(o[0], o[1], o[2], o[3]);
        f32x4 w = {0.f, 0.f, 0.f, 0.f};
        for (int s = I; s < 4; ++s) {                // row I * 16 + r of T^T
            const int t = 16 * s + 4 * g;
            const float* col = Ks + t * LS + ct * 16 + r;
            const float* tt = Ts + t * SCAN_AS + I * 16 + r;
            w += mfma4(rest[t] * col[0], rest[t + 1] * col[LS], rest[t + 2] * col[2 * LS], rest[t + 3] * col[3 * LS],
                       make_float4(tt[0], tt[SCAN_AS], tt[2 * SCAN_AS], tt[3 * SCAN_AS]), (f32x4){0.f, 0.f, 0.f, 0.f});
        }
        const float be = sb[i];
        z[y] = (f32x4){w[0] * be, w[1] * be, w[2] * be, w[3] * be};
    }
    lds_barrier();
#pragma unroll
    for (int y = 0; y < 4 / PER; ++y) {
        const int I = 2 * y + part;
        *reinterpret_cast<float4*>(Qs + (I * 16 + r) * LS + ct * 16 + 4 * g) = make_float4(z[y][0], z[y][1], z[y][2], z[y][3]);
    }
    // the values' first columns are on their way while the transition is formed
    const TV* v = (const TV*)a.v + (size_t)head * a.hv + (size_t)lo * a.ldv;
    const int vt = tid / 8, vc = tid % 8 * 4;
    auto fetch = [&](int col) { return scan_quad(v + (size_t)vt * a.ldv + col, v, vt < nt ? a.Dv - col : 0, a.vec); };
    float4 next = fetch(vc);
    lds_barrier();
    const float whole = sound < SCAN_C ? NAN : (float)(tot[0] * tot[1] * tot[2] * tot[3]);
#pragma unroll
    for (int y0 = 0; y0 < DK / 16 / PER; y0 += 4 / PER) {
        f32x4 s[4 / PER];
#pragma unroll
        for (int y = 0; y < 4 / PER; ++y) s[y] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int m = 0; m < SCAN_C; m += 16)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = m + 4 * g + e;
                const float x = Qs[t * LS + ct * 16 + r], ge = from[t];
#pragma unroll
                for (int y = 0; y < 4 / PER; ++y) {
                    const int c2 = ((y0 + y) * PER + part) * 16 + r;
                    s[y] = __builtin_amdgcn_mfma_f32_16x16x4f32(Ks[t * LS + c2] * ge, x, s[y], 0, 0, 0);
                }
            }
        const int row = ct * 16 + r;
#pragma unroll
        for (int y = 0; y < 4 / PER; ++y) {
            const int c2 = ((y0 + y) * PER + part) * 16 + 4 * g;
            float4 w = make_float4(-s[y][0], -s[y][1], -s[y][2], -s[y][3]);
            if (row == c2) w.x += whole;
            if (row == c2 + 1) w.y += whole;
            if (row == c2 + 2) w.z += whole;
            if (row == c2 + 3) w.w += whole;
            *reinterpret_cast<float4*>(a.moves + slot * DK * DK + ((size_t)(ct * (DK / 16) + (y0 + y) * PER + part) * 64 + lane) * 4) = w;
        }
    }
    const bool by4 = a.Dv % 4 == 0;
    const int tiles = scan_tiles(a.Dv);
    float* adds = a.adds + slot * ((a.D + 15) / 16) * tiles * 256;
    for (int col0 = 0; col0 < a.Dv; col0 += SCAN_VC) {
        lds_barrier();
        if (NT == 512 || tid < 512) *reinterpret_cast<float4*>(Vs + vt * SCAN_VS + vc) = next;
        lds_barrier();
        if (col0 + SCAN_VC < a.Dv) next = fetch(col0 + SCAN_VC + vc);
        scan_values<DK, NW>(a.out, a.H, a.Dv, by4, lo, nt, head, col0, tiles, Qs, Vs, Ms, adds, (a.D + 15) / 16, wave, r, g);
    }
}

// The states in order: a workgroup owns 16 columns of a head's state, transposed in LDS; per chunk its old value goes
// where the addend was (scan_apply reads it there) and S <- (transition) S + addend. The next chunk's transition and
// addend are on their way meanwhile. Workgroups of one head follow each other on one XCD, whose L2 then serves
// the transitions that they all read.
template <int DK>
__global__ void __launch_bounds__(256)
delta_states_kernel(DeltaArgs a, int blocks) {
    constexpr int LS = DK + 4, TILES = DK / 64;       // tiles of 16 channels per wave
    __shared__ __align__(16) float St[2][16][LS];
    const int b = blockIdx.x, head = b / (8 * blocks) * 8 + b % 8, cb = b / 8 % blocks, tid = threadIdx.x;
    ScanPlace at;
    if (head >= a.H || !scan_sequence(a, blockIdx.y, at)) return;
    const int seq = at.seq;
    const int left = a.qstart[seq + 1] - a.qstart[seq] - a.first * SCAN_C;
    if (left <= 0) return;
    const int n = min(a.count, (left + SCAN_C - 1) / SCAN_C);
    const int lane = tid % 64, wave = tid / 64, r = lane % 16, g = lane / 16;
    float* S = a.state + (size_t)a.rows[seq] * a.stride + a.offset + (size_t)head * a.Dv * a.D;
    const size_t slot0 = (size_t)at.slot * a.H + head;
    for (int e = tid; e < 16 * DK; e += 256) {
        const int cl = e / DK, ch = e % DK, col = cb / 2 * 32 + scan_col(cb % 2, cl);
        St[0][cl][ch] = col < a.Dv && ch < a.D ? S[(size_t)col * a.D + ch] : 0.f;
    }
    const int tiles = scan_tiles(a.Dv), ch_tiles = (a.D + 15) / 16;
    struct Next { float4 m[TILES][DK / 16], x[TILES]; } even, odd;
    float4* adds = reinterpret_cast<float4*>(a.adds) + lane;
    auto place = [&](int c, int t) { return (((slot0 + (size_t)c * a.H) * ch_tiles + min(wave * TILES + t, ch_tiles - 1)) * tiles + cb) * 64; };
    auto fetch = [&](int c, Next& to) {
        const float4* m = reinterpret_cast<const float4*>(a.moves) + (slot0 + (size_t)c * a.H) * (DK * DK / 4) + lane;
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
#pragma unroll
            for (int s = 0; s < DK / 16; ++s) to.m[t][s] = m[((wave * TILES + t) * (DK / 16) + s) * 64];
            to.x[t] = adds[place(c, t)];
        }
    };
    fetch(0, even);
    lds_barrier();
    float4 old[TILES];
#pragma unroll
    for (int t = 0; t < TILES; ++t) old[t] = *reinterpret_cast<const float4*>(&St[0][r][(wave * TILES + t) * 16 + 4 * g]);
    auto move = [&](int c, int from, Next& now, Next& then) {
        if (c + 1 < n) fetch(c + 1, then);
        f32x4 part[TILES][4], s[TILES];                 // (a sum in four parts: see sum_pairs)
#pragma unroll
        for (int t = 0; t < TILES; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[t][e] = (f32x4){0.f, 0.f, 0.f, 0.f};
        float4 y[DK / 16];
#pragma unroll
        for (int k = 0; k < DK / 16; ++k) y[k] = *reinterpret_cast<const float4*>(&St[from][r][16 * k + 4 * g]);
#pragma unroll
        for (int k = 0; k < DK / 16; ++k)
#pragma unroll
            for (int t = 0; t < TILES; ++t) {
                part[t][0] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.m[t][k].x, y[k].x, part[t][0], 0, 0, 0);
                part[t][1] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.m[t][k].y, y[k].y, part[t][1], 0, 0, 0);
                part[t][2] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.m[t][k].z, y[k].z, part[t][2], 0, 0, 0);
                part[t][3] = __builtin_amdgcn_mfma_f32_16x16x4f32(now.m[t][k].w, y[k].w, part[t][3], 0, 0, 0);
            }
#pragma unroll
        for (int t = 0; t < TILES; ++t)
            s[t] = (part[t][0] + part[t][1]) + (part[t][2] + part[t][3]) + (f32x4){now.x[t].x, now.x[t].y, now.x[t].z, now.x[t].w};
#pragma unroll
        for (int t = 0; t < TILES; ++t) {
            if (wave * TILES + t < ch_tiles) adds[place(c, t)] = old[t];
            old[t] = wave * TILES + t < ch_tiles ? make_float4(s[t][0], s[t][1], s[t][2], s[t][3]) : make_float4(0.f, 0.f, 0.f, 0.f);
            *reinterpret_cast<float4*>(&St[from ^ 1][r][(wave * TILES + t) * 16 + 4 * g]) = old[t];
        }
        lds_barrier();
    };
    for (int c = 0; c < n; c += 2) {
        move(c, 0, even, odd);
        if (c + 1 < n) move(c + 1, 1, odd, even);
    }
    for (int e = tid; e < 16 * DK; e += 256) {
        const int cl = e / DK, ch = e % DK, col = cb / 2 * 32 + scan_col(cb % 2, cl);
        if (col < a.Dv && ch < a.D) S[(size_t)col * a.D + ch] = St[n % 2][cl][ch];
    }
}

template <int DK>
static void launch_delta(const DeltaArgs& a, int n_long, int slots, int dtype, hipStream_t s) {
    if (dtype == 0) hipLaunchKernelGGL((delta_chunks_kernel<DK, float>), dim3(a.H, slots), dim3(64 * scan_waves(DK, true)), 0, s, a);
    else hipLaunchKernelGGL((delta_chunks_kernel<DK, bf16>), dim3(a.H, slots), dim3(64 * scan_waves(DK, true)), 0, s, a);
    const int blocks = scan_tiles(a.Dv);
    hipLaunchKernelGGL((delta_states_kernel<DK>), dim3((a.H + 7) / 8 * 8 * blocks, n_long), dim3(256), 0, s, a, blocks);
    ScanArgs b = {};
    b.H = a.H; b.D = a.D; b.Dv = a.Dv; b.first = a.first; b.count = a.count; b.compact = a.compact; b.n_seqs = a.n_seqs; b.least = a.least;
    b.qstart = a.qstart;
    b.out = a.out; b.adds = a.adds; b.queries = a.queries;
    if (a.Dv <= 32) hipLaunchKernelGGL((scan_apply_kernel<DK, 1, true, float>), dim3(a.H, slots), dim3(256), 0, s, b);
    else if (a.Dv <= 64) hipLaunchKernelGGL((scan_apply_kernel<DK, 2, true, float>), dim3(a.H, slots), dim3(256), 0, s, b);
    else hipLaunchKernelGGL((scan_apply_kernel<DK, 4, true, float>), dim3(a.H * ((a.Dv + 127) / 128), slots), dim3(256), 0, s, b);
}

// The gated delta rule over chunks first .. first + count - 1 of every sequence of `least` tokens and more, from and into the
// rows' states. qk float32 [N, 2, G, Dp] as soc_delta_prepare leaves it, Dp 64 or 128; v [N, H Dv] in dtype. n_long and
// scratch as for soc_scan, queries
// [slots, H, 64, Dp], moves [slots, H, Dp, Dp].
SOC_EXPORT int soc_delta_scan(const float* qk, const void* v, const float* gates, int G, int H, int D, int Dv, int Dp, float* state,
                              long long stride, int offset, const int* seq_qstart, const int* seq_rows, int n_seqs, int least, int n_long,
                              int slots, int first, int count, int compact, float* out, float* adds, float* queries, float* moves, int dtype, hipStream_t stream) {
    if (n_seqs <= 0 || n_long <= 0 || H <= 0 || count <= 0) return 0;
    if (G < 1 || H % G || D < 1 || Dv < 1 || Dp != (D + 63) / 64 * 64 || Dp > 128 || n_long > 65535 || slots < n_long || slots > 65535 ||
        least < 1 || first < 0 || (compact && first) || (!compact && slots != (long long)n_long * count) || !adds || !queries || !moves)
        return (int)hipErrorInvalidValue;
    DeltaArgs a;
    a.q = qk; a.k = qk + (size_t)G * Dp; a.gates = gates; a.v = v; a.ldq = 2ll * G * Dp; a.ldv = (long long)H * Dv;
    a.hq = Dp; a.hv = Dv; a.group = H / G; a.H = H; a.D = D; a.Dv = Dv;
    a.vec = Dv % 4 == 0 && (uintptr_t)v % (dtype == 0 ? 16 : 8) == 0;
    a.first = first; a.count = count; a.compact = compact; a.n_seqs = n_seqs; a.least = least; a.qstart = seq_qstart; a.rows = seq_rows;
    a.state = state; a.stride = stride; a.offset = offset; a.out = out; a.adds = adds; a.queries = queries; a.moves = moves;
    if (Dp == 64) launch_delta<64>(a, n_long, slots, dtype, stream); else launch_delta<128>(a, n_long, slots, dtype, stream);
    return soc_last_error();
}
