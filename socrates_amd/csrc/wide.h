// Products of many rows on the bfloat16 matrix cores: the loop that a workgroup's tile goes through, and its results.
//
// A workgroup of four waves (2 x 2, one per SIMD) owns 32 MI rows of x and 32 NJ weight rows; a wave multiplies MI x NJ blocks
// of 16 x 16, whose sums stay in its registers (up to 256 of them). 64 k make a step: its rows of x and weights lie in rings
// of RX and RW buffers in LDS that global_load_lds fills, 128 bytes of a row at a time (64 bytes a row and step took the L2
// a quarter longer). A wave holds the operands of half a step in registers while it reads those of the next half, so that
//  * the LDS reads, the loads and the products of a half are issued in turn, evenly: reads in a bunch, or all loads at once,
//    cost 5 to 15 %, since one wave per SIMD issues in order;
//  * a step's buffers are free at the middle of the step, where the only barrier of the step stands.
// Weights are the first operand: a lane ends up with four neighbouring outputs of one row.
// 128 x 128 a wave read LDS for half of the products' time, with writes three quarters (128 x 64: all of it), which is why
// four waves of 256 sums do better than eight of 128. Measured against the library, random data, us (PFLOP/s):
// 2,048 x 8,192 x 4,096 90.4 (1.52) against 88.4; 2,048 x 19,456 x 2,560 160 (1.27) against 176; the card's power holds
// both back (zeros: 72 against 68).
#pragma once

#include "mfma.h"

// LDS in pieces of 4 KB (32 rows of 64 k): 40 of them. The rings are chosen for the number of loads that may still be on their
// way where step s + 1 has to be there: those asked for after its rows of x, and after its weights.
constexpr int wide_newer(int mi, int nj, int rx, int rw) {
    const int x = (rx - 1) * nj + (rx - 2) * mi, w = (rw - 2) * (mi + nj);
    return x < w ? x : w;
}
constexpr int wide_rings(int mi, int nj) {                   // 10 RX + RW
    int best = 22;
    for (int rx = 2; rx <= 5; ++rx)
        for (int rw = 2; rw <= 5; ++rw)
            if (rx * mi + rw * nj <= 40 && wide_newer(mi, nj, rx, rw) > wide_newer(mi, nj, best / 10, best % 10)) best = 10 * rx + rw;
    return best;
}
template <int MI, int NJ> struct WideRings {
    static constexpr int RX = wide_rings(MI, NJ) / 10, RW = wide_rings(MI, NJ) % 10, NEWER = wide_newer(MI, NJ, RX, RW);
    static_assert(RX * MI + RW * NJ <= 40 && NEWER > 0 && NEWER + MI <= 63, "160 KB of LDS, and what the counter of loads holds");
};

// Sixteen bytes per lane from base + off (bytes) to the wave's 1 KB at lds + 16 lane. m0 holds the LDS address.
__device__ __forceinline__ void wide_load(uint32_t lds, uint32_t off, const char* base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "m0");
}

// c += a b on the matrix cores, the sums in the accumulation registers they are in: through the builtin the compiler gave some of
// them new homes in every step (28 moves, each behind the product it waits for: 2,048 x 6,144 x 2,560 took 92 us, not 57).
// It does not look into the instruction for the wait states a vector instruction needs behind it: wide_fence comes before
// the sums are read.
__device__ __forceinline__ void wide_product(f32x4_t& c, bf16x8_t a, bf16x8_t b) {
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void wide_fence() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// The eight pieces of 16 bytes of a row's 64 k are swapped among themselves by a pattern over the rows, so that the 16 rows of
// one k are read without bank conflicts.
__device__ __forceinline__ int wide_swap(int row) { return (row >> 1) & 7; }

template <int H> struct WideHalf { static constexpr int value = H; };

// xo[i], wo[i]: byte offsets of this lane's piece of row (wave MI + i) 8 + lane / 8 (wave NJ + i ... of the weights) at k 0: piece
// (lane % 8) ^ wide_swap(row), of any row that exists for a row outside. steps: K / 64, at least one. acc[i][j] comes back with
// row (2 i + wave / 2) 16 + lane % 16 of x and weight rows (wave % 2 NJ + j) 16 + 4 (lane / 16) + r. All loads have landed.
template <int MI, int NJ>
__device__ __forceinline__ void wide_walk(const char* x, const char* w, const uint32_t (&xo)[MI], const uint32_t (&wo)[NJ], int steps,
                                          uint16_t* lds, f32x4_t (&acc)[MI][NJ]) {
    using Rings = WideRings<MI, NJ>;
    constexpr int RX = Rings::RX, RW = Rings::RW, XS = MI * 2048, WS = NJ * 2048;      // elements of one buffer
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), li = lane % 16, g = lane / 16;
    const int wm = wave / 2, wn = wave % 2;
    const uint32_t base = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint16_t*)lds;
    const uint32_t xl = base + wave * MI * 1024, wl = base + RX * XS * 2 + wave * NJ * 1024;
    uint16_t* const wlds = lds + RX * XS;
    // (past the end the last step is asked for again: what the counter of loads waits for is the same in every step)
    auto load_x = [&](int s, int slot, int i) {
        wide_load(__builtin_amdgcn_readfirstlane(xl + slot * XS * 2 + i * 1024), xo[i], x + (size_t)min(s, steps - 1) * 128);
    };
    auto load_w = [&](int s, int slot, int i) {
        wide_load(__builtin_amdgcn_readfirstlane(wl + slot * WS * 2 + i * 1024), wo[i], w + (size_t)min(s, steps - 1) * 128);
    };
    int at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) at[h] = li * 64 + ((4 * h + g) ^ wide_swap(li)) * 8;
    bf16x8_t a[2][MI], b[2][NJ];
    auto read = [&](int h, const uint16_t* xs, const uint16_t* ws, int r) {            // r-th of MI + NJ: rows and weights in turn
        constexpr int BOTH = 2 * (MI < NJ ? MI : NJ);
        const bool of_x = r < BOTH ? r % 2 == 0 : MI > NJ;
        const int n = r < BOTH ? r / 2 : r - BOTH / 2;
        if (of_x) a[h][n] = *reinterpret_cast<const bf16x8_t*>(&xs[(2 * n + wm) * 1024 + at[h]]);
        else b[h][n] = *reinterpret_cast<const bf16x8_t*>(&ws[(wn * NJ + n) * 1024 + at[h]]);
    };
    // one half: its products, the reads of the next half and one operand's loads of a later step
    auto half = [&](auto second, const uint16_t* xs, const uint16_t* ws, int s, int slot) {
        constexpr int H = decltype(second)::value, T = MI * NJ, R = MI + NJ, L = H ? MI : NJ;
        constexpr int SPAN = T - 3;                          // the last reads come three products before the end
        constexpr int LATER = T / L >= 4 ? 2 : 0;
        static_assert(R <= SPAN && L <= T, "one read and one load before a product");
#pragma unroll
        for (int n = 0; n < T; ++n) {
            // which read (and which load, between two reads) comes before product n
            const int r = (n * R + SPAN - 1) / SPAN, m = n - LATER, l = (m * L + T - 1) / T;
            const bool reads = r < R && (r * SPAN) / R == n, loads = m >= 0 && l < L && (l * T) / L == m;
            if (reads || loads) __builtin_amdgcn_sched_barrier(0);
            if (reads) read(1 - H, xs, ws, r);
            if (loads) {
                if (H) load_x(s, slot, l);
                else load_w(s, slot, l);
            }
            const int i = n / NJ, j = n % NJ;
            wide_product(acc[i][j], b[H][j], a[H][i]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // in the order that the loop would have asked for them
#pragma unroll
    for (int s = -(RX > RW ? RX : RW); s < 0; ++s) {
        if (s + RW - 1 >= 0) {
#pragma unroll
            for (int i = 0; i < NJ; ++i) load_w(s + RW - 1, s + RW - 1, i);
        }
        if (s + RX >= 0) {
#pragma unroll
            for (int i = 0; i < MI; ++i) load_x(s + RX, s + RX, i);
        }
    }
    __builtin_amdgcn_sched_barrier(0);                       // (while they are on their way)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) acc[i][j] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(Rings::NEWER + MI) : "memory");
#pragma unroll
    for (int r = 0; r < MI + NJ; ++r) read(0, lds, wlds, r);
    int sx = 0, sw = 0;                                      // slots of step s
    for (int s = 0; s < steps; ++s) {
        const int sx1 = sx + 1 == RX ? 0 : sx + 1, sw1 = sw + 1 == RW ? 0 : sw + 1, free_w = sw == 0 ? RW - 1 : sw - 1;
        half(WideHalf<0>{}, lds + sx * XS, wlds + sw * WS, s + RW - 1, free_w);       // (the weights of step s - 1 are read)
        // this wave has read step s, and its pieces of step s + 1 have landed; behind the barrier so have everyone's
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(Rings::NEWER) : "memory");
        half(WideHalf<1>{}, lds + sx1 * XS, wlds + sw1 * WS, s + RX, sx);
        sx = sx1;
        sw = sw1;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    wide_fence();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) asm volatile("" : "+a"(acc[i][j]));      // (read behind the fence)
}

// Halves of two blocks' rows change places between lanes 16 apart: out of four neighbouring outputs of block 0 and of block 1
// (packed, u and v) become eight neighbouring ones, of block g % 2 from element 8 (g / 2) on, where g = lane / 16.
__device__ __forceinline__ uint4 wide_eight(uint2 u, uint2 v) {
    const soc_u32x2 p = __builtin_amdgcn_permlane16_swap(u.x, v.x, false, false), q = __builtin_amdgcn_permlane16_swap(u.y, v.y, false, false);
    return make_uint4(p.x, q.x, p.y, q.y);
}

__device__ __forceinline__ float wide_rounded(float v) { return to_float(from_float<bf16>(v)); }

// 1 / (1 + e^-v) by the hardware's power of two and reciprocal, one unit in the last place each, beside an exponent that is off
// by |v| 2^-24 at most: a wave's 16,384 results are computed where nothing else runs, and the division alone is ten instructions.
// What follows is rounded to 8 bits.
__device__ __forceinline__ float wide_sigmoid(float v) {
    return __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-1.4426950408889634f * v));
}

// What becomes of a gate and an up product (both rounded to bfloat16, as they were where they went through memory), or of one.
enum { WIDE_PLAIN = 0, WIDE_SILU = 1, WIDE_GATED = 2, WIDE_GELU = 3, WIDE_SQUARED = 4 };
struct WideGate { float limit, slope, shift; };              // of WIDE_GATED
constexpr bool wide_pairs(int act) { return act == WIDE_SILU || act == WIDE_GATED || act == WIDE_GELU; }

template <int ACT> __device__ __forceinline__ float wide_act(float gate, float up, WideGate k) {
    if constexpr (ACT == WIDE_SQUARED) {
        const float y = fmaxf(gate, 0.f);
        return y * y;
    } else if constexpr (wide_pairs(ACT)) {
        gate = wide_rounded(gate);
        up = wide_rounded(up);
        if constexpr (ACT == WIDE_SILU) return gate * wide_sigmoid(gate) * up;
        if constexpr (ACT == WIDE_GELU)                       // (1 + tanh z) / 2 is the sigmoid of 2 z
            return gate * wide_sigmoid(1.5957691216057308f * (gate + 0.044715f * gate * gate * gate)) * up;
        gate = fminf(gate, k.limit);
        return gate * wide_sigmoid(k.slope * gate) * (fminf(fmaxf(up, -k.limit), k.limit) + k.shift);
    }
    return gate;
}

// A tile's results into rows m0 .. m_end - 1 of out [., n_out], from column c0 on. With pairs, even blocks of weight rows are
// gate rows and odd ones up rows, and a tile has 16 NJ columns instead of 32 NJ. Whole groups of eight columns (four in float32)
// where n_out allows it, ragged: one by one.
template <int MI, int NJ, int ACT, typename TO>
__device__ __forceinline__ void wide_results(const f32x4_t (&acc)[MI][NJ], TO* out, int m0, int m_end, int c0, int n_out, WideGate k, bool ragged) {
    constexpr bool PAIRS = wide_pairs(ACT);
    constexpr int COLS = PAIRS ? NJ / 2 : NJ;                 // blocks of 16 columns
    static_assert(!PAIRS || NJ % 2 == 0, "gate and up blocks in one wave");
    const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), li = lane % 16, g = lane / 16;
    const int wm = wave / 2, wn = wave % 2;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
        const int m = m0 + (2 * i + wm) * 16 + li;
        const bool here = m < m_end;
        TO* const to = out + (size_t)min(m, m_end - 1) * n_out;
        float y[COLS][4];
#pragma unroll
        for (int j = 0; j < COLS; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) y[j][r] = PAIRS ? wide_act<ACT>(acc[i][PAIRS ? 2 * j : j][r], acc[i][PAIRS ? 2 * j + 1 : j][r], k) : wide_act<ACT>(acc[i][j][r], 0.f, k);
        const int c = c0 + wn * COLS * 16;
        if (ragged) {
#pragma unroll
            for (int j = 0; j < COLS; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (here && c + j * 16 + 4 * g + r < n_out) to[c + j * 16 + 4 * g + r] = from_float<TO>(y[j][r]);
        } else if constexpr (sizeof(TO) == 4) {
#pragma unroll
            for (int j = 0; j < COLS; ++j)
                if (here && c + j * 16 + 4 * g < n_out) *reinterpret_cast<float4*>(to + c + j * 16 + 4 * g) = make_float4(y[j][0], y[j][1], y[j][2], y[j][3]);
        } else {
            uint2 u[COLS];
#pragma unroll
            for (int j = 0; j < COLS; ++j) u[j] = make_uint2(pack_bf16x2(y[j][0], y[j][1]), pack_bf16x2(y[j][2], y[j][3]));
#pragma unroll
            for (int j = 0; j + 1 < COLS; j += 2) {
                const uint4 eight = wide_eight(u[j], u[j + 1]);
                const int col = c + j * 16 + g % 2 * 16 + g / 2 * 8;
                if (here && col < n_out) *reinterpret_cast<uint4*>(to + col) = eight;
            }
            if (COLS % 2) {
                const int col = c + (COLS - 1) * 16 + 4 * g;
                if (here && col < n_out) *reinterpret_cast<uint2*>(to + col) = u[COLS - 1];
            }
        }
    }
}
