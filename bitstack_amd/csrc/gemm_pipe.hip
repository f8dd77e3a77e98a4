// The dense product's large tiles on gfx950: y[T, M] = x[T, N] @ w[M, N]^T (+ bias), fp16 in, fp32 accumulation, N % 64 == 0.
//
// A workgroup of 8 waves owns 32 P rows of one operand ("P") x 64 Q rows of the other ("Q") - tokens x features, or
// (SWAP) features x tokens - and walks N in k-steps of 64 columns (one 128-byte line of every row).  Three things
// distinguish it from linear_f16_kernel:
//   - requests write LDS directly (16 bytes per lane): no registers hold pieces on their way and there are no LDS write
//     instructions;
//   - the two waves of every SIMD work in turns.  Waves 0-3 own the upper half of the P rows, waves 4-7 the lower
//     half; a k-step of a wave is a MEMORY phase (all its fragments from LDS into registers) and a MATRIX phase (all its
//     MFMAs), with a barrier behind each, and the lower half runs one phase behind: while one wave of a SIMD
//     multiplies, the other one fetches;
//   - v_mfma_f32_16x16x32_f16 instead of 32x32x16: the same rate per cycle, but under load this part is limited by
//     power, and the smaller form (half the accumulator traffic per product) runs at a higher clock - 1.92 against
//     1.71 GHz in a loop of MFMAs alone, 1.63 against 1.51 GHz in this kernel.
// Measured with random data: 8192 x 8192 x 8192 767 us = 1.43 PFLOP/s (linear_f16_kernel's 256 x 256 tile 883 to 911 us,
// torch's library 711), 16384 x 28672 x 8192 5.38 ms = 1.43 PFLOP/s (6.9 ms; 5.05), 2048 x 14336 x 4096 187 us (222; 179).
// What bounds it: 2560 cycles per k-step of a 256 x 256 tile against 2048 of matrix time (the hand-over of the matrix pipe
// at the two barriers and the issue of the requests), at the clock the power allows.  Measured and not kept: the last MFMAs
// of a phase behind its barrier (841 against 811 us on 8192^3), requests in the MEMORY phases only (916), a single barrier
// per k-step with both waves multiplying at once (846), four waves of 128 x 128 with three fragment sets (870).
//
// Phases are numbered on the wall: the upper half runs MEMORY(s) in phase 2 s and MATRIX(s) in phase 2 s + 1, the lower half
// one later.  Stage s % S holds step s.  The upper P rows of a stage are read in phase 2 s only, the lower ones in
// phase 2 s + 1 only, the Q rows in both; so the requests for step s + S go out
//     upper P rows   by the upper waves in phase 2 s + 1 (their MATRIX(s))
//     lower P rows   by the lower waves in phase 2 s + 2 (their MATRIX(s))
//     Q rows         half by the lower waves in phase 2 s + 2, half by the upper waves in phase 2 s + 2 (their MEMORY(s + 1))
// and are read from phase 2 (s + S) (one later) on: about 2 S - 2 phases cover a request.  A wave waits for ITS requests of a
// step (a counted wait: later ones stay in flight) in front of the barrier that opens the phase in which somebody reads them.
//
// S, the number of stages: what a step of a small tile takes is the latency of its requests over the steps in flight (two stages: 0.5 us whatever the tile, where
// the matrix time of 64 x 128 is 0.19), so the tiles that leave LDS for it have three or four.  us, 2 / 3 / 4 stages: 300 tokens on 1024 x 4096, 64 x 64 26.5 / 16.8 / 13.9,
// 64 x 128 32.8 / 19.7 / 18.3; 509 on 4096 x 4096, 64 x 128 33.9 / 24.5 / 23.1; 1400 on 6144 x 4096, 192 x 192 70.2 / 65.4.  Where a CU has two workgroups these cover each
// other's waits, and the fewer stages that let two fit are ahead (128 x 128 on 257 to 512 workgroups: 1.14 times as long with three).  Five and six stages of 64 x 64: no better.
//
// LDS rows are 128 bytes without padding (a request writes 64 lanes x 16 bytes contiguously); the eight 16-byte pieces of a
// row are XOR-ed with three bits of the row number, chosen so that the 16 lanes LDS serves together in a 16-byte read
// (0-3, 12-15, 20-27 and so on) hit all 64 banks; the lane that requests a piece picks its column accordingly.
// A features fragment takes rows 8 (i / 4) + i % 4 of its 32 features (+ 4 for the other fragment of the pair) as its
// row i: a lane then ends with EIGHT consecutive features of one token, one 16-byte store.
#include "common.h"

#include <type_traits>
#include <utility>

namespace {

template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

constexpr int PK = 64;                        // columns per k-step
typedef __attribute__((address_space(3))) void *lds_ptr;

// wait until at most `n` of this wave's requests are in flight (the LDS counter is not waited for)
template <int n>
__device__ __forceinline__ void wait_requests() {
    __builtin_amdgcn_s_waitcnt((n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8));
}
// wait until this wave's LDS reads have arrived
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8)); }

__device__ __forceinline__ void phase_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// SPLIT: the contracted range is cut into parts of `steps_per_split` k-steps; part p of every tile goes to part[p][T][M] in
// fp32, linear_split_sum_kernel adds them up.
// wide: M % 8 == 0 and y (part) 16-byte aligned: whole 16-byte stores.  Otherwise the outputs of y pass through LDS, so that a
// store instruction still writes whole runs of a row.
template <int P, int Q, bool SWAP, int S, bool SPLIT>
__global__ __launch_bounds__(512, 2) void linear_pipe_kernel(
    const half_t *__restrict__ x, const half_t *__restrict__ w, const half_t *__restrict__ bias,
    half_t *__restrict__ y, float *__restrict__ part, int T, int M, int N, int steps_per_split, int wide) {
    static_assert((SWAP ? P : Q) % 2 == 0, "feature fragments come in pairs");
    constexpr int BP = 32 * P, BQ = 64 * Q;   // P, Q: 16-row fragments of a wave
    constexpr int BT = SWAP ? BQ : BP, BF = SWAP ? BP : BQ;
    constexpr int PJ = (P + 1) / 2, QJ = Q;   // requests per wave and k-step, 8 rows each (an odd P: the last wave's repeat rows of its half)
    // one array per operand and stage: the compiler then knows that a request for one stage does not touch the other.  (It tells eight such arrays apart, hence
    // four stages at most; the two operands of a stage in one array, which would allow more, make it wait for requests that the reads have no part in.)
    __shared__ __attribute__((aligned(1024))) half_t sp0[BP * PK], sp1[BP * PK], sp2[S > 2 ? BP * PK : 1], sp3[S > 3 ? BP * PK : 1];
    __shared__ __attribute__((aligned(1024))) half_t sq0[BQ * PK], sq1[BQ * PK], sq2[S > 2 ? BQ * PK : 1], sq3[S > 3 ? BQ * PK : 1];
    auto p_stage = [&](auto stage) -> half_t * {
        constexpr int k = decltype(stage)::value;
        return k == 0 ? sp0 : k == 1 ? sp1 : k == 2 ? sp2 : sp3;
    };
    auto q_stage = [&](auto stage) -> half_t * {
        constexpr int k = decltype(stage)::value;
        return k == 0 ? sq0 : k == 1 ? sq1 : k == 2 ? sq2 : sq3;
    };

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wp = wave >> 2, wq = wave & 3;
    const int lm = lane & 15, g = lane >> 4;

    // Workgroups are dealt round-robin to the 8 XCDs, each with its own L2: every XCD gets a contiguous run of (split,
    // tile) slots, tiles ordered so that those in flight on it at a time form a compact block (TGROUP token tiles x
    // consecutive feature tiles: 12 tile rows and columns in L2 for 32 tiles instead of 33; 16384 x 28672 x 8192 6.9 -> 6.1 ms
    // from this alone).
    int t0, m0, sp = 0;
    {
        const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, base = nb >> 3, rem = nb & 7;
        int v = xcd * base + min(xcd, rem) + loc;
        constexpr int TGROUP = 4;
        const int tt = (T + BT - 1) / BT, ft = (M + BF - 1) / BF;
        if (SPLIT) {
            sp = v / (tt * ft);
            v -= sp * (tt * ft);
        }
        const int grp = v / (TGROUP * ft), r = v - grp * TGROUP * ft, gs = min(TGROUP, tt - grp * TGROUP);
        m0 = (r / gs) * BF;
        t0 = (grp * TGROUP + r % gs) * BT;
    }
    const int all_steps = N / PK;
    const int s_begin = SPLIT ? sp * steps_per_split : 0;
    const int steps = SPLIT ? min(steps_per_split, all_steps - s_begin) : all_steps;

    const half_t *xo = x + (int64_t)t0 * N + (int64_t)s_begin * PK, *wo = w + (int64_t)m0 * N + (int64_t)s_begin * PK;
    const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc((void *)(SWAP ? wo : xo), 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t rq = __builtin_amdgcn_make_buffer_rsrc((void *)(SWAP ? xo : wo), 0, -1, 0x00020000);
    // three bits of the row number that its pieces are XOR-ed with: for whole runs of 16 rows (tokens), and for the rows a
    // features fragment takes
    auto swizzle = [](bool features, int r) { return features ? ((r >> 1) & 1) | (((r >> 3) & 3) << 1) : (r >> 1) & 7; };
    // request j of this wave: 8 rows x 128 bytes; rows beyond T or M repeat the last one (their outputs are never stored)
    int prow[PJ];
#pragma unroll
    for (int j = 0; j < PJ; j++) prow[j] = (wp * 2 * P + (P % 2 == 0 ? wq * PJ + j : min(wq * PJ + j, 2 * P - 1))) * 8;
    const int qrow = wave * QJ * 8;
    const int p_last = SWAP ? M - 1 - m0 : T - 1 - t0, q_last = SWAP ? T - 1 - t0 : M - 1 - m0;
    uint32_t voff_p[PJ], voff_q[QJ];
#pragma unroll
    for (int j = 0; j < PJ; j++) {
        const int r = prow[j] + (lane >> 3);
        voff_p[j] = (uint32_t)min(r, p_last) * (uint32_t)N * 2u + 16u * ((lane & 7) ^ swizzle(SWAP, r));
    }
#pragma unroll
    for (int j = 0; j < QJ; j++) {
        const int r = qrow + 8 * j + (lane >> 3);
        voff_q[j] = (uint32_t)min(r, q_last) * (uint32_t)N * 2u + 16u * ((lane & 7) ^ swizzle(!SWAP, r));
    }
    // where a step's columns are in the rows, in bytes (steps behind the last: the last again)
    auto column_of = [&](int step_) { return min(step_, steps - 1) * (PK * 2); };
    auto request_p = [&](auto stage, int column, int j) {
        half_t *dst = p_stage(stage) + prow[j] * PK;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rp, (lds_ptr)dst, 16, (int)voff_p[j], column, 0, 0);
    };
    auto request_q = [&](auto stage, int column, int j) {
        half_t *dst = q_stage(stage) + (qrow + 8 * j) * PK;
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rq, (lds_ptr)dst, 16, (int)voff_q[j], column, 0, 0);
    };

    float4_t acc[P][Q];
#pragma unroll
    for (int i = 0; i < P; i++)
#pragma unroll
        for (int j = 0; j < Q; j++) acc[i][j] = (float4_t){0.f, 0.f, 0.f, 0.f};

    // fragment kk (32 columns) of fragment row lm: piece 4 kk + g of row `frow` of the token or feature fragments
    const int fr = 8 * (lm >> 2) + (lm & 3);                                  // this lane's row of a features fragment, + 4 (f & 1) + 32 (f / 2)
    const int frow_p = SWAP ? fr : lm, frow_q = SWAP ? lm : fr;
    const int swz_p = swizzle(SWAP, frow_p), swz_q = swizzle(!SWAP, frow_q);
    auto frag_row = [](bool features, int i) { return features ? 32 * (i >> 1) + 4 * (i & 1) : 16 * i; };
    half8_t fp[2][P], fq[2][Q];
    auto load_frags = [&](auto stage) {
        const half_t *ps = p_stage(stage) + (wp * P * 16 + frow_p) * PK;
        const half_t *qs = q_stage(stage) + (wq * Q * 16 + frow_q) * PK;
#pragma unroll
        for (int kk = 0; kk < 2; kk++) {
            const int pp = 8 * ((4 * kk + g) ^ swz_p), pq = 8 * ((4 * kk + g) ^ swz_q);
#pragma unroll
            for (int j = 0; j < Q; j++) fq[kk][j] = *reinterpret_cast<const half8_t *>(qs + frag_row(!SWAP, j) * PK + pq);
#pragma unroll
            for (int i = 0; i < P; i++) fp[kk][i] = *reinterpret_cast<const half8_t *>(ps + frag_row(SWAP, i) * PK + pp);
        }
    };
    // quarter q of a k-step: columns 32 (q / 2) .. + 31, half of the P fragments (features are the first MFMA operand)
    auto mfmas = [&](int q) {
#pragma unroll
        for (int i = q & 1 ? PJ : 0; i < (q & 1 ? P : PJ); i++)
#pragma unroll
            for (int j = 0; j < Q; j++)
                acc[i][j] = SWAP ? __builtin_amdgcn_mfma_f32_16x16x32_f16(fp[q >> 1][i], fq[q >> 1][j], acc[i][j], 0, 0, 0)
                                 : __builtin_amdgcn_mfma_f32_16x16x32_f16(fq[q >> 1][j], fp[q >> 1][i], acc[i][j], 0, 0, 0);
    };
    auto all_q = [&](auto stage, int step_) {
        const int column = column_of(step_);
#pragma unroll
        for (int j = 0; j < QJ; j++) request_q(stage, column, j);
    };
    auto all_p = [&](auto stage, int step_) {
        const int column = column_of(step_);
#pragma unroll
        for (int j = 0; j < PJ; j++) request_p(stage, column, j);
    };
    // steps 0 .. `steps` - 1, S at a time (no exit between them: a path around one would make the compiler wait for the wrong requests at the top of the loop)
    auto walk = [&](auto &&step) {
        int s = 0;
        for (; s + S - 1 < steps; s += S) static_for<S>([&](auto k) { step(k, s + decltype(k)::value); });
        static_for<S - 1>([&](auto k) {
            if (s + decltype(k)::value < steps) step(k, s + decltype(k)::value);
        });
    };

    // ---- fill: step 0 by everybody, then what the phases before the first would have requested ----------
    all_q(std::integral_constant<int, 0>{}, 0);
    all_p(std::integral_constant<int, 0>{}, 0);
    if (wp == 0) {
        static_for<S - 1>([&](auto k) {
            constexpr int n = decltype(k)::value + 1;
            all_p(std::integral_constant<int, n>{}, n);
            if constexpr (n < S - 1) all_q(std::integral_constant<int, n>{}, n);
        });
        wait_requests<(S - 1) * PJ + (S - 2) * QJ>();
        phase_barrier();
        walk([&](auto stage, int s) {
            using Before = std::integral_constant<int, (decltype(stage)::value + S - 1) % S>;
            // MEMORY(s): the reads first, they are what the phase waits for
            load_frags(stage);
            __builtin_amdgcn_sched_barrier(0);
            all_q(Before{}, s + S - 1);
            wait_lds();
            phase_barrier();
            // MATRIX(s)
            const int column = column_of(s + S);
            __builtin_amdgcn_s_setprio(1);
            static_for<4>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                if constexpr (q < PJ) request_p(stage, column, q);
                mfmas(q);
                __builtin_amdgcn_sched_barrier(0);
            });
            __builtin_amdgcn_s_setprio(0);
            wait_requests<(S - 1) * PJ + (S - 2) * QJ>();      // the Q rows and upper P rows of step s + 1
            phase_barrier();
        });
        phase_barrier();
    } else {
        static_for<S - 1>([&](auto k) {
            constexpr int n = decltype(k)::value + 1;
            all_q(std::integral_constant<int, n>{}, n);
            all_p(std::integral_constant<int, n>{}, n);
        });
        wait_requests<(S - 1) * (PJ + QJ)>();
        phase_barrier();
        phase_barrier();
        walk([&](auto stage, int s) {
            // MEMORY(s)
            load_frags(stage);
            wait_lds();
            wait_requests<PJ + (S - 2) * (PJ + QJ)>();         // the Q rows of step s + 1
            phase_barrier();
            // MATRIX(s)
            const int column = column_of(s + S);
            __builtin_amdgcn_s_setprio(1);
            static_for<4>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                // Q rows first: they are read one phase earlier
                static_for<PJ + QJ>([&](auto jc) {
                    constexpr int j = decltype(jc)::value;
                    if constexpr (j * 4 / (PJ + QJ) == q) {
                        if constexpr (j < QJ) request_q(stage, column, j);
                        else request_p(stage, column, j - QJ);
                    }
                });
                mfmas(q);
                __builtin_amdgcn_sched_barrier(0);
            });
            __builtin_amdgcn_s_setprio(0);
            wait_requests<(S - 1) * (PJ + QJ)>();              // the lower P rows of step s + 1
            phase_barrier();
        });
    }
    wait_requests<0>();                        // (the repeated last step's)

    // D[feature row, token]: the lane holds token lm of token fragment a, and of the pair of feature fragments (2 p, 2 p + 1)
    // the eight features 32 p + 8 g .. + 7
    constexpr int TA = SWAP ? Q : P, FP = (SWAP ? P : Q) / 2;
    const int tw = t0 + (SWAP ? wq * Q : wp * P) * 16, mw = m0 + (SWAP ? wp * P : wq * Q) * 16;
    auto value = [&](int a, int p, int e) { return SWAP ? acc[2 * p + (e >> 2)][a][e & 3] : acc[a][2 * p + (e >> 2)][e & 3]; };
    if (SPLIT || wide) {
#pragma unroll
        for (int p = 0; p < FP; p++) {
            const int m = mw + 32 * p + 8 * g;
            float bv[8];
#pragma unroll
            for (int e = 0; e < 8; e++) bv[e] = !SPLIT && bias && m + e < M ? (float)bias[m + e] : 0.f;
#pragma unroll
            for (int a = 0; a < TA; a++) {
                const int t = tw + 16 * a + lm;
                if (t >= T || m >= M) continue;
                if (SPLIT) {
                    float *o = part + ((int64_t)sp * T + t) * M + m;
                    if (wide) {
                        *reinterpret_cast<float4_t *>(o) = (float4_t){value(a, p, 0), value(a, p, 1), value(a, p, 2), value(a, p, 3)};
                        *reinterpret_cast<float4_t *>(o + 4) = (float4_t){value(a, p, 4), value(a, p, 5), value(a, p, 6), value(a, p, 7)};
                    } else {
#pragma unroll
                        for (int e = 0; e < 8; e++)
                            if (m + e < M) o[e] = value(a, p, e);
                    }
                } else {
                    half8_t v;
#pragma unroll
                    for (int e = 0; e < 8; e++) v[e] = (half_t)(value(a, p, e) + bv[e]);
                    *reinterpret_cast<half8_t *>(y + (int64_t)t * M + m) = v;
                }
            }
        }
    } else {
        // 16 tokens x 32 features at a time through 1 KB of LDS per wave; 32 lanes then write 64 bytes of a row
        phase_barrier();                       // (everybody's requests have landed)
        half_t *buf = sq0 + wave * 512;
        const int f = lane & 31, th = lane >> 5;
#pragma unroll
        for (int p = 0; p < FP; p++) {
            const int m = mw + 32 * p + f;
            const float bv = bias && m < M ? (float)bias[m] : 0.f;
#pragma unroll
            for (int a = 0; a < TA; a++) {
                float4_t lo = {value(a, p, 0), value(a, p, 1), value(a, p, 2), value(a, p, 3)}, hi = {value(a, p, 4), value(a, p, 5), value(a, p, 6), value(a, p, 7)};
                half8_t v;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    v[e] = (half_t)(lo[e] + __shfl(bv, 8 * g + e, 64));
                    v[e + 4] = (half_t)(hi[e] + __shfl(bv, 8 * g + e + 4, 64));
                }
                *reinterpret_cast<half8_t *>(buf + lm * 32 + 8 * g) = v;
                asm volatile("" ::: "memory");   // (the LDS operations of a wave execute in order)
#pragma unroll
                for (int r = 0; r < 8; r++) {
                    const int t = tw + 16 * a + 2 * r + th;
                    const half_t o = buf[(2 * r + th) * 32 + f];
                    if (t < T && m < M) y[(int64_t)t * M + m] = o;
                }
                asm volatile("" ::: "memory");
            }
        }
    }
}

// y = fp16(sum over the parts in order + bias): eight outputs per thread (WIDE: M % 8 == 0, 16-byte aligned y), or one
template <bool WIDE>
__global__ __launch_bounds__(256) void linear_split_sum_kernel(const float *__restrict__ part, const half_t *__restrict__ bias,
                                                               half_t *__restrict__ y, int splits, int64_t total, int M) {
    const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * (WIDE ? 8 : 1);
    if (i >= total) return;
    const int m = (int)(i % M);
    if (WIDE) {
        float4_t a = {0.f, 0.f, 0.f, 0.f}, b = a;
        for (int s = 0; s < splits; s++) {
            const float *p = part + s * total + i;
            a += *reinterpret_cast<const float4_t *>(p);
            b += *reinterpret_cast<const float4_t *>(p + 4);
        }
        half8_t v;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            v[e] = (half_t)(a[e] + (bias ? (float)bias[m + e] : 0.f));
            v[e + 4] = (half_t)(b[e] + (bias ? (float)bias[m + e + 4] : 0.f));
        }
        *reinterpret_cast<half8_t *>(y + i) = v;
    } else {
        float a = 0.f;
        for (int s = 0; s < splits; s++) a += part[s * total + i];
        y[i] = (half_t)(a + (bias ? (float)bias[m] : 0.f));
    }
}

// A tile of P x Q fragments; S stages where the grid leaves a CU one workgroup, S_TWO where it has more (fewer of them, so that two fit its LDS) and up to FEW k-steps: requests
// for steps behind the last are made for nothing, one step's more with every stage.  us, S / S_TWO stages: 128 x 256, 1794 tokens on 2719 x 256 11.9 / 11.5, x 512 14.0 / 13.7, x 640 15.3 / 15.1,
// x 1024 18.2 / 18.2, x 2048 31.6 / 35.9, 755 on 8066 x 320 12.8 / 12.4, x 512 14.7 / 14.7, x 1024 23.4 / 24.2; 128 x 128, 600 on 5000 x 128 5.9 / 5.6, x 192 6.5 / 6.2, x 256 6.6 / 6.7.
template <int P_, int Q_, bool SWAP_, int S_, int S_TWO_, int FEW_>
struct PipeBuild {
    static constexpr int P = P_, Q = Q_, S = S_, S_TWO = S_TWO_, FEW = FEW_;
    static constexpr bool SWAP = SWAP_;
    static constexpr int BT = SWAP ? 64 * Q : 32 * P, BF = SWAP ? 32 * P : 64 * Q;
    static constexpr bool PAIR = S_TWO != S && S_TWO * (BT + BF) * PK * 2 <= 80 * 1024;      // two workgroups fit the LDS of a CU
    static_assert(S * (BT + BF) * PK * 2 <= 160 * 1024, "LDS of a CU");
};
struct PipePlan {
    int steps, parts, stages;                 // of a part; every part holds at least one k-step
    unsigned tiles;
};
template <class B>
PipePlan pipe_plan(int T, int M, int N, int splits) {
    PipePlan p;
    p.tiles = (unsigned)(bs_cdiv(T, B::BT) * bs_cdiv(M, B::BF));
    p.steps = (int)bs_cdiv(N / PK, splits);
    p.parts = (int)bs_cdiv(N / PK, p.steps);
    p.stages = p.steps <= B::FEW || (B::PAIR && (int64_t)p.tiles * p.parts > 256) ? B::S_TWO : B::S;
    return p;
}

template <class B>
int launch_pipe(const half_t *x, const half_t *w, const half_t *bias, half_t *y, int T, int M, int N, int splits, float *part, hipStream_t s) {
    constexpr int P = B::P, Q = B::Q, S = B::S, S_TWO = B::S_TWO;
    constexpr bool SWAP = B::SWAP;
    const PipePlan p = pipe_plan<B>(T, M, N, splits);
    const int wide = M % 8 == 0 && bs_aligned(y, 16) && bs_aligned(part, 16);
    // (All tiles sum in the order of the columns: equal rows of x or w have equal outputs.  XCDs that each start an eighth further along the rows ask different memory channels, 14336 x
    // 4096, 4 blocks, 300 tokens 89.6 / 84.7 us, but a token's sums would then depend on where its tile lies.)
    if (p.parts == 1) {
        if (p.stages != S) linear_pipe_kernel<P, Q, SWAP, S_TWO, false><<<p.tiles, 512, 0, s>>>(x, w, bias, y, nullptr, T, M, N, p.steps, wide);
        else linear_pipe_kernel<P, Q, SWAP, S, false><<<p.tiles, 512, 0, s>>>(x, w, bias, y, nullptr, T, M, N, p.steps, wide);
    } else if constexpr (B::BF == 64) {
        return BS_ERR_SHAPE;                  // (never cut: see linear_choice)
    } else {
        if (p.stages != S) linear_pipe_kernel<P, Q, SWAP, S_TWO, true><<<p.tiles * p.parts, 512, 0, s>>>(x, w, bias, y, part, T, M, N, p.steps, wide);
        else linear_pipe_kernel<P, Q, SWAP, S, true><<<p.tiles * p.parts, 512, 0, s>>>(x, w, bias, y, part, T, M, N, p.steps, wide);
        BS_LAUNCH_CHECK();
        const int64_t total = (int64_t)T * M;
        if (wide) linear_split_sum_kernel<true><<<(unsigned)bs_cdiv(total, 8 * 256), 256, 0, s>>>(part, bias, y, p.parts, total, M);
        else linear_split_sum_kernel<false><<<(unsigned)bs_cdiv(total, 256), 256, 0, s>>>(part, bias, y, p.parts, total, M);
    }
    BS_LAUNCH_CHECK();
    return BS_OK;
}

// f on the build of a tile of bt x bf (tokens x features per workgroup)
template <class F>
int with_pipe_build(int bt, int bf, F &&f) {
    switch (bt * 1000 + bf) {
#define PIPE_CASE(bt, bf, ...) \
    case bt * 1000 + bf: { \
        typedef PipeBuild<__VA_ARGS__> B; \
        static_assert(B::BT == bt && B::BF == bf, "the tile"); \
        return f(B()); \
    }
        PIPE_CASE(256, 256, 8, 4, false, 2, 2, 0) PIPE_CASE(224, 256, 7, 4, false, 2, 2, 0) PIPE_CASE(192, 256, 6, 4, false, 2, 2, 0) PIPE_CASE(256, 192, 6, 4, true, 2, 2, 0)
        PIPE_CASE(160, 256, 5, 4, false, 3, 3, 0) PIPE_CASE(192, 192, 6, 3, true, 3, 3, 0) PIPE_CASE(256, 128, 8, 2, false, 3, 3, 0) PIPE_CASE(128, 256, 8, 2, true, 3, 2, 8)
        PIPE_CASE(224, 128, 7, 2, false, 3, 3, 0) PIPE_CASE(192, 128, 6, 2, false, 3, 3, 0) PIPE_CASE(128, 192, 6, 2, true, 3, 3, 0) PIPE_CASE(160, 128, 5, 2, false, 3, 2, 2)
        PIPE_CASE(128, 128, 4, 2, false, 4, 2, 3) PIPE_CASE(96, 128, 3, 2, false, 4, 2, 3) PIPE_CASE(64, 128, 2, 2, false, 4, 3, 3) PIPE_CASE(64, 64, 2, 1, true, 4, 4, 0)
#undef PIPE_CASE
        default: return BS_ERR_SHAPE;
    }
}

}  // namespace

// splits > 1: part holds splits * T * M floats.
int bs_launch_linear_pipe(const half_t *x, const half_t *w, const half_t *bias, half_t *y, int T, int M, int N, int bt, int bf,
                          int splits, float *part, hipStream_t s) {
    if (N % PK != 0 || splits < 1 || (splits > 1 && !part)) return BS_ERR_SHAPE;
    return with_pipe_build(bt, bf, [&](auto b) { return launch_pipe<decltype(b)>(x, w, bias, y, T, M, N, splits, part, s); });
}

// the parts and stages that it runs with
int bs_linear_pipe_plan(int T, int M, int N, int bt, int bf, int splits, int *parts, int *stages) {
    return with_pipe_build(bt, bf, [&](auto b) {
        const PipePlan p = pipe_plan<decltype(b)>(T, M, N, splits);
        *parts = p.parts;
        *stages = p.stages;
        return (int)BS_OK;
    });
}
