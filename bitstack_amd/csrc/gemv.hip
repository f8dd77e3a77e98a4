// Packed-sign GEMV for decode (1..8 tokens) on gfx950.
//
//   y[t, m] = sum_i sum_r u_i[m, r] * ( sum_n s_i[m, n] * vt_i[r, n] * x[t, n] )
//
// The inner sum is a matrix product  Z (16 ranks x N)  x  S^T (N x rows)  with
// Z[r, n] = vt_i[r, n] * x[t, n], so it runs on v_mfma_f32_16x16x32_f16:
// A = a 16 x 32 patch of Z (fp16), B = 32 signs of 16 rows, D[r, m] in fp32.
// A lane ends up with four ranks of ONE row, multiplies them by
// u_i[m, 4g..4g+3], and two cross-lane adds finish the row.
//
// ---- sign decode without shifts ------------------------------------------
// Decoding a bit to fp16 +-1 costs a shift and a mask per two signs, which is
// more VALU time than the MFMA it feeds.  Instead the bit is left WHERE IT IS
// in its 16-bit half and merged into a constant with one v_and_or_b32:
//     v = (w & (0x00010001 << j)) | base_j
// so the fp16 operand is one of two values {a_j, b_j} that depend on the bit
// position j, chosen such that b_j - a_j = 2 exactly:
//     j = 15 (sign)        {+1, -1}      mid  0   (Z is stored negated here)
//     j = 14 (exponent)    {0, 2}        mid  1
//     j = 9..4 (mantissa)  {4,6} {8,10} {16,18} {32,34} {64,66} {128,130}
// Then s = v - mid_j, and   sum_n s_n z_n = sum_n v_n z_n - sum_n mid_n z_n.
// The first sum is what the MFMAs accumulate; the second does not depend on
// the row; the waves of a workgroup share it out (16 / WAVES steps each, one extra
// MFMA per step against a constant operand) and exchange their shares through LDS
// when a row is flushed.  All codes are exact in fp16 and every product is exact
// in fp32, so the only extra error is fp32 accumulation of terms up to 129x
// larger than z (about 1e-5 relative, far below the fp16 rounding of y).
// Bit positions 10..13 and 0..3 have no such code (or a badly conditioned
// one), so the word is used three times: as loaded (positions 15,14,9..4),
// shifted left by 2 (positions 15,14 = original bits 13,12) and by 4
// (positions 15,14,7..4 = original bits 11,10,3..0): 2 shifts + 16 merges per
// 32 signs.
//
// ---- work split ------------------------------------------------------------
// The matrix stack is cut into UNITS: (block i, row tile of WAVES*R*16 rows,
// 512-column chunk), ordered with the chunk fastest.  The grid is persistent:
// about two workgroups per CU (one for three or four tokens), each owning one
// contiguous range of units of equal length, so the load is balanced for any
// shape and each workgroup pays its pipeline fill once.  Up to four matrices that
// read the same x share a launch: the grid is cut into one run of workgroups per
// matrix.  Per unit every lane reads its 16 bytes of signs
// (128 columns of one row) with one 128-bit load per row tile, one unit ahead
// of use; Z for unit u+1 is produced by all threads (vt and x loads issued
// before the MFMA loop of unit u, finished after it) into the other half of a
// double-buffered LDS image laid out in MFMA operand order: one barrier per
// unit.  Accumulators are flushed whenever the range crosses into another
// (block, row tile): scaled by u, reduced over ranks, written as a partial
// row sum to scratch [I, KMAX, T, M] (fp32); the workgroup that ends a row of
// units also writes zeros to the slots above its own (a row is spread over at
// most KMAX workgroups, often fewer).  A second kernel adds the KMAX slots of
// every block in a fixed order, adds the bias, rounds to fp16 and applies
// the epilogue (none, + residual, silu(a) * b): deterministic, no atomics.  Workgroups with neighbouring ranges - which read
// the same slices of vt - sit on the same XCD (and share its L2).
#include "common.h"
#include "gemv_shared.h"

#include <algorithm>

#include <type_traits>
#include <utility>

namespace {

// Compile-time loop: the step tables below must fold to immediates.
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

constexpr int CH = 512;   // columns per chunk: 4 lane groups x 16 bytes of signs
// Sign bytes per launch from which the block-scaled kernel is preferred to the sparse one.  us sparse / block-scaled, one token: 4096 x 4096, 4 blocks (8 MiB) 9.4 / 9.3,
// 8 blocks 13.7 / 12.6, 14336 x 4096, 8 blocks 30.6 / 28.7; two tokens: 8 blocks of 4096 x 4096 (16 MiB) 16.8 / 17.6, 6144 x 4096, 6 blocks 20.4 / 22.2, 4096 x 14336, 3 (21 MiB)
// 22.5 / 22.9, 14336 x 4096, 8 (56 MiB) 38.9 / 39.9, 4096 x 14336, 16 (112 MiB) 65.1 / 60.9.
// One token from 8 MiB on too where the sparse kernel, whose units are half as wide, leaves 200 partial sums per output or more: few rows of many columns (355 x 15872, 16
// blocks, 496 sums against 144, 15.7 / 12.2; 925 x 11776, 9, 207 against 108, 13.2 / 11.6; of 120 drawn calls from 8 to 12 MiB 2 are more than 3 % behind the block-scaled
// kernel, without it 19, 28 % at worst; over all of them 0.93 of its time).  Two tokens: of 120 from 8 to 24 MiB none.
constexpr int64_t MX_MIN_SIGN_BYTES = 12 << 20, MX_MIN_SIGN_BYTES_TWO = 24 << 20, MX_MIN_SIGN_BYTES_MANY_SUMS = 8 << 20;
constexpr int MX_MANY_SUMS = 200;


// step -> bit position used in that step; steps 0-7 read the word as loaded,
// 8-9 after `<< 2`, 10-15 after `<< 4`.
__host__ __device__ constexpr int step_pos(int st) {
    constexpr int P[16] = {15, 14, 9, 8, 7, 6, 5, 4, 15, 14, 15, 14, 7, 6, 5, 4};
    return P[st];
}
// original bit (within its 16-bit half) -> step that consumes it
__host__ __device__ constexpr int bit_step(int b) {
    constexpr int S[16] = {15, 14, 13, 12, 7, 6, 5, 4, 3, 2, 11, 10, 9, 8, 1, 0};
    return S[b];
}
__host__ __device__ constexpr uint32_t pos_base(int j) {
    return j == 15 ? 0x3C003C00u : j == 14 ? 0u : j == 9 ? 0x44004400u : j == 8 ? 0x48004800u
         : j == 7 ? 0x4C004C00u : j == 6 ? 0x50005000u : j == 5 ? 0x54005400u : 0x58005800u;
}
__host__ __device__ constexpr float pos_mid(int j) {
    return j == 15 ? 0.f : j == 14 ? 1.f : j == 9 ? 5.f : j == 8 ? 9.f : j == 7 ? 17.f
         : j == 6 ? 33.f : j == 5 ? 65.f : 129.f;
}

// mid of the position each step reads (0 for the sign position)
__constant__ float step_mid_table[16] = {0.f, 1.f, 5.f, 9.f, 17.f, 33.f, 65.f, 129.f,
                                         0.f, 1.f, 0.f, 1.f, 17.f, 33.f, 65.f, 129.f};

// LDS image of Z for one chunk: [t][step (16)][g (4)][r (16)][slot (8)] halves.
__device__ inline int z_index(int t, int st, int g, int r) { return (((t * 16 + st) * 4 + g) * 16 + r) * 8; }

// (w & mask) | base as ONE v_and_or_b32.  VOP3 takes no literal and one scalar
// operand, so the two constants are first pinned into registers (mask scalar, base
// vector) with empty asm statements the optimiser cannot see through; the merge
// itself stays an ordinary expression.  It must not be written as an asm
// instruction: the compiler's hazard recogniser does not look inside inline asm,
// and a VALU write to registers that an MFMA issued just before still reads as its
// accumulator input (the MFMA reads SrcC several cycles after issue) corrupts that
// MFMA unless the recogniser can see the write and pad it.
__device__ inline uint32_t pin_scalar(uint32_t v) {
    asm("" : "+s"(v));
    return v;
}
__device__ inline uint32_t pin_vector(uint32_t v) {
    asm("" : "+v"(v));
    return v;
}
__device__ inline uint32_t and_or(uint32_t w, uint32_t mask, uint32_t base) { return (w & mask) | base; }

// One producer item: rank r, lane group pg, word p, byte pair (JB, JB + 2) of
// the word.  Two 16-byte pieces of vt (8 consecutive columns each) times x
// give 8 (slot 2p, slot 2p+1) pairs, one per bit of the byte.
template <int JB>
__device__ inline void produce_finish(half_t *zt, int pg, int p, int r, half8_t v0, half8_t v1,
                                      half8_t x0, half8_t x1) {
    const half8_t z0 = v0 * x0, z1 = v1 * x1;
    static_for<8>([&](auto ec) {
        constexpr int e = decltype(ec)::value;
        constexpr int st = bit_step(8 * JB + 7 - e);
        constexpr bool neg = step_pos(st) == 15;
        half2_t o = {z0[e], z1[e]};
        if (neg) o = -o;
        *reinterpret_cast<half2_t *>(zt + z_index(0, st, pg, r) + 2 * p) = o;
    });
}

template <int T, int WAVES, int R>
__global__ __launch_bounds__(64 * WAVES, (T == 1 ? (WAVES == 16 ? 1 : WAVES == 4 && R == 4 ? 3 : 4) : (T == 2 ? (WAVES == 8 && R == 2 ? 4 : 2) : 1))) void gemv_kernel(
    const GemvGroup grp, const half_t *__restrict__ x, int N, int K, int n_chunks) {
    constexpr int RW = WAVES * R * 16;          // rows per workgroup
    constexpr int COMBOS = WAVES >= 8 ? 1 : 8 / WAVES;   // (jb, pg) producer combos per wave (waves 8.. of 16 have none)
    constexpr int ZHALVES = T * 16 * 4 * 16 * 8;   // one Z buffer
    constexpr int CSTEPS = 16 / WAVES;          // correction steps handled by each wave
    extern __shared__ __attribute__((aligned(16))) half_t lds[];
    half_t *zl = lds;                                              // [2][ZHALVES]
    float *corrl = reinterpret_cast<float *>(lds + 2 * ZHALVES);   // [2][WAVES][T][16], alternating per flush

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // wave-uniform, keep it scalar
    const int lm = lane & 15, g = lane >> 4;

    // XCD-aware slot -> range: hardware deals workgroups round-robin to 8 XCDs;
    // give each XCD a contiguous run of ranges.
    int wg;
    {
        const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
        const int base = nb >> 3, rem = nb & 7;
        wg = xcd * base + min(xcd, rem) + loc;
    }
    // which matrix this workgroup belongs to (all of it is wave-uniform)
    GemvMat mat = grp.m[0];
#pragma unroll
    for (int j = 1; j < GEMV_MAX_GROUP; j++)
        if (j < grp.n && wg >= grp.m[j].first_wg) mat = grp.m[j];
    wg -= mat.first_wg;
    const int pair = mat.pair, cq = pair ? (wg & 1) : 0;      // chunk parity this workgroup takes
    const int wv = wg >> pair;                                // its place in the partition
    const int nch = n_chunks >> pair;                         // units per row of units
    const uint8_t *__restrict__ packed = mat.packed;
    const half_t *__restrict__ u = mat.u;
    const half_t *__restrict__ vt = mat.vt;
    float *__restrict__ part = mat.part;
    const int M = mat.M, row_tiles = mat.row_tiles, kmax = mat.kmax;
    const Split sp = mat.sp;
    const int u_begin = sp.start(wv), u_end = sp.start(wv + 1);
    if (u_begin >= u_end) return;

    const int64_t row_bytes = N >> 3;
    const int pp = lane & 3, pr = lane >> 2;      // producer role: word, rank
    const bool r_live = pr < K;

    // Addresses are a wave-uniform base (block i, kept in scalar registers) plus a
    // 32-bit per-lane byte offset that only changes with the row tile.
    const uint8_t *qbase;       // packed signs of block i
    const half_t *vbase;
    uint32_t qoff[R];           // this lane's row in each row tile of the wave
    const uint32_t voff = ((uint32_t)(r_live ? pr : 0) * (uint32_t)N + 32u * pp) * 2u;   // producer role
    auto set_row = [&](int rowid) {
        const int i = rowid / row_tiles, rt = rowid % row_tiles;
        qbase = packed + (int64_t)i * M * row_bytes;
        vbase = vt + (int64_t)i * K * N;
#pragma unroll
        for (int jr = 0; jr < R; jr++) {
            const uint32_t row = (uint32_t)min(rt * RW + (wave * R + jr) * 16 + lm, M - 1);
            qoff[jr] = row * (uint32_t)row_bytes + 16u * g;
        }
    };
    auto mid_operand = [&](int k) {   // constant MFMA operand for the correction sums of this wave's steps
        const half_t m = (half_t)step_mid_table[wave * CSTEPS + k];
        return (half8_t){m, m, m, m, m, m, m, m};
    };

    float4_t acc[R][T];
    float4_t corr[T];
    auto clear_acc = [&]() {
#pragma unroll
        for (int t = 0; t < T; t++) {
            corr[t] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int jr = 0; jr < R; jr++) acc[jr][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
        }
    };
    clear_acc();

    half8_t pv[COMBOS][2];        // vt pieces in flight for the next unit
    half8_t px[COMBOS][T][2];     // x pieces in flight for the next unit
    auto produce_issue = [&](int c) {
        if (WAVES > 8 && wave >= 8) return;
#pragma unroll
        for (int k = 0; k < COMBOS; k++) {
            const int combo = wave + k * WAVES, pg = combo & 3, jb = combo >> 2;
            const int col = c * CH + 128 * pg + 8 * jb;            // wave-uniform
            const uint8_t *vs = reinterpret_cast<const uint8_t *>(vbase + col) + voff;
            pv[k][0] = *reinterpret_cast<const half8_t *>(vs);
            pv[k][1] = *reinterpret_cast<const half8_t *>(vs + 32);
#pragma unroll
            for (int t = 0; t < T; t++) {
                const uint8_t *xs = reinterpret_cast<const uint8_t *>(x + (int64_t)t * N + col) + 64u * pp;
                px[k][t][0] = *reinterpret_cast<const half8_t *>(xs);
                px[k][t][1] = *reinterpret_cast<const half8_t *>(xs + 32);
            }
        }
    };
    auto produce_write = [&](int buf) {
        if (WAVES > 8 && wave >= 8) return;
        half_t *zbuf = zl + buf * ZHALVES;
#pragma unroll
        for (int k = 0; k < COMBOS; k++) {
            const int combo = wave + k * WAVES, pg = combo & 3, jb = combo >> 2;
            half8_t v0 = pv[k][0], v1 = pv[k][1];
            if (!r_live) { v0 = (half8_t){0, 0, 0, 0, 0, 0, 0, 0}; v1 = v0; }
#pragma unroll
            for (int t = 0; t < T; t++) {
                half_t *zt = zbuf + z_index(t, 0, 0, 0);
                if (jb) produce_finish<1>(zt, pg, pp, pr, v0, v1, px[k][t][0], px[k][t][1]);
                else    produce_finish<0>(zt, pg, pp, pr, v0, v1, px[k][t][0], px[k][t][1]);
            }
        }
    };

    auto consume = [&](uint4_t (&w)[R], int buf) {
        const half_t *zbuf = zl + buf * ZHALVES;
        // Z fragments are fetched one step ahead of the MFMAs that use them: all
        // waves of a workgroup leave the barrier together, so nobody else would
        // cover the LDS latency.
        half8_t zf[2][T];
#pragma unroll
        for (int t = 0; t < T; t++) zf[0][t] = *reinterpret_cast<const half8_t *>(zbuf + z_index(t, 0, g, lm));
        static_for<16>([&](auto stc) {
            constexpr int st = decltype(stc)::value;
            if (st + 1 < 16) {
#pragma unroll
                for (int t = 0; t < T; t++)
                    zf[(st + 1) & 1][t] = *reinterpret_cast<const half8_t *>(zbuf + z_index(t, st + 1, g, lm));
            }
            if (st == 8 || st == 10) {
#pragma unroll
                for (int jr = 0; jr < R; jr++) w[jr] = w[jr] << 2;
            }
            constexpr int j = step_pos(st);
            constexpr uint32_t mask_c = 0x00010001u << j;
            const uint32_t mask = pin_scalar(mask_c), base = j == 14 ? 0u : pin_vector(pos_base(j));
#pragma unroll
            for (int jr = 0; jr < R; jr++) {
                uint4_t sb;
#pragma unroll
                for (int p = 0; p < 4; p++) sb[p] = (j == 14) ? (w[jr][p] & mask) : and_or(w[jr][p], mask, base);
                const half8_t sf = __builtin_bit_cast(half8_t, sb);
#pragma unroll
                for (int t = 0; t < T; t++)
                    acc[jr][t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(zf[st & 1][t], sf, acc[jr][t], 0, 0, 0);
            }
        });
        // row-independent correction: this wave's share of the 16 steps
#pragma unroll
        for (int k = 0; k < CSTEPS; k++) {
#pragma unroll
            for (int t = 0; t < T; t++) {
                const half8_t zc = *reinterpret_cast<const half8_t *>(zbuf + z_index(t, wave * CSTEPS + k, g, lm));
                corr[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(zc, mid_operand(k), corr[t], 0, 0, 0);
            }
        }
    };

    auto load_signs = [&](uint4_t (&w)[R], int c) {
#pragma unroll
        for (int jr = 0; jr < R; jr++) w[jr] = *reinterpret_cast<const uint4_t *>(qbase + c * (CH >> 3) + qoff[jr]);
    };

    // D[r, m]: the lane holds ranks 4g..4g+3 of row (tile jr, lm).  Subtract the
    // correction (summed over waves in a fixed order), scale by u, add the four
    // lane groups, write the partial row sum, start the next row from zero.
    int flush_parity = 0;
    auto flush = [&](int rowid, bool row_done) {
        // Two flushes can follow each other with no barrier in between (a row that
        // ends on the last prefetching unit, then the drain), so the exchange area
        // alternates: a wave still reading the previous sums is never overwritten.
        float *cx = corrl + flush_parity * (WAVES * T * 16);
        flush_parity ^= 1;
        const int i = rowid / row_tiles, rt = rowid % row_tiles;
        half4_t uc[R];      // u[i, row, 4g .. 4g+3]
#pragma unroll
        for (int jr = 0; jr < R; jr++) {
            const int row = min(rt * RW + (wave * R + jr) * 16 + lm, M - 1);
            const half_t *up = u + ((int64_t)i * M + row) * K + 4 * g;
            if (K == 16) {
                uc[jr] = *reinterpret_cast<const half4_t *>(up);
            } else {
#pragma unroll
                for (int v = 0; v < 4; v++) uc[jr][v] = (4 * g + v < K) ? up[v] : (half_t)0;
            }
        }
        if (lm == 0) {
#pragma unroll
            for (int t = 0; t < T; t++) *reinterpret_cast<float4_t *>(cx + (wave * T + t) * 16 + 4 * g) = corr[t];
        }
        __syncthreads();
        const int slot = ((wv - sp.owner(rowid * nch)) << pair) + cq;
#pragma unroll
        for (int t = 0; t < T; t++) {
            float4_t cz = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < WAVES; w++) cz += *reinterpret_cast<const float4_t *>(cx + (w * T + t) * 16 + 4 * g);
#pragma unroll
            for (int jr = 0; jr < R; jr++) {
                const int row = rt * RW + (wave * R + jr) * 16 + lm;
                float val = (acc[jr][t][0] - cz[0]) * (float)uc[jr][0] + (acc[jr][t][1] - cz[1]) * (float)uc[jr][1] +
                            (acc[jr][t][2] - cz[2]) * (float)uc[jr][2] + (acc[jr][t][3] - cz[3]) * (float)uc[jr][3];
                val += __shfl_xor(val, 16, 64);
                val += __shfl_xor(val, 32, 64);
                if (g == 0 && row < M) {
                    part[(((int64_t)i * kmax + slot) * T + t) * M + row] = val;
                    // The workgroup that finishes a row of units holds its highest live slot: it fills the
                    // slots nobody writes with zeros, so the summing kernel adds all kmax slots blindly.
                    if (row_done)
                        for (int dead = slot + (1 << pair); dead < kmax; dead += 1 << pair)
                            part[(((int64_t)i * kmax + dead) * T + t) * M + row] = 0.f;
                }
            }
        }
        clear_acc();
    };

    // ---- pipeline fill: first unit's signs and Z -----------------------------
    int rowid = u_begin / nch, c = u_begin % nch;
    set_row(rowid);
    uint4_t cur[R], nxt[R];
    auto chunk_of = [&](int unit_c) { return (unit_c << pair) + cq; };   // unit within its row -> 512-column chunk
    produce_issue(chunk_of(c));                     // first: Z production only waits for these
    load_signs(cur, chunk_of(c));
    uint32_t warm0;      // loaded for its side effect only (the line ends up in L2)
    {
        // the flush after the last unit is not preceded by a crossing inside the loop:
        // pull the u rows it needs towards L2 now (value unused)
        const int lrow = (u_end - 1) / nch, fi = lrow / row_tiles, frt = lrow % row_tiles;
        const int frow = min(frt * RW + wave * (R * 16) + (lane & (R * 16 - 1)), M - 1);
        warm0 = *reinterpret_cast<const uint32_t *>(u + ((int64_t)fi * M + frow) * K);
    }
    produce_write(0);
    __syncthreads();
    asm volatile("" ::"v"(warm0));                  // keeps the load; by now it has long arrived

    // ---- steady state -------------------------------------------------------
    int buf = 0;
    uint32_t warm_in = 0;
    for (int unit = u_begin; unit + 1 < u_end; unit++) {
        const bool crossing = c + 1 == nch;         // the next unit starts another row
        const int cn = crossing ? 0 : c + 1;
        if (crossing) {
            // the row ends with this unit: pull its u rows towards L2 now (one
            // dword per row, value unused) so the flush below does not wait on HBM
            const int fi = rowid / row_tiles, frt = rowid % row_tiles;
            const int frow = min(frt * RW + wave * (R * 16) + (lane & (R * 16 - 1)), M - 1);
            warm_in = *reinterpret_cast<const uint32_t *>(u + ((int64_t)fi * M + frow) * K);
            set_row(rowid + 1);                     // address arithmetic only
        }
        produce_issue(chunk_of(cn));                // L2-resident: first, so waiting for them does not wait for HBM
        load_signs(nxt, chunk_of(cn));
        __builtin_amdgcn_sched_barrier(0);          // keep the prefetch at the top of the unit
        consume(cur, buf);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::"v"(warm_in));              // keeps the load alive; waited for only here, behind the MFMA loop
        produce_write(buf ^ 1);
        __syncthreads();
        if (crossing) {
            flush(rowid, true);
            rowid++;
        }
#pragma unroll
        for (int jr = 0; jr < R; jr++) cur[jr] = nxt[jr];
        c = cn;
        buf ^= 1;
    }
    // ---- drain: last unit, nothing left to prefetch -----------------------------
    consume(cur, buf);
    flush(rowid, u_end % nch == 0);
}

// y[t, off + m] = epilogue( fp16( sum_i sum_k part[i, k, t, m] + bias[m] ) ): every one of the I * kmax
// slots of an output holds a number (the decode kernels zero-fill the slots nobody needed; the strip
// kernels write one partial per strip group, I = groups and kmax = 1), added up in a fixed order.
// Epilogues (applied to the fp16-rounded sums, the way separate fp16 ops would):
//   EPI_NONE      the matrices' outputs side by side in one row of `ldy` halves
//   EPI_RESIDUAL  the same plus residual[t, off + m]
//   EPI_SWIGLU    two matrices of equal M: silu(first) * second, one row of M
constexpr int RED_MAXBLOCKS = 1024;      // a sanity limit on the block count

struct RedMat {
    const float *part;
    const half_t *bias;
    int I, M, kmax, y_off, first_block;
};
struct RedGroup {
    RedMat m[GEMV_MAX_GROUP];
    int n, mode;
    // input RMS scale: when xin is set, every sum is multiplied by rsqrt(mean(xin[t, :]^2) + eps)
    // before the bias - the scalar half of an RMSNorm in front of the matrices (its weight
    // vector belongs folded into vt by the caller)
    const half_t *xin;
    int n_in;
    float eps;
    // the same scale from ready-made partial sums of squares, ssq[g * T + t] for g < ssq_n
    // (written by the strip kernel); takes precedence over xin
    const float *ssq;
    int ssq_n;
};

// No slot counts, no divisions, and the loads of a thread depend on nothing but its index, so the
// kernel is one memory round trip long.  A workgroup produces 256 / SL consecutive outputs of one
// token; SL threads per output take every SL-th of the I * kmax slots (SL = 1: no LDS, no barrier).
// SCALED: the input RMS scale of RedGroup::xin or RedGroup::ssq.
constexpr int FLAT_BATCH = 8, RED_WIDE = 1024;     // (RED_WIDE: outputs per workgroup of gemv_reduce_wide_kernel)
template <int SL>
__device__ __forceinline__ float flat_slice_sum(const RedMat &r, int T, int t, int m, int ks) {
    const int total = r.I * r.kmax;
    const int64_t stride = (int64_t)T * r.M;
    const float *base = r.part + (int64_t)t * r.M + m;
    float acc = 0.f;
    for (int s0 = ks; s0 < total; s0 += FLAT_BATCH * SL) {
        float v[FLAT_BATCH];
#pragma unroll
        for (int j = 0; j < FLAT_BATCH; j++) {
            const int s = s0 + j * SL;
            v[j] = base[(int64_t)(s < total ? s : 0) * stride];
        }
#pragma unroll
        for (int j = 0; j < FLAT_BATCH; j++) acc += (s0 + j * SL < total) ? v[j] : 0.f;
    }
    return acc;
}

// this wave's share of a workgroup's sum of squares of the input
__device__ __forceinline__ float input_squares(const RedGroup &grp, int T, int t) {
    float q = 0.f;
    if (grp.ssq) {                               // sums of squares per strip group, left by the strip kernel
        for (int c = threadIdx.x; c < grp.ssq_n; c += 256) q += grp.ssq[c * T + t];
    } else {
        const half_t *xr = grp.xin + (int64_t)t * grp.n_in;
        for (int c = threadIdx.x * 8; c < grp.n_in; c += 256 * 8) {
            const half8_t v = *reinterpret_cast<const half8_t *>(xr + c);
#pragma unroll
            for (int e = 0; e < 8; e++) q += (float)v[e] * (float)v[e];
        }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) q += __shfl_xor(q, o, 64);
    return q;
}
__device__ __forceinline__ half_t swiglu(float a0, float a1) {
    const float gate = (float)(half_t)a0, up = (float)(half_t)a1;
    const half_t act = (half_t)(gate / (1.f + __expf(-gate)));
    return (half_t)((float)act * up);
}

template <int SL, bool SCALED>
__global__ __launch_bounds__(256) void gemv_reduce_flat_kernel(
    const RedGroup grp, const half_t *__restrict__ residual, half_t *__restrict__ y, int T, int ldy) {
    constexpr int RUN = 256 / SL;
    __shared__ float red[2][SL][RUN];
    __shared__ float ssq[4];
    const int lo = threadIdx.x % RUN, ks = threadIdx.x / RUN;
    const bool two = grp.mode == EPI_SWIGLU;
    int j = 0;
    if (!two) {
#pragma unroll
        for (int q = 1; q < GEMV_MAX_GROUP; q++)
            if (q < grp.n && (int)blockIdx.x >= grp.m[q].first_block) j = q;
    }
    const RedMat &r = grp.m[j];
    const int local = blockIdx.x - r.first_block;
    const int per_t = (r.M + RUN - 1) / RUN;
    const int t = local / per_t, m = (local - t * per_t) * RUN + lo;
    const bool live = m < r.M;
    // everything this thread reads is requested before anything is waited for
    float s0 = live ? flat_slice_sum<SL>(r, T, t, m, ks) : 0.f;
    float s1 = (two && live) ? flat_slice_sum<SL>(grp.m[1], T, t, m, ks) : 0.f;
    float extra0 = 0.f, extra1 = 0.f, res = 0.f;
    if (ks == 0 && live) {
        if (r.bias) extra0 = (float)r.bias[m];
        if (two && grp.m[1].bias) extra1 = (float)grp.m[1].bias[m];
        if (grp.mode == EPI_RESIDUAL) res = (float)residual[(int64_t)t * ldy + r.y_off + m];
    }
    float scale = 1.f;
    if (SCALED) {
        const float q = input_squares(grp, T, t);
        if ((threadIdx.x & 63) == 0) ssq[threadIdx.x >> 6] = q;
    }
    if (SL > 1) {
        red[0][ks][lo] = s0;
        if (two) red[1][ks][lo] = s1;
    }
    if (SL > 1 || SCALED) __syncthreads();
    if (SCALED) scale = rsqrtf((ssq[0] + ssq[1] + ssq[2] + ssq[3]) / (float)grp.n_in + grp.eps);
    if (ks != 0 || !live) return;
    if (SL > 1) {
        s0 = 0.f;
        s1 = 0.f;
#pragma unroll
        for (int k = 0; k < SL; k++) s0 += red[0][k][lo];
        if (two) {
#pragma unroll
            for (int k = 0; k < SL; k++) s1 += red[1][k][lo];
        }
    }
    const float a0 = s0 * scale + extra0;
    if (two) {
        const float a1 = s1 * scale + extra1;
        y[(int64_t)t * ldy + m] = swiglu(a0, a1);
    } else {
        half_t v = (half_t)a0;
        if (grp.mode == EPI_RESIDUAL) v = (half_t)(res + (float)v);
        y[(int64_t)t * ldy + r.y_off + m] = v;
    }
}

// The same sums in the same order (above FLAT_BATCH slots even and odd ones apart), four neighbouring outputs per thread (16-byte loads, 8-byte stores) and a token per
// blockIdx.y: for many outputs of up to 16 slots, where a thread per output is bound by its own index arithmetic (14336 x 100 outputs of four slots: 7 us, VALU 62 % of
// the cycles).  Now memory.  S: most slots of a matrix.  us of a call, flat / this: 28672 x 8192, 3 blocks, 80 tokens 109.7 / 104.9, 14336 x 4096, 5, 100 58.4 / 56.2, 8, 24 52.2 / 50.4,
// 5000 x 4096, 6, 37 26.5 / 26.0, 10240 x 1024, 4, 16 15.2 / 14.4, 2048 x 2048, 3, 64 13.9 / 13.4, 28672 x 4096, 2, 5 (140 workgroups) 28.8 / 28.6.
template <int S, bool SCALED>
__global__ __launch_bounds__(256) void gemv_reduce_wide_kernel(const RedGroup grp, const half_t *__restrict__ residual, half_t *__restrict__ y, int T, int ldy) {
    __shared__ float ssq[4];
    const bool two = grp.mode == EPI_SWIGLU;
    int j = 0;
    if (!two) {
#pragma unroll
        for (int q = 1; q < GEMV_MAX_GROUP; q++)
            if (q < grp.n && (int)blockIdx.x >= grp.m[q].first_block) j = q;
    }
    const RedMat &r = grp.m[j];
    const int t = blockIdx.y, m = ((int)blockIdx.x - r.first_block) * RED_WIDE + 4 * threadIdx.x;
    const bool live = m < r.M;
    const int at = live ? m : 0;
    auto sums = [&](const RedMat &mat) {
        const int total = mat.I * mat.kmax;
        const float *base = mat.part + (int64_t)t * mat.M + at;
        float4_t v[S];
#pragma unroll
        for (int k = 0; k < S; k++) v[k] = *reinterpret_cast<const float4_t *>(base + (int64_t)min(k, total - 1) * T * mat.M);
        float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int k = 0; k < S; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) acc[S > FLAT_BATCH ? k & 1 : 0][e] += k < total ? v[k][e] : 0.f;
        if (S > FLAT_BATCH) {
#pragma unroll
            for (int e = 0; e < 4; e++) acc[0][e] = acc[0][e] + acc[1][e];
        }
        return acc[0];
    };
    const float4_t s0 = sums(r), s1 = two ? sums(grp.m[1]) : (float4_t){0.f, 0.f, 0.f, 0.f};
    const half4_t none = {(half_t)0, (half_t)0, (half_t)0, (half_t)0};
    half4_t bias0 = none, bias1 = none, res = none;
    if (r.bias) bias0 = *reinterpret_cast<const half4_t *>(r.bias + at);
    if (two && grp.m[1].bias) bias1 = *reinterpret_cast<const half4_t *>(grp.m[1].bias + at);
    half_t *const to = y + (int64_t)t * ldy + (two ? 0 : r.y_off) + at;
    if (grp.mode == EPI_RESIDUAL) res = *reinterpret_cast<const half4_t *>(residual + (int64_t)t * ldy + r.y_off + at);
    float scale = 1.f;
    if (SCALED) {
        const float q = input_squares(grp, T, t);
        if ((threadIdx.x & 63) == 0) ssq[threadIdx.x >> 6] = q;
        __syncthreads();
        scale = rsqrtf((ssq[0] + ssq[1] + ssq[2] + ssq[3]) / (float)grp.n_in + grp.eps);
    }
    half4_t out;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const float a0 = s0[e] * scale + (float)bias0[e];
        if (two) {
            const float a1 = s1[e] * scale + (float)bias1[e];
            out[e] = swiglu(a0, a1);
        } else {
            half_t v = (half_t)a0;
            if (grp.mode == EPI_RESIDUAL) v = (half_t)((float)res[e] + (float)v);
            out[e] = v;
        }
    }
    if (live) *reinterpret_cast<half4_t *>(to) = out;
}

template <int SL>
void launch_reduce_flat(int blocks, const RedGroup &r, const half_t *residual, half_t *y, int T, int ldy, hipStream_t s) {
    if (r.xin || r.ssq)
        gemv_reduce_flat_kernel<SL, true><<<blocks, 256, 0, s>>>(r, residual, y, T, ldy);
    else
        gemv_reduce_flat_kernel<SL, false><<<blocks, 256, 0, s>>>(r, residual, y, T, ldy);
}

// Whether the four-at-a-time kernel takes the sums, and its launch: `slots` at most 16, sizes and addresses of whole fours, a workgroup for every other CU, and four times as many
// where an output is made of two sums (2 x 28672 rows, 8 tokens, 224 workgroups, flat / this: 8 slots 5.5 / 5.7 us, 16 slots 6.2 / 7.3).
constexpr int64_t RED_WIDE_MIN = 128;
bool launch_reduce_wide(int slots, const RedGroup &r, const half_t *residual, half_t *y, int T, int ldy, hipStream_t s) {
    RedGroup g = r;
    int blocks = 0;
    bool fours = slots <= 2 * FLAT_BATCH && bs_aligned(y, 8) && bs_aligned(residual, 8) && ldy % 4 == 0 && T <= 65535;
    for (int j = 0; j < r.n; j++) {
        const RedMat &m = r.m[j];
        fours = fours && m.M % 4 == 0 && m.y_off % 4 == 0 && bs_aligned(m.bias, 8) && bs_aligned(m.part, 16);
        g.m[j].first_block = blocks;
        if (r.mode != EPI_SWIGLU || j == 0) blocks += (int)bs_cdiv(m.M, RED_WIDE);
    }
    if (!fours || (int64_t)blocks * T < RED_WIDE_MIN * (r.mode == EPI_SWIGLU ? 4 : 1)) return false;
    const bool scaled = r.xin || r.ssq;
    const dim3 grid(blocks, T);
    switch (slots <= 8 ? slots : slots <= 12 ? 12 : 16) {
#define RED_CASE(k) \
    case k: \
        if (scaled) gemv_reduce_wide_kernel<k, true><<<grid, 256, 0, s>>>(g, residual, y, T, ldy); \
        else gemv_reduce_wide_kernel<k, false><<<grid, 256, 0, s>>>(g, residual, y, T, ldy); \
        break;
        RED_CASE(1) RED_CASE(2) RED_CASE(3) RED_CASE(4) RED_CASE(5) RED_CASE(6) RED_CASE(7) RED_CASE(8) RED_CASE(12) RED_CASE(16)
#undef RED_CASE
        default: return false;
    }
    return true;
}

struct Plan {
    int waves, R, n_chunks, grid, n, pair;
    int mx;        // 1: the block-scaled fp4 x fp6 kernel (gemv_mx.hip), units of MX_UNIT_COLS columns
    int sparse;    // 1: the sparse kernel (gemv_sparse.hip)
    double us;     // ... of it: what the choice of R takes a call for, partial sums left out
    int row_tiles[GEMV_MAX_GROUP], kmax[GEMV_MAX_GROUP], first_wg[GEMV_MAX_GROUP];
    Split sp[GEMV_MAX_GROUP];
    int64_t part_off[GEMV_MAX_GROUP];      // in floats; part_off[n] = total
    int64_t part_total;
};

// One instantiation and one grid for the whole group; every matrix gets a share of
// the workgroups in proportion to its units.
// Which kernel a call of one to four tokens runs on: 0 by shape, 1 always gemv_kernel, 2 for one and two tokens the block-scaled one
// wherever it takes the shape (bs_set_decode_kernel, for tests and benchmarks).  Per calling thread: a size query
// and the forward behind it on one thread agree whatever other threads set.
thread_local int g_decode_kernel = 0;

int most_sparse_sums(const int *I, const int *M, int n, int N);
// Rows per workgroup of the block-scaled kernel for these matrices (0: it does not run them).
int mx_rows_per_tile(const int *I, const int *M, int n, int N, int K, int T) {
    if (g_decode_kernel == 1 || !bs_gemv_mx_takes(N, K, 1, T)) return 0;
    const int n_units = (int)bs_cdiv(N, MX_UNIT_COLS / T);
    int pick = 0;
    for (int r = 4; r >= 1; r >>= 1) {
        const int rw = 8 * r * 16;
        bool tall = true;
        int64_t units = 0;
        for (int j = 0; j < n; j++) {
            tall = tall && M[j] >= rw;
            units += bs_cdiv(M[j], rw) * I[j] * n_units;
        }
        if ((tall && units >= 256) || r == 1) { pick = r; break; }
    }
    if (g_decode_kernel == 2) return pick;
    // by shape: the long-stack cases, where the contraction loop and not the fixed cost of a launch decides
    int64_t bytes = 0;
    for (int j = 0; j < n; j++) bytes += (int64_t)I[j] * M[j] * (N / 8);
    if (pick < 2) return 0;
    if (bytes >= (T == 1 ? MX_MIN_SIGN_BYTES : MX_MIN_SIGN_BYTES_TWO)) return pick;
    return T == 1 && bytes >= MX_MIN_SIGN_BYTES_MANY_SUMS && most_sparse_sums(I, M, n, N) >= MX_MANY_SUMS ? pick : 0;
}

// The grid of the block-scaled and the sparse kernel: one workgroup of 8 waves, 128 R rows, per CU.
void one_per_cu(Plan &p, const int *I, const int *M, int T) {
    const int n = p.n;
    p.waves = 8;
    p.pair = 0;
    int units[GEMV_MAX_GROUP], total = 0, biggest = 0;
    for (int j = 0; j < n; j++) {
        p.row_tiles[j] = (int)bs_cdiv(M[j], 8 * p.R * 16);
        units[j] = I[j] * p.row_tiles[j] * p.n_chunks;
        total += units[j];
        if (units[j] > units[biggest]) biggest = j;
    }
    int grid = total < 256 ? total : 256, gj[GEMV_MAX_GROUP], sum = 0;
    for (int j = 0; j < n; j++) {
        gj[j] = n == 1 ? grid : (int)(((int64_t)grid * units[j] + total / 2) / total);
        if (gj[j] < 1) gj[j] = 1;
        if (gj[j] > units[j]) gj[j] = units[j];
        sum += gj[j];
    }
    while (sum > grid && gj[biggest] > 1) { gj[biggest]--; sum--; }
    int first = 0;
    int64_t off = 0;
    for (int j = 0; j < n; j++) {
        p.first_wg[j] = first;
        first += gj[j];
        p.sp[j].q = units[j] / gj[j];
        p.sp[j].rem = units[j] % gj[j];
        int kmax = (int)bs_cdiv(p.n_chunks - 1, p.sp[j].q) + 1;
        if (kmax > gj[j]) kmax = gj[j];
        p.kmax[j] = kmax;
        p.part_off[j] = off;
        off += (int64_t)I[j] * kmax * T * M[j];
    }
    p.grid = first;
    p.part_total = off;
}

// mx_r: what mx_rows_per_tile says, where the caller has asked already.
void make_plan(Plan &p, const int *I, const int *M, int n, int N, int K, int T, int mx_r = -1) {
    p.n = n;
    p.n_chunks = N / CH;
    p.mx = p.sparse = 0;
    if (mx_r < 0) mx_r = mx_rows_per_tile(I, M, n, N, K, T);
    if (mx_r > 0) {
        // units are (block, row tile, 1024 columns), never paired
        p.mx = 1;
        p.R = mx_r;
        p.n_chunks = (int)bs_cdiv(N, MX_UNIT_COLS / T);
        one_per_cu(p, I, M, T);
        return;
    }
    // gemv_kernel.  By shape it has four tokens where the tile kernel declines, the passes of two to four that five to eight tokens are cut into where the strip
    // kernel declines, one token below a MiB of sign bytes (64-row tiles), and what the sparse kernel's offsets or scratch do not allow.  Otherwise one to three
    // tokens run here under bs_set_decode_kernel only, so do one token's taller tiles, pairs and 16 waves.
    // Rows per workgroup: 512 (8 waves x 4 tiles), 256, 128, 64; resident workgroups per CU.
    // Three or four tokens need more than the 128 registers a lane has with two 8-wave
    // workgroups per CU: there it is one workgroup of 8 waves per CU (two waves per SIMD
    // to overlap sign decode and MFMA), four row tiles per wave (each Z fragment read
    // from LDS feeds four MFMAs per token) or two when the layer has too few units.
    const int cand1[4][3] = {{8, 4, 2}, {4, 4, 3}, {4, 2, 4}, {4, 1, 4}};
    const int wide1[3] = {16, 4, 1};
    const int cand3[4][3] = {{8, 4, 1}, {8, 2, 1}, {4, 2, 1}, {4, 1, 1}};
    const int cand2[4][3] = {{8, 2, 2}, {4, 4, 2}, {4, 2, 2}, {4, 1, 2}};
    const int (*cand)[3] = T > 2 ? cand3 : T == 2 ? cand2 : cand1;
    int pick = 3;
    for (int k = 0; k < 4; k++) {
        const int rw = cand[k][0] * cand[k][1] * 16;
        bool tall = true;
        int64_t units = 0;
        for (int j = 0; j < n; j++) {
            tall = tall && M[j] >= rw;
            units += bs_cdiv(M[j], rw) * I[j] * p.n_chunks;
        }
        // enough units that every CU gets one
        if (tall && units >= 256) { pick = k; break; }
    }
    // One token, long stacks (under BS_DECODE_F16): one workgroup of 16 waves per CU.  Two 8-wave workgroups on a CU do
    // not share it evenly (the older one is served first and finishes a third earlier, the
    // younger one then runs on a half-empty CU); sixteen waves that meet at one barrier do.
    const int *choice = cand[pick];
    if (T == 1) {
        bool tall = true;
        int64_t units = 0;
        for (int j = 0; j < n; j++) {
            tall = tall && M[j] >= 1024;
            units += bs_cdiv(M[j], 1024) * I[j] * p.n_chunks;
        }
        if (tall && units >= GEMV_WIDE_MIN_UNITS) choice = wide1;
    }
    p.waves = choice[0];
    p.R = choice[1];
    int units[GEMV_MAX_GROUP], total = 0;
    for (int j = 0; j < n; j++) {
        p.row_tiles[j] = (int)bs_cdiv(M[j], p.waves * p.R * 16);
        units[j] = I[j] * p.row_tiles[j] * p.n_chunks;
        total += units[j];
    }
    int grid = 256 * (T == 1 ? choice[2] : T == 2 ? 2 : 1);
    // prefer two units per workgroup (one pipeline fill amortised over two units) as
    // long as every CU still gets a workgroup
    if (grid > total / 2) grid = total / 2 >= 256 ? total / 2 : (total < 256 ? total : 256);
    if (grid < 1) grid = 1;
    // Paired workgroups (GemvMat::pair) once a workgroup has several units to stream: the
    // grid is then a multiple of 16, so that the contiguous run of workgroups an XCD gets
    // starts and ends on a pair.
    p.pair = (p.n_chunks % 2 == 0 && total >= GEMV_PAIR_MIN_UNITS * grid && grid >= 16 * n) ? 1 : 0;
    int gj[GEMV_MAX_GROUP], sum = 0, biggest = 0;
    for (int j = 0; j < n; j++) {
        gj[j] = n == 1 ? grid : (int)(((int64_t)grid * units[j] + total / 2) / total);
        if (p.pair) gj[j] &= ~1;
        if (gj[j] < 1 + p.pair) gj[j] = 1 + p.pair;
        if (gj[j] > units[j]) gj[j] = units[j];
        sum += gj[j];
        if (units[j] > units[biggest]) biggest = j;
    }
    if (p.pair) {
        // round the grid to a multiple of 16 on the largest matrix (down when it can spare them)
        const int over = sum % 16;
        if (over && gj[biggest] > over + 16) gj[biggest] -= over;
        else if (over && gj[biggest] + 16 - over <= units[biggest]) gj[biggest] += 16 - over;
        else if (over) p.pair = 0;
        if (!p.pair)      // back to the plain plan
            for (int j = 0; j < n; j++) {
                gj[j] = n == 1 ? grid : (int)(((int64_t)grid * units[j] + total / 2) / total);
                if (gj[j] < 1) gj[j] = 1;
                if (gj[j] > units[j]) gj[j] = units[j];
            }
    }
    if (!p.pair && n > 1) {
        // rounding per matrix may leave one workgroup too many: it would wait for a free slot
        // and run after the others (a launch of 513 takes a fifth longer than one of 512)
        sum = 0;
        for (int j = 0; j < n; j++) sum += gj[j];
        while (sum > grid && gj[biggest] > 1) { gj[biggest]--; sum--; }
    }
    int first = 0;
    int64_t off = 0;
    for (int j = 0; j < n; j++) {
        const int places = gj[j] >> p.pair, uj = units[j] >> p.pair, nch = p.n_chunks >> p.pair;
        p.first_wg[j] = first;
        first += gj[j];
        p.sp[j].q = uj / places;
        p.sp[j].rem = uj % places;
        // most places a row of nch units can be spread over
        int kmax = (int)bs_cdiv(nch - 1, p.sp[j].q) + 1;
        if (kmax > places) kmax = places;
        p.kmax[j] = kmax << p.pair;
        p.part_off[j] = off;
        off += (int64_t)I[j] * p.kmax[j] * T * M[j];
    }
    p.grid = first;
    p.part_total = off;
}

// The plan of the sparse kernel where it serves these matrices, for the rules at sparse_plan.
void sparse_plan_of(Plan &p, const int *I, const int *M, int n, int N, int T) {
    p.n = n;
    p.mx = 0;
    p.sparse = 1;
    p.n_chunks = (int)bs_cdiv(N, CH);
    // Row tiles per wave by the time of the busiest workgroup (us, a replayed graph, the summing launch included): what a call with one unit per workgroup takes
    // and what each further unit adds, fitted to 33 shapes (4096 x 11008, 4 blocks, one token, R = 1, 2, 4: 21.8, 18.3, 17.7; 1024 x 4096, 3 blocks 7.2, 7.8, 8.7;
    // 20000 x 1408, 2 blocks 12.1, 10.8, 9.0; 6144 x 4096, 6 blocks, two tokens 22.6, 20.4, 21.9).
    static const double base[3][3] = {{5.25, 5.45, 5.9}, {5.7, 5.9, 5.8}, {5.5, 5.85, 6.0}}, unit[3][3] = {{1.18, 1.45, 2.0}, {1.43, 2.0, 3.56}, {1.95, 2.68, 5.03}};
    double best = 0;
    for (int k = 0; k < 3; k++) {
        int64_t units = 0;
        for (int j = 0; j < n; j++) units += bs_cdiv(M[j], 128 << k) * I[j] * p.n_chunks;
        const double us = base[T - 1][k] + unit[T - 1][k] * bs_cdiv(units, 256);
        if (k == 0 || us < best) {
            best = us;
            p.R = 1 << k;
        }
    }
    p.us = best;
    one_per_cu(p, I, M, T);
}

// Most partial sums per output that the sparse kernel leaves of one token.
int most_sparse_sums(const int *I, const int *M, int n, int N) {
    Plan p;
    sparse_plan_of(p, I, M, n, N, 1);
    int most = 0;
    for (int j = 0; j < n; j++) most = std::max(most, I[j] * p.kmax[j]);
    return most;
}

// us of one matrix's call on the sparse kernel, and on the tile and strip kernels (estimates for the choice between them, fitted to 900 calls on rotating
// sizes, each within 4 to 5 % as a rule, the strip kernel's 8).  The summing launch adds a slot in 7 to 9 ns: few rows of many columns have hundreds.
double sparse_call_us(const Plan &p, int I, int T) {
    static const double c[3][4] = {{-2.53, 1.388, 0.0071, 0.138}, {-2.67, 1.357, 0.0082, 0.315}, {-2.47, 1.302, 0.0092, 0.206}};
    const double *k = c[T - 1];
    return k[0] + k[1] * p.us + k[2] * I * p.kmax[0] - k[3] * std::max(0., p.us - 15.);
}
double tile_call_us(double cycles, int groups, int N, int T) {
    const double width = groups == bs_cdiv(N, 256) ? 0.8 : groups == bs_cdiv(N, 512) ? 1. : 1.08;        // (columns per workgroup: narrow ones cost less than the plan's cycles say)
    return T < 3 ? 5.34 + 3.98e-4 * width * cycles : 4.99 + 4.76e-4 * width * cycles;
}
double strip_call_us(long steps, int I) { return 6.8 + steps * (0.271 + 0.381 * I); }

struct GroupArgs {          // host-side view of one call
    int n;
    const uint8_t *packed[GEMV_MAX_GROUP];
    const half_t *u[GEMV_MAX_GROUP], *vt[GEMV_MAX_GROUP], *bias[GEMV_MAX_GROUP];
    int I[GEMV_MAX_GROUP], M[GEMV_MAX_GROUP];
};

template <int T, int WAVES, int R>
int launch_one(const Plan &p, const GemvGroup &grp, const half_t *x, int N, int K, hipStream_t s) {
    const size_t lds = (size_t)2 * T * 16384 + (size_t)2 * WAVES * T * 64;
    static bs_lds_grant granted[BS_MAX_DEVICES];      // per instantiation
    const int st = bs_allow_lds((const void *)gemv_kernel<T, WAVES, R>, lds, granted);
    if (st != BS_OK) return st;
    gemv_kernel<T, WAVES, R><<<p.grid, 64 * WAVES, lds, s>>>(grp, x, N, K, p.n_chunks);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

// Only the (WAVES, R) pairs make_plan can choose for T tokens exist; any other pair is refused
// rather than run on a tile of another height (the reduce kernel and the partial layout are
// built for exactly waves * R * 16 rows per tile).
template <int T>
int launch_T(const Plan &p, const GemvGroup &grp, const half_t *x, int N, int K, hipStream_t s) {
    const int w = p.waves, r = p.R;
    if constexpr (T == 1) {
        if (w == 16 && r == 4) return launch_one<1, 16, 4>(p, grp, x, N, K, s);
        if (w == 8 && r == 4) return launch_one<1, 8, 4>(p, grp, x, N, K, s);
    } else if constexpr (T == 2) {
        if (w == 8 && r == 2) return launch_one<2, 8, 2>(p, grp, x, N, K, s);
    } else {
        if (w == 8 && r == 4) return launch_one<T, 8, 4>(p, grp, x, N, K, s);
        if (w == 8 && r == 2) return launch_one<T, 8, 2>(p, grp, x, N, K, s);
    }
    if constexpr (T <= 2) {
        if (w == 4 && r == 4) return launch_one<T, 4, 4>(p, grp, x, N, K, s);
    }
    if (w == 4 && r == 2) return launch_one<T, 4, 2>(p, grp, x, N, K, s);
    if (w == 4 && r == 1) return launch_one<T, 4, 1>(p, grp, x, N, K, s);
    return BS_ERR_SHAPE;
}

// per-block byte offsets, of signs and of vt, are kept in 32 bits inside the kernels
bool block_fits(int I, int M, int N, int K) {
    return I >= 1 && I <= RED_MAXBLOCKS && M >= 1 && (int64_t)M * N < ((int64_t)1 << 31) && (int64_t)K * N * 2 < ((int64_t)1 << 32);
}
bool gemv_shape_ok(int I, int M, int N, int K, int T) { return block_fits(I, M, N, K) && T >= 1 && T <= 8 && N % CH == 0; }

// Tokens are processed in passes of at most four (LDS holds Z for four tokens).
int pass_tokens(int T) { return T <= 4 ? T : (T + 1) / 2; }

// From this many tokens on the strip kernel (weight patches rebuilt in registers and
// multiplied at once) is faster than passes of the factor-through kernel, which needs 16
// rank-MFMAs per token and patch where the strip kernel needs one for 16 tokens.
constexpr int STRIP_MIN_T = 5, STRIP_MAX_T = BS_PANEL_MAX_T;       // (49 tokens and more: the walked and panel kernels, single matrices only)

bool strip_group_ok(const int *I, const int *M, int n, int N, int K, int T) {
    for (int j = 0; j < n; j++)
        if (bs_strip_partials(I[j], M[j], N, K, T) == 0) return false;
    return true;
}
bool gemv_group_ok(const int *I, const int *M, int n, int N, int K, int T) {
    for (int j = 0; j < n; j++)
        if (!gemv_shape_ok(I[j], M[j], N, K, T)) return false;
    return true;
}
// 1: strip kernel, 0: factor-through kernel (either may leave the call to the sparse kernel, see sparse_plan), -1: neither takes the shapes
int group_path(const int *I, const int *M, int n, int N, int K, int T) {
    if (n < 1 || n > GEMV_MAX_GROUP) return -1;
    if (T >= STRIP_MIN_T && T <= STRIP_MAX_T && strip_group_ok(I, M, n, N, K, T)) return 1;
    if (gemv_group_ok(I, M, n, N, K, T)) return 0;
    // One to four tokens on column counts that are multiples of 128 but not of 512, of which sparse_plan takes most at one and two: the tile and strip kernels
    // round the weight to fp16 once and multiply with fp32 sums, as the rebuild and the dense product do that such shapes would take otherwise, and no less
    // exactly (error against float64 within 0.05 % of theirs: 11 shapes, three decomposed weights, 1, 2 and 4 tokens).  gemv_kernel would round vt * x: 7 %
    // further from float64 with 2 blocks of 11008 columns (2.94e-4 against 2.75e-4), 11 % on the block-scaled one.  us rebuild / strip, one token: 4096 x
    // 11008, 1 block 52 / 14, 4 blocks 72 / 28, 8 blocks 91 / 47; 2048 x 5504, 3 blocks 32 / 12; 8192 x 3200, 4 blocks 40 / 21.
    return N % CH != 0 && T < STRIP_MIN_T && strip_group_ok(I, M, n, N, K, T) ? 1 : -1;
}
int64_t tile_part_floats(const int *I, const int *M, int n, int N, int K, int T, double *cycles = nullptr) {
    int groups[GEMV_MAX_GROUP];
    if (!bs_tile_partials(I, M, n, N, K, T, groups, cycles)) return 0;
    int64_t total = (int64_t)groups[0] * T;
    for (int j = 0; j < n; j++) total += (int64_t)groups[j] * T * M[j];
    return total;
}
// Three and four tokens: the factor-through kernel needs 16 products per sign and token, the tile kernel one weight for all of them.  It takes them with
// the weight in two fp16 terms, so that only y is rounded (error against float64 0.7 of the other's).  us, factor-through / tiles:
//   4 tokens: 4096 x 14336, 4 blocks 38.4 / 35.5; 14336 x 4096, 8 60.5 / 47.1; 4096 x 4096, 3 17.3 / 15.3, 2 11.3 / 11.8; 14720 x 11776, 2 50.4 / 56.2; 2288 x 7168, 6 26.8 / 19.6
//   3 tokens: 14336 x 4096, 8 49.3 / 47.3, 5 37.2 / 35.8, 3 26.6 / 27.1; 4096 x 14336, 4 30.3 / 33.7; 4096 x 4096, 3 14.9 / 15.3, 2 9.9 / 11.7; 7605 x 2560, 2 15.6 / 15.5
// (over drawn shapes 1.27 and 1.12 on average, 1 and 8 % of them more than 5 % behind)
// and below a MiB of sign bytes both are a chain of latencies (366 x 512, 14 blocks, 3 tokens 8.3 / 10.6; 1536 x 512, 4, 4 tokens 8.9 / 7.7).
// Neither where a single workgroup has more than 50,000 cycles per token of it: the factor-through kernel streams there (us: 5114 x 27136, 6 blocks, 3 tokens
// 83.9 / 104; 23 drawn shapes at three tokens 0.94 of its rate, from 120,000 to 150,000 cycles 1.02; 11 at four 0.89 and 1.12).  Nor a group
// of three tokens from 16,000 cycles on up to 8 MiB of sign bytes in all, which the factor-through kernel has in one round (2 x 8192 x 2048,
// 2 blocks 14.2 / 18.2; 240 of 986 drawn groups, 0.95 on average; the others 1.05).
// (What a group's matrices do alone is another matter: make_tile_plan compares single ones with the strip kernel too.)
// Nor three tokens of one matrix with 4096 columns or more where the sparse kernel is the faster one by the estimates above (us tile / sparse: 4096 x 4096, 4 blocks 16.6 /
// 13.1, 8 23.1 / 19.9; 1024 x 4096, 3 10.0 / 7.9; but 144 x 26112, 8 11.1 / 17.1, 260 x 30208, 8 16.3 / 24.2, 4882 x 8192, 10 41.5 / 45.3.  Of 237 drawn calls, half of them of
// up to 1000 rows, 8 are more than 3 % behind the tile kernel, 7 % at worst; all of them on the sparse kernel: 85, 55 %).
// (sparse: its plan, where it serves the call)
bool split_tiles(const int *I, const int *M, int n, int N, int K, int T, const Plan *sparse) {
    if ((T != 3 && T != 4) || K != 16 || g_decode_kernel != 0) return false;
    int64_t bytes = 0;
    for (int j = 0; j < n; j++) {
        const bool large = (int64_t)M[j] * N > (24ll << 20);
        bytes += (int64_t)I[j] * M[j] * (N / 8);
        if (I[j] < 2 || (int64_t)I[j] * M[j] * (N / 8) < (1 << 20)) return false;
        if ((T == 3 && large && I[j] < 6) || (I[j] == 2 && N >= 4096)) return false;
    }
    // (never with more partial sums than bs_forward_static's scratch holds: long stacks take 256 columns per workgroup, 16 blocks of 17317 x 111104, 3 tokens 86 MiB
    // where the factor-through kernel needs 6)
    double cycles;
    const int64_t floats = tile_part_floats(I, M, n, N, K, T, &cycles);
    if (floats == 0 || floats * (int64_t)sizeof(float) > BS_STATIC_SCRATCH_BYTES) return false;
    if (T == 3 && n == 1 && N >= 4096 && sparse && sparse_call_us(*sparse, I[0], T) <= tile_call_us(cycles, (int)(floats / T / (M[0] + 1)), N, T)) return false;
    return cycles <= 50000. * T && !(T == 3 && n > 1 && bytes <= (8 << 20) && cycles > 16000.);
}
// The sparse kernel's plan where it serves the call; false: another kernel does.
//   N % 512 == 0: one to three tokens in the place of gemv_kernel.  us gemv_kernel / sparse, one token: 1024 x 4096, 3 blocks 8.1 / 7.2, 4096 x 4096, 2 8.6 / 7.8, 14336 x 4096, 1
//     10.7 / 9.1 (below a MiB of sign bytes either is a chain of latencies, gemv_kernel's the shorter one: 355 x 2560, 4 6.3 / 6.9, 308 x 3584, 5 6.9 / 7.1); two: 1024 x 4096, 3 10.4 / 7.6, 4096 x 4096, 1 8.9 / 7.7, 14336 x 4096, 1 13.1 / 10.8; three: 4096 x 14336, 16 87.5 / 83.4, 3
//     31.1 / 27.8, 28672 x 8192, 2 52.0 / 47.6, 1024 x 4096, 1 8.6 / 7.4.  Four: 4096 x 14336, 16 104 / 116, 28672 x 8192, 2 58.6 / 64.1: gemv_kernel keeps them.
//   Other multiples of 128 columns, one and two tokens: us tile or strip kernel / sparse, one token: 4096 x 11008, 4 blocks 25.7 / 17.7, 8 39.3 / 25.6, 2 18.3 / 13.0;
//     20000 x 1408, 2 15.6 / 9.0; 2048 x 5504, 3 11.9 / 9.0; two: 24.7 / 22.6, 39.1 / 32.8, 18.5 / 15.5, 15.3 / 10.5, 12.0 / 10.3; three: 24.7 / 27.4, 39.6 / 42.0.  Not
//     where few rows of many columns leave hundreds of partial sums, or up to 256 columns half of a unit empty, and the other kernel is the faster one by the estimates (28 x 27392, 8 blocks, two
//     tokens 8.8 / 12.4; 20204 x 128, 16 15.7 / 20.8).  At rank 16 it starts at half a MiB of sign bytes, though it is ahead below that too (300 drawn calls on the tile kernel 7.3 to 8.1 us, 0.85 of
//     that at one token, 0.9 at two): the tile kernel's tests at one and two tokens are calls of that size.
// Replayed on the same inputs, drawn calls take 0.84 of gemv_kernel's time (351 of one to three tokens, N % 512 == 0; one is more than 3 % behind, 4 %) and 0.75 of the tile and strip kernels' (357 of
// one and two tokens at other column counts; 2, 5 %), groups of two to four matrices 0.76 (214; 1, 7 %).  A call as short as 8 us is bound by the host: 1024 x 4096, 3 blocks, one token by
// BitStackLinear.forward 8.6 / 8.45.  It rounds nothing but y: error against float64 before that rounding 1e-7 to 4e-7 on drawn factors.  (Never with more partial sums than bs_forward_static's
// scratch holds.)
constexpr int64_t SPARSE_MIN_UNEVEN = 512 << 10, SPARSE_MIN_ONE = 1 << 20;
// (path: what group_path says; mx_r: what mx_rows_per_tile says at one to three tokens and N % 512 == 0)
bool sparse_plan(Plan &p, const int *I, const int *M, int n, int N, int K, int T, int path, int mx_r) {
    const bool even = N % CH == 0;
    if (g_decode_kernel != 0 || T > (even ? 3 : 2) || path != (even ? 0 : 1) || !bs_gemv_sparse_takes(N, K, 1, T) || (even && mx_r > 0)) return false;
    int64_t bytes = 0;
    for (int j = 0; j < n; j++) {
        if (!block_fits(I[j], M[j], N, K)) return false;
        bytes += (int64_t)I[j] * M[j] * (N / 8);
    }
    if ((!even && K == 16 && bytes < SPARSE_MIN_UNEVEN) || (even && T == 1 && bytes < SPARSE_MIN_ONE)) return false;
    sparse_plan_of(p, I, M, n, N, T);
    if (p.part_total * (int64_t)sizeof(float) > BS_STATIC_SCRATCH_BYTES) return false;
    if (even || n > 1) return true;
    const int slots = I[0] * p.kmax[0];
    double cycles;
    int groups[GEMV_MAX_GROUP];
    if ((slots >= 64 || p.n_chunks == 1) && bs_tile_partials(I, M, 1, N, K, T, groups, &cycles)) return sparse_call_us(p, I[0], T) <= tile_call_us(cycles, groups[0], N, T);
    return slots < 250 || sparse_call_us(p, I[0], T) <= strip_call_us(bs_strip_steps(I[0], M[0], N, T), I[0]);
}
int64_t strip_part_floats(const int *I, const int *M, int n, int N, int K, int T) {
    int64_t total = (int64_t)bs_strip_partials(I[0], M[0], N, K, T) * T;      // sums of squares of x per strip group
    for (int j = 0; j < n; j++) total += (int64_t)bs_strip_partials(I[j], M[j], N, K, T) * T * M[j];
    // room for the tile kernel's partial sums too: the choice also depends on how u is aligned
    return std::max(total, tile_part_floats(I, M, n, N, K, T));
}

// Everything that a call's sizes decide, worked out once per size query and once per call: a forward of some 8 us is bound by the host.  ns of a size query, every
// kernel's plan and the path asked for where they are needed / once: 1024 x 4096, 3 blocks, one token 106 / 47, 4096 x 11008, 4 blocks 175 / 50, 14336 x 4096, 8 blocks
// 54 / 42; us of a BitStackLinear.forward of the first, a size query and two plans less: 8.8 / 8.45 (8.6 with gemv_kernel alone to plan).
struct CallPlan {
    int path;          // group_path
    bool split;        // three or four tokens on the tile kernel where u's alignment allows it
    bool sparse;       // the sparse kernel, in gemv_kernel's (path 0) or the strip kernel's place (path 1)
    Plan gemv;         // of the first pass, where it is no strips
    int64_t floats;    // scratch
};
void plan_call(CallPlan &c, const int *I, const int *M, int n, int N, int K, int T) {
    c.path = group_path(I, M, n, N, K, T);
    c.split = c.sparse = false;
    c.floats = 0;
    if (c.path < 0) return;
    const int tp = pass_tokens(T), mx_r = c.path == 0 ? mx_rows_per_tile(I, M, n, N, K, tp) : 0;
    c.sparse = sparse_plan(c.gemv, I, M, n, N, K, T, c.path, mx_r);
    if (c.sparse) {
        c.floats = c.gemv.part_total;
    } else if (c.path == 1) {
        c.floats = strip_part_floats(I, M, n, N, K, T);
    } else {
        if (T % tp) {                                // a shorter last pass
            make_plan(c.gemv, I, M, n, N, K, T % tp);
            c.floats = c.gemv.part_total;
        }
        make_plan(c.gemv, I, M, n, N, K, tp, mx_r);
        c.floats = std::max(c.floats, c.gemv.part_total);
    }
    c.split = c.path == 0 && split_tiles(I, M, n, N, K, T, c.sparse ? &c.gemv : nullptr);
    if (c.split) c.floats = std::max(c.floats, tile_part_floats(I, M, n, N, K, T));
}
int64_t scratch_bytes(const CallPlan &c) { return (c.floats * (int64_t)sizeof(float) + 255) / 256 * 256; }

// Strip path: one launch writes part[strip group, t, m] of every matrix; the reduce kernel
// reads that as "one partial per block" with the strip groups in the place of the blocks.
int launch_group_strips(const GroupArgs &a, int N, int K, const half_t *x, int T, int mode, const half_t *residual,
                        half_t *y, bool input_rms, float eps, void *workspace, bool split, hipStream_t s) {
    float *part = (float *)workspace;
    RedGroup r;
    r.n = a.n;
    r.mode = mode;
    r.xin = nullptr;
    r.n_in = N;
    r.eps = eps;
    float *parts[GEMV_MAX_GROUP];
    // The tile kernel (from 49 tokens the column kernel) where it takes the matrices; the strip and panel kernels for ranks below 4, long stacks, small matrices and, at rank 16, u
    // off a 16-byte boundary.  Ranks 4 to 15 have builds of their own of both (us, strip, walked or panel kernel / that, rank 12: 28672 x 8192, 3 blocks, 8 tokens 102.2 / 60.5, 40 tokens 154 / 124;
    // 14336 x 4096, 8, 8 tokens 69.0 / 43.4; 5, 100 tokens 77.6 / 58.4; 5000 x 4096, 6, 37 tokens 39.4 / 27.7; 4096 x 14336, 8, 509 tokens 151.2 / 118.3, rebuild and product).
    int column_groups[GEMV_MAX_GROUP];
    bool tiles = bs_tile_partials(a.I, a.M, a.n, N, K, T, column_groups);
    for (int j = 0; j < a.n; j++) tiles = tiles && bs_aligned(a.u[j], K == 16 ? 16 : 2);
    // threads per output of the summing kernel, as behind the decode kernels (the column groups are its slots)
    int slots = 0;
    for (int j = 0; j < a.n; j++) {
        if (!tiles) column_groups[j] = bs_strip_partials(a.I[j], a.M[j], N, K, T);
        const int groups = column_groups[j];
        if (groups > slots) slots = groups;
    }
    const int sl = slots <= FLAT_BATCH ? 1 : slots <= 2 * FLAT_BATCH ? 2 : slots <= 4 * FLAT_BATCH ? 4 : 8;
    const int run = 256 / sl;
    int ldy = 0, blocks = 0;
    int64_t off = 0;
    for (int j = 0; j < a.n; j++) {
        const int groups = column_groups[j];
        parts[j] = part + off;
        r.m[j] = RedMat{part + off, a.bias[j], groups, a.M[j], 1, ldy, blocks};
        off += (int64_t)groups * T * a.M[j];
        ldy += a.M[j];
        if (mode != EPI_SWIGLU || j == 0) blocks += T * (int)bs_cdiv(a.M[j], run);
    }
    r.ssq = input_rms ? part + off : nullptr;
    r.ssq_n = r.m[0].I;
    float *ssq = input_rms ? part + off : nullptr;
    const int st = tiles ? bs_launch_tile_group(a.n, a.packed, a.u, a.vt, a.I, a.M, parts, ssq, x, N, K, T, split, s)
                         : bs_launch_strip_group(a.n, a.packed, a.u, a.vt, a.I, a.M, parts, ssq, x, N, K, T, s);
    if (st != BS_OK) return st;
    if (mode == EPI_SWIGLU) ldy = a.M[0];
    for (int j = a.n; j < GEMV_MAX_GROUP; j++) r.m[j] = r.m[0];
    if (!launch_reduce_wide(slots, r, residual, y, T, ldy, s)) switch (sl) {
        case 1: launch_reduce_flat<1>(blocks, r, residual, y, T, ldy, s); break;
        case 2: launch_reduce_flat<2>(blocks, r, residual, y, T, ldy, s); break;
        case 4: launch_reduce_flat<4>(blocks, r, residual, y, T, ldy, s); break;
        default: launch_reduce_flat<8>(blocks, r, residual, y, T, ldy, s); break;
    }
    BS_LAUNCH_CHECK();
    return BS_OK;
}

// *taken = false (and BS_ERR_SHAPE): no packed-sign kernel takes the shapes.  The scratch is looked at before anything is enqueued.
int launch_group(const GroupArgs &a, int N, int K, const half_t *x, int T, int mode, const half_t *residual,
                 half_t *y, bool input_rms, float eps, void *workspace, int64_t workspace_bytes, bool *taken, hipStream_t s) {
    CallPlan c;
    plan_call(c, a.I, a.M, a.n, N, K, T);
    *taken = c.path >= 0;
    if (c.path < 0) return BS_ERR_SHAPE;
    if (!workspace || workspace_bytes < scratch_bytes(c) || !bs_aligned(workspace, 256)) return BS_ERR_WORKSPACE;
    if (!bs_aligned(x, 16)) return BS_ERR_SHAPE;
    if (mode == EPI_SWIGLU && (a.n != 2 || a.M[0] != a.M[1])) return BS_ERR_SHAPE;
    for (int j = 0; j < a.n; j++)
        if (!bs_aligned(a.packed[j], 16) || !bs_aligned(a.vt[j], 16) || !bs_aligned(a.u[j], 8)) return BS_ERR_SHAPE;
    bool split = c.split;
    for (int j = 0; j < a.n; j++) split = split && bs_aligned(a.u[j], 16);
    if (split || (c.path == 1 && !c.sparse)) return launch_group_strips(a, N, K, x, T, mode, residual, y, input_rms, eps, workspace, split, s);
    int ldy = 0;
    for (int j = 0; j < a.n; j++) ldy += a.M[j];
    if (mode == EPI_SWIGLU) ldy = a.M[0];
    // Tokens go in passes of tp, the last one possibly shorter.  Every pass length has its own
    // plan (instantiation, grid, partial layout): the kernel a plan names exists for that token
    // count only.  Passes run one after the other on the stream and share the workspace.
    const int tp = pass_tokens(T);
    float *part = (float *)workspace;
    for (int t0 = 0; t0 < T; t0 += tp) {
        const int tn = (T - t0 < tp) ? T - t0 : tp;
        if (tn != tp) make_plan(c.gemv, a.I, a.M, a.n, N, K, tn);
        const Plan &p = c.gemv;
        GemvGroup g;
        RedGroup r;
        g.n = r.n = a.n;
        r.mode = mode;
        r.n_in = N;
        r.eps = eps;
        r.ssq = nullptr;
        r.ssq_n = 0;
        // threads per output of the summing kernel: at most FLAT_BATCH loads in flight per thread where the slots allow
        int slots = 0;
        for (int j = 0; j < a.n; j++)
            if (a.I[j] * p.kmax[j] > slots) slots = a.I[j] * p.kmax[j];
        const int sl = slots <= FLAT_BATCH ? 1 : slots <= 2 * FLAT_BATCH ? 2 : slots <= 4 * FLAT_BATCH ? 4 : 8;
        const int run = 256 / sl;
        int y_off = 0, blocks = 0;
        for (int j = 0; j < a.n; j++) {
            g.m[j] = GemvMat{a.packed[j], a.u[j], a.vt[j], part + p.part_off[j], a.M[j], p.row_tiles[j], p.kmax[j],
                             p.first_wg[j], p.sp[j], p.pair};
            r.m[j] = RedMat{part + p.part_off[j], a.bias[j], a.I[j], a.M[j], p.kmax[j], y_off, blocks};
            y_off += a.M[j];
            if (mode != EPI_SWIGLU || j == 0) blocks += tn * (int)bs_cdiv(a.M[j], run);
        }
        for (int j = a.n; j < GEMV_MAX_GROUP; j++) { g.m[j] = g.m[0]; r.m[j] = r.m[0]; }
        const half_t *xp = x + (int64_t)t0 * N;
        r.xin = input_rms ? xp : nullptr;
        int st;
        if (p.sparse) st = bs_launch_gemv_sparse(p.R, tn, p.grid, g, xp, N, K, p.n_chunks, s);
        else if (p.mx) st = bs_launch_gemv_mx(p.R, tn, p.grid, g, xp, N, K, p.n_chunks, s);
        else switch (tn) {
            case 1: st = launch_T<1>(p, g, xp, N, K, s); break;
            case 2: st = launch_T<2>(p, g, xp, N, K, s); break;
            case 3: st = launch_T<3>(p, g, xp, N, K, s); break;
            default: st = launch_T<4>(p, g, xp, N, K, s); break;
        }
        if (st != BS_OK) return st;
        const half_t *res_p = residual ? residual + (int64_t)t0 * ldy : nullptr;
        half_t *y_p = y + (int64_t)t0 * ldy;
        switch (sl) {
            case 1: launch_reduce_flat<1>(blocks, r, res_p, y_p, tn, ldy, s); break;
            case 2: launch_reduce_flat<2>(blocks, r, res_p, y_p, tn, ldy, s); break;
            case 4: launch_reduce_flat<4>(blocks, r, res_p, y_p, tn, ldy, s); break;
            default: launch_reduce_flat<8>(blocks, r, res_p, y_p, tn, ldy, s); break;
        }
        BS_LAUNCH_CHECK();
    }
    return BS_OK;
}

}  // namespace

// Bytes of scratch the packed-sign paths (factor-through or strip kernel) need for these
// matrices and token count; 0 when neither takes them.
int64_t bs_gemv_group_workspace_bytes(const int *I, const int *M, int n, int N, int K, int T) {
    CallPlan c;
    plan_call(c, I, M, n, N, K, T);
    return scratch_bytes(c);
}

// Which instantiation and grid a decode forward of these dimensions runs
// (0 in *waves when the decode kernel does not take them).
void bs_gemv_plan_info(int I, int M, int N, int K, int T, int *waves, int *row_tiles_per_wave, int *grid, int *kmax) {
    *waves = *row_tiles_per_wave = *grid = *kmax = 0;
    CallPlan c;
    plan_call(c, &I, &M, 1, N, K, T);
    if (c.path != 0 && !c.sparse) return;
    const Plan &p = c.gemv;
    *waves = p.waves;
    *row_tiles_per_wave = p.R;
    *grid = p.grid;
    *kmax = p.kmax[0];
}

// The kernel family a single-matrix forward of these dimensions runs on (values of BS_PATH_* in the public header).
int bs_gemv_forward_path(int I, int M, int N, int K, int T) {
    const int path = group_path(&I, &M, 1, N, K, T);
    if (path < 0) return BS_PATH_REBUILD;
    if (path == 1) {
        const int c = bs_strip_kernel_choice(I, M, N, K, T);
        return c == 1 ? BS_PATH_STRIP : c == 2 ? BS_PATH_WALKED : BS_PATH_PANEL;
    }
    return mx_rows_per_tile(&I, &M, 1, N, K, pass_tokens(T)) > 0 ? BS_PATH_DECODE_MX : BS_PATH_DECODE_F16;
}

// 1: gemv_sparse_kernel runs these matrices, of three tokens only with u off a 16-byte boundary where split_tiles has the tile kernel take them
int bs_gemv_sparse_serves(const int *I, const int *M, int n, int N, int K, int T) {
    CallPlan c;
    plan_call(c, I, M, n, N, K, T);
    return c.sparse && !c.split;
}

// Which call of the tile and column kernels serves these matrices, with u on 16-byte boundaries (values of BS_TILE_* in the public header).
int bs_gemv_tile_kernel(const int *I, const int *M, int n, int N, int K, int T, int *columns) {
    const int path = group_path(I, M, n, N, K, T);
    Plan p;
    const bool sparse = T <= 3 && sparse_plan(p, I, M, n, N, K, T, path, path == 0 ? mx_rows_per_tile(I, M, n, N, K, T) : 0);
    if (path == 1 && sparse) return BS_TILE_NONE;
    if (path == 1 && (n == 1 || T <= 48)) return !bs_tile_columns(I, M, n, N, K, T, columns) ? BS_TILE_NONE : T > 48 ? BS_TILE_COLUMN : BS_TILE_FORWARD;
    if (path == 0) return split_tiles(I, M, n, N, K, T, sparse ? &p : nullptr) && bs_tile_columns(I, M, n, N, K, T, columns) ? BS_TILE_TWO_TERMS : BS_TILE_NONE;
    for (int j = 0; j < n; j++)
        if (bs_gemv_forward_path(I[j], M[j], N, K, T) != BS_PATH_REBUILD) return BS_TILE_NONE;
    return bs_tile_columns(I, M, n, N, K, 0, columns) ? BS_TILE_REBUILD : BS_TILE_NONE;
}

// 0: not a decode-kernel shape, 1: gemv_kernel (fp16 MFMA), 2: gemv_mx_kernel (block-scaled fp4 x fp6 MFMA)
int bs_gemv_plan_kernel(int I, int M, int N, int K, int T) {
    if (group_path(&I, &M, 1, N, K, T) != 0) return 0;
    return mx_rows_per_tile(&I, &M, 1, N, K, pass_tokens(T)) > 0 ? 2 : 1;
}

int bs_gemv_set_kernel(int mode) {
    if (mode < 0 || mode > 2) return BS_ERR_SHAPE;
    g_decode_kernel = mode;
    return BS_OK;
}

// *taken = false when the fast path does not apply (the caller falls
// back to rebuilding the weight); otherwise the status is final.
int bs_launch_gemv(const uint8_t *packed, const half_t *u, const half_t *vt, const half_t *x,
                   const half_t *bias, half_t *y, int I, int M, int N, int K, int T,
                   void *workspace, int64_t workspace_bytes, bool *taken, hipStream_t s) {
    GroupArgs a;
    a.n = 1;
    a.packed[0] = packed; a.u[0] = u; a.vt[0] = vt; a.bias[0] = bias; a.I[0] = I; a.M[0] = M;
    return launch_group(a, N, K, x, T, EPI_NONE, nullptr, y, false, 0.f, workspace, workspace_bytes, taken, s);
}

int bs_launch_gemv_group(int n, const uint8_t *const *packed, const half_t *const *u, const half_t *const *vt,
                         const half_t *const *bias, const int *I, const int *M, int N, int K, const half_t *x, int T,
                         int mode, const half_t *residual, half_t *y, int input_rms, float eps, void *workspace,
                         int64_t workspace_bytes, hipStream_t s) {
    if (n < 1 || n > GEMV_MAX_GROUP) return BS_ERR_SHAPE;
    if (mode == EPI_RESIDUAL && !residual) return BS_ERR_NULL;
    bool taken;
    GroupArgs a;
    a.n = n;
    for (int j = 0; j < n; j++) {
        a.packed[j] = packed[j]; a.u[j] = u[j]; a.vt[j] = vt[j]; a.bias[j] = bias ? bias[j] : nullptr;
        a.I[j] = I[j]; a.M[j] = M[j];
    }
    return launch_group(a, N, K, x, T, mode, residual, y, input_rms != 0, eps, workspace, workspace_bytes, &taken, s);
}
