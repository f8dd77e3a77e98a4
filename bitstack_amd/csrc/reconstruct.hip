// Weight reconstruction for gfx950:
//   w[m, n] = fp16( sum_i s_i[m, n] * sum_r u_i[m, r] * vt_i[r, n] )
// fp32 everywhere until the single final rounding.
//
// Packed signs at rank 16 are rebuilt by the kernel in tile.hip where it takes the shape (bs_launch_reconstruct_packed; us, this one / that: 28672 x 8192, 3 blocks
// 176 / 113, 14336 x 4096, 8 69 / 50, 4096 x 4096, 8 22.4 / 20.2, 5000 x 1408, 6 15.4 / 11.9).  Here: the rest, and int8 signs.
//
// Tiled kernel.  A workgroup owns a strip of 128 columns and a range of rows.
// It first stages the strip's slice of vt for ALL blocks in LDS, transposed to
// [block][column][rank] (vt is stored rank-major, the MFMA wants the rank
// index contiguous per lane; 16 halves per column plus 4 after every 8 columns keeps
// the 8-byte fragment reads aligned and off each other's banks), then walks its rows 16 per wave at a time with
// no further barrier.  Per block the rank-k product of a 16 x 16 patch is one
// v_mfma_f32_16x16x16_f16 computed TRANSPOSED, D[n, m] = sum_r vt[r, n] u[m, r],
// so that a lane ends up with four consecutive columns of one row - one nibble
// of that row's packed sign byte - and, over a pair of patches, with a whole byte
// (eight consecutive columns, one 16-byte store).  A nibble addresses a 16-entry
// table in LDS that holds its four signs as halves of +-1.0, which a mixed-precision
// FMA (fp32 product x fp16 sign + fp32 sum) multiplies in: half a VALU instruction per
// sign for the lookup instead of two for shifting and merging each sign bit.  Signs and u of the
// next block are loaded while the current block is multiplied.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int RT_COLS = 128;   // columns per workgroup strip
constexpr int VSTRIDE = 16;    // halves per column in LDS: the 16 ranks, contiguous
constexpr int VGROUP_PAD = 4;  // extra halves after every 8 columns (keeps the fragment reads off each other's banks)
constexpr int VBLOCK = RT_COLS * VSTRIDE + (RT_COLS / 8) * VGROUP_PAD;   // halves per block in LDS
constexpr int RT_MAXB = 36;    // most blocks whose vt strip fits in LDS (36 x 4.1 KB)
constexpr int MASK_TABLE = 256;       // bytes: 16 nibbles x 4 sign masks
constexpr int SIGN_LUT_HALVES = 64;   // 16 nibbles x 4 signs (reconstruct_byte_kernel)
constexpr int RA_MAXB = 39;    // ... of reconstruct_byte_kernel (39 x 4 KB beside its sign table)

// K16: the rank is 16 (every u fragment is one 8-byte load).  Smaller ranks pick their halves one by one behind
// branches, and the compiler then waits for every load in flight where the branches meet: that instantiation runs
// one pair ahead at best.
// FLIP (ranks 4 to 16): the sums of the kernel in tile.hip, bit for bit: the sum over the blocks is kept divided by the block's sign, it changes sign where two
// blocks differ (a nibble's four masks come from the table instead of its four signs) and the matrix instruction adds the next product to it.  It takes the int8
// signs, and what that kernel cannot read, of the shapes that it takes.  us, product and FMA / this: int8 signs, 14336 x 4096, 8 blocks 163 / 154, 4096 x 4096, 8
// 45 / 42; packed signs level where rows are long (14336 x 4096, 8 blocks 69.4 / 69.8) and behind where they are not (20000 x 896, 2 blocks 13.0 / 14.1).
template <bool PACKED, bool K16, bool FLIP>
__global__ __launch_bounds__(256, 4) void reconstruct_tile_kernel(
    const uint8_t *__restrict__ packed, const int8_t *__restrict__ sign,
    const half_t *__restrict__ u, const half_t *__restrict__ vt, half_t *__restrict__ w,
    int I, int M, int N, int K, int rows_per_wg) {
    // First, at LDS address 0 (the kernel has no other LDS), a table of the 16 nibbles: four halves each of +-1.0 (+1.0 for a set bit, first
    // column in the top bit) or, FLIP, four masks (the sign bit of an fp32 for a set bit).  Then [I][VBLOCK]: column c of a block at
    // c * 16 + (c / 8) * 4.
    extern __shared__ __attribute__((aligned(256))) half_t lds_all[];
    constexpr int TABLE = FLIP ? MASK_TABLE : SIGN_LUT_HALVES * 2;        // bytes
    half_t *const vl = lds_all + TABLE / 2;
    typedef const __attribute__((address_space(3))) half4_t *lds_half4_ptr;
    typedef const __attribute__((address_space(3))) uint4_t *lds_uint4_ptr;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);   // the same in every lane: loop counts that depend on it stay scalar
    const int lm = lane & 15, g = lane >> 4;
    // Workgroups are dealt round-robin to the 8 XCDs, each with its own L2.  The eight
    // strips that share one 128-byte line of sign bytes must meet in ONE L2, and so
    // should the row groups that re-read one strip of vt: every XCD gets a contiguous
    // run of slots ordered (octet of strips, row group, strip within the octet).  The
    // grid is padded to whole octets; slots beyond the last strip do nothing.
    int n0, row_begin;
    {
        const int nb = gridDim.x * gridDim.y, lin = blockIdx.x + gridDim.x * blockIdx.y;
        const int xcd = lin & 7, loc = lin >> 3, base = nb >> 3, rem = nb & 7;
        const int v = xcd * base + min(xcd, rem) + loc;
        const int rest = v >> 3, strip = (rest / (int)gridDim.y) * 8 + (v & 7);
        if (strip * RT_COLS >= N) return;
        n0 = strip * RT_COLS;
        row_begin = (rest % (int)gridDim.y) * rows_per_wg;
    }
    const int row_end = min(row_begin + rows_per_wg, M);
    const int64_t row_bytes = N >> 3;
    const int64_t block_bytes = (int64_t)M * row_bytes;

    // staging role: rank index fastest across lanes, 16 pieces of 8 columns
    const int sr = tid & 15, sp = tid >> 4;
    // Patches come in pairs: of a 32-column group, patch 2q takes columns 8g'..8g'+3 and patch
    // 2q+1 columns 8g'+4..8g'+7 (g' = 0..3), so that a lane (row lm, group g) ends up with EIGHT
    // consecutive columns of its row - one byte of the packed signs, one 16-byte store.
    // The lane's byte of a sign word is byte g; its two nibbles address the table, times 8:
    // (word >> sh_hi) & 0x78 for the first four columns, (word rotated right by sh_lo) & 0x78 for the others; or times 16.
    const int sh_hi = 8 * g + 1, sh_lo = (8 * g - 3) & 31, byte_at = 8 * g;
    // this lane's A-fragment column within a 32-column group (n-index lm of either patch, less 4 * (s & 1))
    const int acol = 8 * (lm >> 2) + (lm & 3);
    const int aoff = acol * VSTRIDE + (lm >> 2) * VGROUP_PAD + 4 * g;

    {
        const int i0 = 0, ib = I;
        // u rows and sign words of one (row step, block); requested one block ahead, also
        // across the end of a row step (first block of the next 16 rows), and issued for
        // the very first block before the vt strip is staged
        // Addresses are a wave-uniform 64-bit base (the block: scalar arithmetic) plus a 32-bit
        // offset per lane that depends on the row only and is renewed once per row step.
        uint32_t off_u;                             // bytes: this lane's u row (its four ranks)
        auto load_u = [&](int i, half4_t &b) {
            const char *ub = reinterpret_cast<const char *>(u) + (int64_t)i * M * K * 2;
            const half_t *up = reinterpret_cast<const half_t *>(ub + off_u);
            if (K16) {
                b = *reinterpret_cast<const half4_t *>(up);
            } else {
#pragma unroll
                for (int j = 0; j < 4; j++) b[j] = (4 * g + j < K) ? up[j] : (half_t)0;
            }
        };
        // The (row step, block) pairs of this wave form one sequence.  u rows are requested pair by pair, three pairs
        // ahead, into four register sets used in turn (the loop is written out eight pairs at a time, so that no set is
        // ever copied into another: a copy waits for the load it copies).  Sign words are requested FOUR PAIRS PER
        // INSTRUCTION: lane group g loads the 16 bytes of pair 4 q + g of the sequence (its row's sign bytes of this
        // strip in that pair's block), and the pair that is being multiplied fetches its words from the group that
        // holds them with four cross-lane reads.  Loaded pair by pair, all four lane groups requested the same 16
        // bytes per row, and a load instruction costs the memory pipeline its 16 rows' lines whatever it brings.
        half4_t b_set[4];
        uint4_t quad[2];
        const int first_row = row_begin + wave * 16;
        // Requests are unconditional (behind the last pair they repeat its row step): a
        // branch around a load makes the compiler wait for every load in flight at the join.
        const int last_m0 = first_row + ((max(row_end - first_row, 1) - 1) / 64) * 64;
        int pf_i = 0, pf_m0 = first_row;           // the pair the next u request is for
        auto set_row = [&](int m0) {
            const int row = min(min(m0, last_m0) + lm, M - 1);
            off_u = (uint32_t)(row * K + 4 * g) * 2u;
        };
        set_row(pf_m0);
        auto request_u = [&](half4_t &b) {
            load_u(i0 + pf_i, b);
            if (++pf_i == ib) {
                pf_i = 0;
                pf_m0 += 64;
                set_row(pf_m0);
            }
        };
        // the pair this lane loads for the next quad: block ql_i of the row step at ql_m0 (per lane: the groups differ)
        int ql_i = g, ql_m0 = first_row;
        auto wrap_quad = [&]() {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (ql_i >= ib) {
                    ql_i -= ib;
                    ql_m0 += 64;
                }
        };
        wrap_quad();
        auto request_quad = [&](uint4_t &qd) {
            if (PACKED) {
                const int row = min(min(ql_m0, last_m0) + lm, M - 1);
                qd = *reinterpret_cast<const uint4_t *>(packed + (int64_t)(i0 + ql_i) * block_bytes + (n0 >> 3) + (int64_t)row * row_bytes);
            }
            ql_i += 4;
            wrap_quad();
        };
        // the sign words of pair `sel` (0..3) of a quad, for every lane group
        auto sign_words = [&](const uint4_t &qd, int sel) {
            const int from = (16 * sel + lm) * 4;
            uint4_t r;
#pragma unroll
            for (int d = 0; d < 4; d++) r[d] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)qd[d]);
            return r;
        };
        quad[0] = quad[1] = (uint4_t){0, 0, 0, 0};
        request_quad(quad[0]);
#pragma unroll
        for (int k = 0; k < 3; k++) request_u(b_set[k]);

        // four blocks at a time, so that their loads are in flight together
        for (int q0 = 0; q0 < ib; q0 += 4) {
            half8_t v[4];
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const int i = min(q0 + k, ib - 1);
                v[k] = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
                if (sr < K) v[k] = *reinterpret_cast<const half8_t *>(vt + ((int64_t)i * K + sr) * N + n0 + 8 * sp);
            }
#pragma unroll
            for (int k = 0; k < 4; k++) {
                if (q0 + k < ib) {
#pragma unroll
                    for (int e = 0; e < 8; e++) vl[(q0 + k) * VBLOCK + (8 * sp + e) * VSTRIDE + sp * VGROUP_PAD + sr] = v[k][e];
                }
            }
        }
        if (PACKED && tid < 64) {
            const bool set = ((tid >> 2) >> (3 - (tid & 3))) & 1;
            if (FLIP) reinterpret_cast<uint32_t *>(lds_all)[tid] = set ? 0x80000000u : 0u;
            else lds_all[tid] = set ? (half_t)1.f : (half_t)-1.f;
        }
        __syncthreads();

        // 16 rows per wave and step; the current pair is (rows m0.., block i)
        // The first block of a row step starts the sums (a product, not a sum with zero): cleared accumulators
        // would meet the running ones where the paths join, and the compiler then copies two dozen registers per block.
        float4_t acc[8];
        uint4_t before;                             // the sign words of the pair before this one (int8 signs: t_before)
        uint32_t t_before[8];
        int i = 0, m0 = first_row;
        // a patch's sums change sign where `flip` has a set bit
        auto masks = [&](uint32_t flips, int half) { return *(lds_uint4_ptr)(uintptr_t)((half ? flips << 4 : flips) & 0xF0u); };
        auto change = [&](float4_t &sum, const uint4_t &m) {
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float v = sum[j];
                const uint32_t mj = m[j];
                sum[j] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v) ^ mj);
            }
        };
        // (int8 signs: negative ones have bit 7 set)
        auto masks_of = [&](uint32_t t) { return (uint4_t){(t << 24) & 0x80000000u, (t << 16) & 0x80000000u, (t << 8) & 0x80000000u, t & 0x80000000u}; };
        auto consume = [&](const half4_t &b_cur, const uint4_t &swc, auto first_tag) {
            constexpr bool FIRST = decltype(first_tag)::value;
            const int row = min(m0 + lm, M - 1);
            const half_t *vb = vl + i * VBLOCK + aoff;
            // all eight fragments first: the LDS latency does not sit in front of the products
            half4_t a[8];
#pragma unroll
            for (int s = 0; s < 8; s++)
                a[s] = *reinterpret_cast<const half4_t *>(vb + (32 * (s >> 1) + 4 * (s & 1)) * VSTRIDE + 4 * (s >> 1) * VGROUP_PAD);
            uint4_t m[8];
            if constexpr (!FLIP) {
                // the signs of a patch as four halves of +-1.0 from the table (16 entries of 8 bytes: one entry per
                // pair of banks, equal nibbles read the same address), multiplied in by a mixed-precision FMA
                half4_t sv[8];
                if (PACKED) {
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const uint32_t hi = ((swc[q] >> sh_hi) & 0x78u);
                        const uint32_t lo = (__builtin_amdgcn_alignbit(swc[q], swc[q], sh_lo) & 0x78u);
                        sv[2 * q] = *reinterpret_cast<lds_half4_ptr>(hi);
                        sv[2 * q + 1] = *reinterpret_cast<lds_half4_ptr>(lo);
                    }
                }
                float4_t p_next = __builtin_amdgcn_mfma_f32_16x16x16f16(a[0], b_cur, (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    const float4_t p = p_next;
                    if (s + 1 < 8)
                        p_next = __builtin_amdgcn_mfma_f32_16x16x16f16(a[s + 1], b_cur, (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    if (PACKED) {
#pragma unroll
                        for (int j = 0; j < 4; j++) acc[s][j] = __builtin_fmaf(p[j], (float)sv[s][j], FIRST ? 0.f : acc[s][j]);   // (a plain product would not become a mixed-precision instruction)
                    } else {
                        uint32_t t = *reinterpret_cast<const uint32_t *>(
                            sign + ((int64_t)(i0 + i) * M + row) * N + n0 + 32 * (s >> 1) + 8 * g + 4 * (s & 1));
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            uint32_t sf = ((t << (24 - 8 * j)) & 0x80000000u) | 0x3F800000u;
                            acc[s][j] = FIRST ? p[j] * __builtin_bit_cast(float, sf) : __builtin_fmaf(p[j], __builtin_bit_cast(float, sf), acc[s][j]);
                        }
                    }
                }
            } else {
                uint32_t t[8];
                if (!PACKED) {
#pragma unroll
                    for (int s = 0; s < 8; s++)
                        t[s] = *reinterpret_cast<const uint32_t *>(sign + ((int64_t)(i0 + i) * M + row) * N + n0 + 32 * (s >> 1) + 8 * g + 4 * (s & 1));
                }
                if (!FIRST) {
#pragma unroll
                    for (int s = 0; s < 8; s++) m[s] = PACKED ? masks((before[s >> 1] ^ swc[s >> 1]) >> byte_at, s & 1) : masks_of(t_before[s] ^ t[s]);
                }
#pragma unroll
                for (int s = 0; s < 8; s++) {
                    if (FIRST) {
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x16f16(a[s], b_cur, (float4_t){0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                    } else {
                        change(acc[s], m[s]);
                        acc[s] = __builtin_amdgcn_mfma_f32_16x16x16f16(a[s], b_cur, acc[s], 0, 0, 0);
                    }
                }
                if (PACKED) before = swc;
                else {
#pragma unroll
                    for (int s = 0; s < 8; s++) t_before[s] = t[s];
                }
            }
            if (++i == ib) {
                if constexpr (FLIP) {
#pragma unroll
                    for (int s = 0; s < 8; s++) m[s] = PACKED ? masks(~before[s >> 1] >> byte_at, s & 1) : masks_of(t_before[s]);
#pragma unroll
                    for (int s = 0; s < 8; s++) {
                        change(acc[s], m[s]);
                        asm("" : "+v"(acc[s]));     // (else the optimiser pairs values of different patches, two moves for each)
                    }
                }
                if (m0 + lm < M) {
                    half_t *wp = w + (int64_t)(m0 + lm) * N + n0 + 8 * g;
#pragma unroll
                    for (int s = 0; s < 8; s += 2) {
                        half8_t o = {(half_t)acc[s][0], (half_t)acc[s][1], (half_t)acc[s][2], (half_t)acc[s][3],
                                     (half_t)acc[s + 1][0], (half_t)acc[s + 1][1], (half_t)acc[s + 1][2], (half_t)acc[s + 1][3]};
                        *reinterpret_cast<half8_t *>(wp + 16 * s) = o;      // 32 columns per pair of patches
                    }
                }
                i = 0;
                m0 += 64;
            }
        };
        const int n_pairs = first_row < row_end ? ((row_end - first_row + 63) / 64) * ib : 0;
        for (int p = 0; p < n_pairs; p += 8) {
#pragma unroll
            for (int idx = 0; idx < 8; idx++) {
                if (idx > 0 && p + idx >= n_pairs) break;
                const int h = idx >> 2, k = idx & 3;
                if (k == 0) request_quad(quad[h ^ 1]);          // the next quad, into the set consumed last
                request_u(b_set[(k + 3) & 3]);
                const uint4_t swc = sign_words(quad[h], k);
                if (i == 0)
                    consume(b_set[k], swc, std::true_type{});
                else
                    consume(b_set[k], swc, std::false_type{});
            }
        }
    }
}

// Column counts that are multiples of 8 but not of 128 (and what else the tiled kernel declines of those): rows of sign bytes then start anywhere, and the last
// columns fill no strip.  A workgroup of 8 waves takes 128 columns, whose vt fragments of all blocks it leaves in LDS first; a wave has 64 of them and every fourth
// step of 32 rows, in two patches of v_mfma_f32_32x32x16_f16, D[column, row], with the columns dealt so that a lane ends with 32 consecutive ones of one row: one
// unaligned word of signs, four 16-byte stores.  u rows and signs are requested one (row step, block) ahead, in two register sets that take turns.  Signs come out of
// the tiled kernel's table and go in by the same mixed-precision FMA (int8 signs: converted; the same sum).
// What bounds it: the vector instructions, 24 per step of 1024 signs, and its stores.  Rebuilds at rank 16, us, one output per thread / this: 4096 x 4104
// of 1 block 101 / 18, of 4 385 / 23; 6144 x 6136 of 8 1641 / 53; 512 x 6008 of 4 63 / 8.2; 1000 x 1000 of 4 23 / 5.4.  (Four waves, each with 128 columns as the
// tiled kernel has them, and vt fragments in registers for the block at hand: 23 to 85 where this takes 19 to 53.)
constexpr int RA_COLS = 128, RA_ROWS = 32, RA_WAVES = 8, RA_STREAMS = 4;         // columns per workgroup, rows per step, waves, waves side by side in rows
template <bool PACKED, bool K16>
__global__ __launch_bounds__(64 * RA_WAVES, PACKED ? 4 : 2) void reconstruct_byte_kernel(
    const uint8_t *__restrict__ packed, const int8_t *__restrict__ sign, const half_t *__restrict__ u, const half_t *__restrict__ vt, half_t *__restrict__ w,
    int I, int M, int N, int K, int strips, int steps_per_wg) {
    extern __shared__ __attribute__((aligned(128))) half_t lds_all[];
    typedef const __attribute__((address_space(3))) half4_t *lds_half4_ptr;
    const uint32_t lut = (uint32_t)reinterpret_cast<uintptr_t>((const __attribute__((address_space(3))) half_t *)lds_all);
    half8_t *const frags = reinterpret_cast<half8_t *>(lds_all + SIGN_LUT_HALVES);      // [block][64 columns: 2][patch: 2][lane]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 31, h = lane >> 5;
    // every XCD gets a contiguous run of (row group, strip), strips fastest: neighbours share lines of sign bytes and u rows
    const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, base = nb >> 3, rem = nb & 7;
    const int v = xcd * base + min(xcd, rem) + loc, group = v / strips, strip = (v - group * strips) * RA_COLS;
    if (tid < SIGN_LUT_HALVES) lds_all[tid] = ((tid >> 2) >> (3 - (tid & 3))) & 1 ? (half_t)1.f : (half_t)-1.f;
    // patch p, row a of D: column 32 ((a / 4) % 2) + 16 p + 4 (a / 8) + a % 4
    for (int item = wave; item < 4 * I; item += RA_WAVES) {
        const int i = item >> 2, col = min(strip + 64 * ((item >> 1) & 1) + 32 * ((row >> 2) & 1) + 16 * (item & 1) + 4 * (row >> 3) + (row & 3), N - 1);
        half8_t f;
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const half_t val = vt[((int64_t)i * K + (K16 ? 8 * h + r : min(8 * h + r, K - 1))) * N + col];
            f[r] = K16 || 8 * h + r < K ? val : (half_t)0;
        }
        frags[64 * item + lane] = f;
    }
    __syncthreads();

    const int c0 = strip + 64 * (wave & 1) + 32 * h;             // this lane's columns; beyond N: others are read, nothing is stored
    const int first = group * steps_per_wg + (wave >> 1), last = min((group + 1) * steps_per_wg, (M + RA_ROWS - 1) / RA_ROWS);
    const int cr = min(c0, N - 32), late = min(c0 - cr, 31);     // (the last columns' word starts earlier, by a multiple of 8 signs)
    struct Ahead {
        half8_t u;
        uint32_t bits;                               // packed
        uint2_t bytes[4];                            // int8
    };
    int ask_step = first, ask_i = 0;
    auto request = [&](Ahead &a) {                   // (behind the last one that one is requested again)
        const int m = min(ask_step * RA_ROWS + row, M - 1);
        const half_t *up = u + ((int64_t)ask_i * M + m) * K;
        if (K16) {
            const half4_t lo = *reinterpret_cast<const half4_t *>(up + 8 * h), hi = *reinterpret_cast<const half4_t *>(up + 8 * h + 4);
            a.u = (half8_t){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        } else {
#pragma unroll
            for (int r = 0; r < 8; r++) a.u[r] = up[min(8 * h + r, K - 1)];
        }
        const int64_t at = ((int64_t)ask_i * M + m) * N;
        if (PACKED) {
            __builtin_memcpy(&a.bits, packed + ((at + cr) >> 3), 4);
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++) a.bytes[e] = *reinterpret_cast<const uint2_t *>(sign + at + min(c0 + 8 * e, N - 8));
        }
        if (ask_step + RA_STREAMS < last || ask_i + 1 < I) {
            if (++ask_i == I) {
                ask_i = 0;
                ask_step += RA_STREAMS;
            }
        }
    };
    float16_t acc[2];
    int step = first, i = 0;
    auto consume = [&](const Ahead &a) {
        if (i == 0) acc[0] = acc[1] = (float16_t){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        half8_t b = a.u;
        if (!K16) {
#pragma unroll
            for (int r = 0; r < 8; r++) b[r] = 8 * h + r < K ? b[r] : (half_t)0;
        }
        float16_t p[2];
#pragma unroll
        for (int k = 0; k < 2; k++)
            p[k] = __builtin_amdgcn_mfma_f32_32x32x16_f16(frags[64 * (4 * i + 2 * (wave & 1) + k) + lane], b,
                                (float16_t){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        if (PACKED) {
            const uint32_t bits = a.bits >> late;
#pragma unroll
            for (int q = 0; q < 8; q++) {            // columns 4 q .. 4 q + 3: the upper half of byte q / 2 first
                constexpr uint32_t NIBBLE = 0x78u;
                const int sh = 8 * (q >> 1) + (q & 1 ? -3 : 1);
                const half4_t sv = *reinterpret_cast<lds_half4_ptr>((uintptr_t)((((sh < 0 ? bits << 3 : bits >> sh)) & NIBBLE) | lut));
#pragma unroll
                for (int j = 0; j < 4; j++) acc[q >> 2][4 * (q & 3) + j] = __builtin_fmaf(p[q >> 2][4 * (q & 3) + j], (float)sv[j], acc[q >> 2][4 * (q & 3) + j]);
            }
        } else {
#pragma unroll
            for (int k = 0; k < 32; k++)
                acc[k >> 4][k & 15] = __builtin_fmaf(p[k >> 4][k & 15], (float)(int8_t)(a.bytes[k >> 3][(k >> 2) & 1] >> (8 * (k & 3))), acc[k >> 4][k & 15]);
        }
        if (++i == I) {
            const int m = step * RA_ROWS + row;
            if (m < M) {
                half_t *to = w + (int64_t)m * N + c0;
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    half8_t o;
#pragma unroll
                    for (int k = 0; k < 8; k++) o[k] = (half_t)acc[e >> 1][8 * (e & 1) + k];
                    if (c0 + 8 * e < N) *reinterpret_cast<half8_t *>(to + 8 * e) = o;
                }
            }
            i = 0;
            step += RA_STREAMS;
        }
    };
    if (first >= last || strip + 64 * (wave & 1) >= N) return;
    Ahead even, odd;
    const int n = ((last - first + RA_STREAMS - 1) / RA_STREAMS) * I;
    request(even);
    for (int k = 0; k < n; k += 2) {
        request(odd);
        consume(even);
        if (k + 1 == n) break;
        request(even);
        consume(odd);
    }
}

// Any shape (also rows that do not start on a byte boundary): one output per
// thread, bit addressed through the flat element index.
template <bool PACKED>
__global__ __launch_bounds__(256) void reconstruct_generic_kernel(
    const uint8_t *__restrict__ packed, const int8_t *__restrict__ sign,
    const half_t *__restrict__ u, const half_t *__restrict__ vt, half_t *__restrict__ w,
    int I, int M, int N, int K) {
    const int64_t total = (int64_t)M * N;
    const int64_t block_bytes = (total + 7) >> 3;
    int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; e < total; e += stride) {
        const int m = (int)(e / N), n = (int)(e % N);
        float acc = 0.f;
        for (int i = 0; i < I; i++) {
            float p = 0.f;
            for (int r = 0; r < K; r++)
                p = __builtin_fmaf((float)u[((int64_t)i * M + m) * K + r],
                                   (float)vt[((int64_t)i * K + r) * N + n], p);
            float s;
            if (PACKED)
                s = ((packed[i * block_bytes + (e >> 3)] >> (7 - (int)(e & 7))) & 1) ? 1.f : -1.f;
            else
                s = (float)sign[(int64_t)i * total + e];
            acc += s * p;
        }
        w[e] = (half_t)acc;
    }
}

// Steps of 32 rows per workgroup of reconstruct_byte_kernel: four workgroups per CU, and a step or more for each of the four waves side by side in rows.
int byte_steps(int M, int N) {
    const int64_t strips = bs_cdiv(N, RA_COLS), steps = bs_cdiv(M, RA_ROWS);
    const int64_t groups = std::max<int64_t>(1, std::min<int64_t>(bs_cdiv(1024, strips), bs_cdiv(steps, RA_STREAMS)));
    return (int)bs_cdiv(bs_cdiv(steps, groups), RA_STREAMS) * RA_STREAMS;
}
// At rank 16 always.  Below, u is read half by half, and a wave's chain of (row step, block) pairs is some 1.15 us each; one output per thread takes 0.1 + 0.11 us
// per rank and block, or its products' time where there are many (fitted to 400 rebuilds from int8 signs, up to 12 blocks and 6 million weights; from packed signs the
// former is up to half slower, but the weight is the same bit for bit whatever it is made from, so both go one way).  us from int8 signs, that / byte kernel: 1211 x 432, 11 blocks,
// rank 5 11.7 / 16.3, 257 x 1928, 5, rank 6 7.5 / 10.2, 511 x 912, 1, rank 11 4.6 / 5.9; 523 x 4704, 7, rank 10 73.1 / 15.7; from packed signs 520 x 248, 9, rank 8 10.8 / 24.5,
// 4096 x 4104, 4, rank 8 244 / 39.  Of the 400 8 are more than 3 % behind one output per thread, 34 % at worst (150 x 3392, 8, rank 8), and from packed signs
// 1, 6 %.
bool byte_kernel_pays(int I, int M, int N, int K) {
    const double chain = 4.0 + 1.15 * I * (byte_steps(M, N) / RA_STREAMS);
    return K == 16 || chain <= std::max(2.5 + (0.1 + 0.11 * K) * I, 1.5 + (0.9e-6 + 0.3e-6 * K) * M * N * I);
}

template <bool PACKED>
int launch_reconstruct(const uint8_t *packed, const int8_t *sign, const half_t *u, const half_t *vt,
                       half_t *w, int I, int M, int N, int K, hipStream_t s) {
    // the tiled kernel addresses a block's u and sign rows with 32-bit byte offsets
    const bool small = (int64_t)M * (N >> 3) < ((int64_t)1 << 32) && (int64_t)M * K * 2 < ((int64_t)1 << 32);
    const bool tiled = (N % RT_COLS == 0) && I >= 1 && I <= RT_MAXB && small && bs_aligned(vt, 16) && bs_aligned(w, 16) &&
                       bs_aligned(u, 8) && (PACKED ? bs_aligned(packed, 16) : bs_aligned(sign, 4));
    const bool bytes = N % 8 == 0 && N >= 32 && I >= 1 && I <= RA_MAXB && bs_aligned(w, 16) && (K != 16 || bs_aligned(u, 8)) && (PACKED || bs_aligned(sign, 8)) &&
                       byte_kernel_pays(I, M, N, K);
    if (tiled) {
        // One wave of workgroups: as many row groups as the resident slots allow (LDS decides
        // how many workgroups a CU holds), so that no second, partial wave trails behind.
        // Every workgroup re-stages its vt strip, so rows per workgroup stay a multiple of 64.
        // (The weight has the same bits whatever it is made from: where the kernel in tile.hip takes the shape, its sums.)
        int columns;
        const bool flip = bs_tile_columns(&I, &M, 1, N, K, 0, &columns);
        const int strips = N / RT_COLS, strips8 = (int)bs_cdiv(strips, 8) * 8;
        const size_t lds_need = (size_t)I * VBLOCK * sizeof(half_t) + (flip ? MASK_TABLE : SIGN_LUT_HALVES * sizeof(half_t));   // vt images + table
        int per_cu = (int)((160 * 1024) / lds_need);
        if (per_cu > 8) per_cu = 8;
        if (per_cu < 1) per_cu = 1;
        int row_groups = (256 * per_cu) / strips8;
        if (row_groups < 1) row_groups = 1;
        int rows_per_wg = (int)bs_cdiv(bs_cdiv(M, row_groups), 64) * 64;
        row_groups = (int)bs_cdiv(M, rows_per_wg);
        const size_t lds = lds_need;
        static bs_lds_grant granted[4][BS_MAX_DEVICES];
        const auto kernel = flip ? (K == 16 ? reconstruct_tile_kernel<PACKED, true, true> : reconstruct_tile_kernel<PACKED, false, true>) : K == 16 ? reconstruct_tile_kernel<PACKED, true, false> : reconstruct_tile_kernel<PACKED, false, false>;
        const int st = bs_allow_lds((const void *)kernel, lds, granted[2 * flip + (K == 16)]);
        if (st != BS_OK) return st;
        dim3 grid((unsigned)bs_cdiv(strips, 8) * 8, row_groups);
        kernel<<<grid, 256, lds, s>>>(packed, sign, u, vt, w, I, M, N, K, rows_per_wg);
    } else if (bytes) {
        const int strips = (int)bs_cdiv(N, RA_COLS), steps = (int)bs_cdiv(M, RA_ROWS), per = byte_steps(M, N);
        const size_t lds = SIGN_LUT_HALVES * sizeof(half_t) + (size_t)I * 256 * sizeof(half8_t);
        static bs_lds_grant granted[2][BS_MAX_DEVICES];
        const void *kernel = K == 16 ? (const void *)reconstruct_byte_kernel<PACKED, true> : (const void *)reconstruct_byte_kernel<PACKED, false>;
        const int st = bs_allow_lds(kernel, lds, granted[K == 16]);
        if (st != BS_OK) return st;
        const int grid = strips * (int)bs_cdiv(steps, per);
        if (K == 16)
            reconstruct_byte_kernel<PACKED, true><<<grid, 64 * RA_WAVES, lds, s>>>(packed, sign, u, vt, w, I, M, N, K, strips, per);
        else
            reconstruct_byte_kernel<PACKED, false><<<grid, 64 * RA_WAVES, lds, s>>>(packed, sign, u, vt, w, I, M, N, K, strips, per);
    } else {
        int64_t blocks = bs_cdiv((int64_t)M * N, 256);
        if (blocks > 256 * 64) blocks = 256 * 64;
        reconstruct_generic_kernel<PACKED><<<(int)blocks, 256, 0, s>>>(packed, sign, u, vt, w, I, M, N, K);
    }
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int check_dims(int I, int M, int N, int K) {
    if (I < 0 || M <= 0 || N <= 0) return BS_ERR_SHAPE;
    if (K < 1 || K > 16) return BS_ERR_RANK;
    if ((int64_t)M * N > ((int64_t)1 << 40)) return BS_ERR_SHAPE;
    return BS_OK;
}

}  // namespace

int bs_launch_reconstruct_packed(const uint8_t *packed, const half_t *u, const half_t *vt,
                                 half_t *w, int I, int M, int N, int K, hipStream_t s) {
    const int st = bs_launch_tile_rebuild(1, &packed, &u, &vt, &I, &M, &w, N, K, s);
    if (st != BS_ERR_SHAPE) return st;
    return launch_reconstruct<true>(packed, nullptr, u, vt, w, I, M, N, K, s);
}

extern "C" int bs_reconstruct_w(const uint8_t *packed, const void *u, const void *vt, void *w,
                                int I, int M, int N, int K, void *stream) {
    int st = check_dims(I, M, N, K);
    if (st != BS_OK) return st;
    if (!w || (I > 0 && (!packed || !u || !vt))) return BS_ERR_NULL;
    if (!bs_aligned(u, 2) || !bs_aligned(vt, 2) || !bs_aligned(w, 2)) return BS_ERR_ALIGN;
    return bs_launch_reconstruct_packed(packed, (const half_t *)u, (const half_t *)vt, (half_t *)w, I, M, N, K, (hipStream_t)stream);
}

extern "C" int bs_reconstruct_w_from_sign(const int8_t *sign, const void *u, const void *vt, void *w,
                                          int I, int M, int N, int K, void *stream) {
    int st = check_dims(I, M, N, K);
    if (st != BS_OK) return st;
    if (!w || (I > 0 && (!sign || !u || !vt))) return BS_ERR_NULL;
    if (!bs_aligned(u, 2) || !bs_aligned(vt, 2) || !bs_aligned(w, 2)) return BS_ERR_ALIGN;
    return launch_reconstruct<false>(nullptr, sign, (const half_t *)u, (const half_t *)vt,
                                     (half_t *)w, I, M, N, K, (hipStream_t)stream);
}
