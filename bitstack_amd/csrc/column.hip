// Forward for 49 to 128 tokens on gfx950, rank 16 (and 4 to 15: column_ranks.hip), up to 8 blocks: the tile kernel's rebuild (tile.hip) with the loops turned round.
//
//   part[cg, t, m] = sum_{n in column group cg} x[t, n] * fp16( sum_i s_i[m, n] * sum_r u_i[m, r] * vt_i[r, n] )
//
// With this many tokens the y tile of 32 rows is too large to be handed over per tile, so a workgroup of 8 waves stays with 256 rows (32 per
// wave, the u rows of all blocks and y[T, 32 rows] in registers) and walks a run of columns, 64 at a time: the chunk's vt of all blocks (turned
// to [column][rank]) and x travel through registers into one of two LDS images while the other one is used, one barrier per chunk.  Sign
// words are the lane's own: 16 consecutive bytes of its row per block serve four chunks (a chunk is 32 columns of either half of
// 256, so that lane half h finds word q of its 16 bytes in chunk q), and are requested again right behind their last use.
// Per block and chunk two v_mfma_f32_32x32x16_f16 and one v_xor_b32 per weight, as in tile.hip; then the rounded weights are the B operand of
// y += x . w on v_mfma_f32_16x16x32_f16, x read from LDS.  Scratch holds one partial per column group, the summing kernel adds them up.
//
// What bounds it: the vector instructions of the sign flips, as in tile.hip, and as much waiting: by the counters 40 % of a SIMD's cycles (the matrix cores
// 21), the waves 39 % of their time at a barrier or for data.  14336 x 4096, 5 blocks, 100 tokens, cycles per chunk of 64 columns and
// wave: 2,400 in ten steps (200 each would be the instructions alone; the two waves of a SIMD compete), 1,000 in the second product (32 matrix
// instructions and 16 x reads), 280 for the next image, 390 at the barrier; 16 chunks, and 8,000 to 15,000 cycles before the first.
// us, walked or panel kernel -> this one, summing launch included: 14336 x 4096 x 5 blocks x 100 tokens 74.7 -> 57.6, 28672 x 8192 x 3 x 80
// 161 -> 105, 12621 x 13056 x 6 190 -> 129, 15100 x 10240 x 1 x 110 111 -> 63, 4096 x 4096 x 4 x 64 22.3 -> 21.0.
// Also tried: a higher wave priority for one wave of each SIMD, and one of them multiplying a chunk later than the other (three images): no
// difference or 3 % slower.
#include "common.h"
#include "rebuild_shared.h"

#include <type_traits>
#include <utility>

struct ColumnMat {
    const uint8_t *packed;
    const half_t *u, *vt;
    float *part;
    int M, row_groups, spans;                       // spans of 256 columns per column group
};

// The kernels for ranks 4 to 15 are the same code with a rank that is not known at compile time, in a translation unit of their own (column_ranks.hip includes this file): with
// one kernel for all ranks 14336 x 4096, 5 blocks, 100 tokens took 57.3 us for 55.0.
#ifdef COLUMN_RANKS
constexpr bool CL_K16 = false;
#else
constexpr bool CL_K16 = true;
#endif
int bs_launch_column_ranks(const ColumnMat &m, int I, int grid, const half_t *x, int N, int T, int K, hipStream_t s);

namespace {

constexpr int CL_WAVES = 8, CL_ROWS = 256, CL_TABLE = 512, CL_HALVES = 256, CL_MIN_T = 49, CL_MAX_T = 128;
constexpr int CL_IMAGE = 64 * 32;                   // bytes: a block's vt of a chunk, or 16 tokens of x

template <class F, int... Is>
__device__ __forceinline__ void cl_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void cl_for(F &&f) {
    cl_for_impl(f, std::make_integer_sequence<int, N>{});
}

typedef half8_t cl_half8_any __attribute__((aligned(2)));
typedef half4_t cl_half4_any __attribute__((aligned(2)));
typedef __attribute__((address_space(3))) char *cl_bytes;
typedef const __attribute__((address_space(3))) half8_t *cl_half8;
typedef __attribute__((address_space(3))) half8_t *cl_half8_rw;
typedef __attribute__((address_space(3))) half2_t *cl_half2_rw;
typedef const __attribute__((address_space(3))) uint4_t *cl_uint4;
typedef const __attribute__((address_space(3))) uint2_t *cl_uint2;

// TT: token tiles of 16
template <int TT, int I>
__global__ __launch_bounds__(64 * CL_WAVES, 2) void column_forward_kernel(const ColumnMat mat, const half_t *__restrict__ x, int N, int T, int ranks) {
    const int K = CL_K16 ? 16 : ranks;
    extern __shared__ __attribute__((aligned(1024))) char cl_lds[];
    const cl_bytes lds = (cl_bytes)cl_lds;
    // Behind the last block the sums round first and the sign changes on the rounded pairs: half the operations, the same bits.  Of the time with the change in fp32, average over seven matrices
    // from 20000 x 640 to 28672 x 8192 (56, 100 and 124 tokens): one block 0.978 to 0.985, two to four 0.980 to 1.002, five to eight with four token tiles 0.986 to 0.994 (28672 x 8192, 6 blocks, 56
    // tokens 179.5 / 176.5 us), five and six with more 0.995 to 0.999, not worth the sizes that lose (14336 x 4096, 5 blocks, 100 tokens 57.6 / 58.1): these keep to fp32.
    constexpr bool PAIRS = I <= 4 || TT == 4;
    constexpr int VT = I * CL_IMAGE, BUFFER = VT + TT * CL_IMAGE, XK = (TT + 3) / 4;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int row = lane & 31, h = lane >> 5;       // in the rebuild
    const int lm = lane & 15, g = lane >> 4;        // in the second product
    // nibble v, column j of its four (first in the top bit): the sign bit of an fp32 where the bit is set; at LDS address 0
    // and behind it the sign bits of two pairs of fp16
    if (tid < 64) {
        const uint32_t v = tid >> 2, j = tid & 3, first = v >> (3 - 2 * (j & 1)) & 1, second = v >> (2 - 2 * (j & 1)) & 1;
        ((__attribute__((address_space(3))) uint32_t *)lds)[tid] = v >> (3 - j) & 1 ? 0x80000000u : 0u;
        ((__attribute__((address_space(3))) uint32_t *)lds)[CL_HALVES / 4 + tid] = first << 15 | second << 31;
    }
    // every XCD gets a contiguous run of (column group, rows), rows fastest: workgroups with the same slices of x and vt share an L2
    const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, base = nb >> 3, rem = nb & 7;
    const int v = xcd * base + min(xcd, rem) + loc, cg = v / mat.row_groups, rg = v - cg * mat.row_groups;
    const int M = mat.M, all = (N + 255) >> 8, first = cg * mat.spans, last = min(first + mat.spans, all) - 1;
    const uint32_t row_bytes = (uint32_t)N >> 3;
    const int64_t block_bytes = (int64_t)M * row_bytes;

    const int m0 = rg * CL_ROWS + wave * 32, my_row = min(m0 + row, M - 1);
    half8_t uf[I];
    uint4_t sw[I];
    const uint8_t *const signs = mat.packed + (uint64_t)((uint32_t)my_row * row_bytes);
    auto request_signs = [&](int i, int span) {
        sw[i] = *reinterpret_cast<const uint4_t *>(signs + i * block_bytes + min((uint32_t)(span * 32 + 16 * h), row_bytes - 16u));
    };
#pragma unroll
    for (int i = 0; i < I; i++) {
        const half_t *ur = mat.u + ((int64_t)i * M + my_row) * K;
        if (K >= 8) {
            uf[i] = *reinterpret_cast<const cl_half8_any *>(ur + (h ? K - 8 : 0));       // (fewer than 16 ranks: the row's last eight)
        } else {
            const half4_t a = *reinterpret_cast<const cl_half4_any *>(ur), b = *reinterpret_cast<const cl_half4_any *>(ur + K - 4);
            uf[i] = (half8_t){a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]};           // (fewer than 8: its first and last four)
        }
        request_signs(i, first);
    }

    if (K < 16) {                                   // ranks in their places, zeros in those of the ones that do not exist
#pragma unroll
        for (int i = 0; i < I; i++) {
            half8_t o = uf[i];
#pragma unroll
            for (int e = 0; e < 8; e++) {
#pragma unroll
                for (int d = 0; d < 8; d++)
                    if (K >= 8 ? h && d == e + 16 - K : e >= 4 && d == e + 8 - K) o[e] = uf[i][d];
                if (8 * h + e >= K) o[e] = (half_t)0;
            }
            uf[i] = o;
        }
    }

    // ---- staging: image column 32 h' + c is column 128 h' + 32 q + c of the span; columns beyond N are zero -------------------
    // vt: wave = block, lane = (rank pair, piece of 8 columns); x: a thread's pieces of 8 columns of a token
    half8_t vpre[2], xpre[XK];
    const int rp = lane & 7, pc = lane >> 3;
    auto request = [&](int span, int q) {
        const int n0 = span * 256 + 32 * q;
        if (wave < I) {
            const int col = n0 + 128 * (pc >> 2) + 8 * (pc & 3);
            const half_t *src = mat.vt + (int64_t)wave * K * N + min(col, N - 8);
#pragma unroll
            for (int r = 0; r < 2; r++) {
                vpre[r] = *reinterpret_cast<const half8_t *>(src + (int64_t)min(2 * rp + r, K - 1) * N);
                if (col >= N || 2 * rp + r >= K) vpre[r] = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
            }
        }
#pragma unroll
        for (int k = 0; k < XK; k++) {
            const int t = (tid >> 3) + 64 * k, c = tid & 7, col = n0 + 128 * (c >> 2) + 8 * (c & 3);
            xpre[k] = *reinterpret_cast<const half8_t *>(x + (int64_t)min(t, T - 1) * N + min(col, N - 8));
            if (col >= N) xpre[k] = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
        }
    };
    auto write = [&](int buffer) {
        const cl_bytes to = lds + CL_TABLE + buffer * BUFFER;
        if (wave < I) {
#pragma unroll
            for (int e = 0; e < 8; e++) *(cl_half2_rw)(to + wave * CL_IMAGE + (8 * pc + (e ^ pc)) * 32 + 4 * rp) = (half2_t){vpre[0][e], vpre[1][e]};
        }
#pragma unroll
        for (int k = 0; k < XK; k++) {
            const int t = (tid >> 3) + 64 * k, c = tid & 7;
            if (TT % 4 == 0 || t < TT * 16) *(cl_half8_rw)(to + VT + t * 128 + ((c ^ ((t >> 1) & 7)) * 16)) = xpre[k];
        }
    };

    float4_t y[TT][2];
#pragma unroll
    for (int tt = 0; tt < TT; tt++) y[tt][0] = y[tt][1] = (float4_t){0.f, 0.f, 0.f, 0.f};
    const int acol = 32 * ((row >> 2) & 1) + 4 * (row >> 3) + (row & 3);     // this lane's column of a vt fragment, + 16 p
    const int vread[2] = {(acol ^ ((acol >> 3) & 7)) * 32 + 16 * h, ((acol + 16) ^ (((acol + 16) >> 3) & 7)) * 32 + 16 * h};

    request(first, 0);
    write(0);
#pragma clang loop unroll(disable)
    for (int span = first; span <= last; span++) {
        cl_for<4>([&](auto qc) {
            constexpr int q = decltype(qc)::value, buffer = q & 1;
            __syncthreads();                         // the image is complete, and nobody reads the other one any more
            if (q < 3)
                request(span, q + 1);
            else
                request(min(span + 1, last), 0);     // (behind the last chunk: its image is not used)
            const cl_bytes image = lds + CL_TABLE + buffer * BUFFER;
            // Steps s = 2 i + p: the sums of patch p change sign ahead of block i (i = I: behind the last), then block i's product is added;
            // masks and vt fragments are looked up a step ahead (see tile.hip)
            float16_t acc[2];
            uint4_t mask[2][4];
            uint2_t pair_mask[2][4];                 // behind the last block: of rounded pairs
            uint4_t wt[2][2];                        // the rounded patches: columns 8 e .. + 7 of this lane's 16
            half8_t vf[2];
            uint32_t flip = 0, flip4 = 0;
            auto look_up = [&](auto sc) {
                constexpr int s = decltype(sc)::value, i = s / 2, p = s % 2;
                if constexpr (s < 2 * I + 2) {
                    if constexpr (p == 0) {
                        flip = i < I ? sw[i - 1][q] ^ sw[i < I ? i : 0][q] : ~sw[i - 1][q];
                        flip4 = flip << 4;
                        asm("" : "+v"(flip4));
                        if constexpr (q == 3) request_signs(i - 1, min(span + 1, last));
                    }
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const uint32_t at = ((k & 1 ? flip4 : flip) >> (8 * (2 * p + (k >> 1)))) & 0xF0u;
                        if constexpr (i < I || !PAIRS) mask[s & 1][k] = *(cl_uint4)(uintptr_t)at;
                        else pair_mask[s & 1][k] = *(cl_uint2)(uintptr_t)(at + CL_HALVES);
                    }
                    if constexpr (i < I) vf[s & 1] = *(cl_half8)(image + i * CL_IMAGE + vread[p]);
                }
            };
#pragma unroll
            for (int p = 0; p < 2; p++)
                acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(*(cl_half8)(image + vread[p]), uf[0], (float16_t){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            look_up(std::integral_constant<int, 2>{});
            __builtin_amdgcn_sched_barrier(0);
            cl_for<2 * I>([&](auto kc) {
                constexpr int s = decltype(kc)::value + 2, i = s / 2, p = s % 2;
                const half8_t a = vf[s & 1];
                look_up(std::integral_constant<int, s + 1>{});
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (i < I || !PAIRS) {
                    asm volatile("" : "+v"(mask[s & 1][0]), "+v"(mask[s & 1][1]), "+v"(mask[s & 1][2]), "+v"(mask[s & 1][3]));   // (one wait for the four)
#pragma unroll
                    for (int k = 0; k < 16; k++) {
                        const float sum = acc[p][k];
                        const uint32_t m = mask[s & 1][k / 4][k % 4];
                        acc[p][k] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, sum) ^ m);
                    }
                    if constexpr (i < I) acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, uf[i < I ? i : 0], acc[p], 0, 0, 0);
                    asm volatile("" : "+v"(acc[p]));
                } else {
                    // (rounded first, once, to fp16, the sign changed on the rounded pairs: half the operations, the same bits)
                    asm volatile("" : "+v"(pair_mask[s & 1][0]), "+v"(pair_mask[s & 1][1]), "+v"(pair_mask[s & 1][2]), "+v"(pair_mask[s & 1][3]));
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const half2_t two = {(half_t)acc[p][2 * k], (half_t)acc[p][2 * k + 1]};
                        wt[p][k / 4][k % 4] = __builtin_bit_cast(uint32_t, two) ^ pair_mask[s & 1][k / 2][k % 2];
                    }
                    asm volatile("" : "+v"(wt[p][0]), "+v"(wt[p][1]));
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            // The rows sorted out (see tile.hip): lane group g holds columns 32 (g / 2) + 16 p + 8 (g % 2) .. + 7 of the image
#pragma unroll
            for (int p = 0; p < 2; p++) {
                if constexpr (!PAIRS) {
#pragma unroll
                    for (int k = 0; k < 8; k++) wt[p][k / 4][k % 4] = __builtin_bit_cast(uint32_t, (half2_t){(half_t)acc[p][2 * k], (half_t)acc[p][2 * k + 1]});
                }
                uint4_t lo, hi;
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const auto r = __builtin_amdgcn_permlane16_swap(wt[p][0][k], wt[p][1][k], false, false);
                    lo[k] = r[0];
                    hi[k] = r[1];
                }
                half8_t w0 = __builtin_bit_cast(half8_t, lo), w1 = __builtin_bit_cast(half8_t, hi);
                if (span * 256 + 128 >= N && g >= 2) w0 = w1 = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};   // no such columns: an infinity in u must not make a NaN of them
                const cl_bytes xrow = image + VT + lm * 128 + (((4 * (g >> 1) + 2 * p + (g & 1)) ^ ((lm >> 1) & 7)) * 16);
#pragma unroll
                for (int tt = 0; tt < TT; tt++) {
                    const half8_t xf = *(cl_half8)(xrow + tt * CL_IMAGE);
                    y[tt][0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf, w0, y[tt][0], 0, 0, 0);
                    y[tt][1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf, w1, y[tt][1], 0, 0, 0);
                }
            }
            write(buffer ^ 1);
        });
    }
    float *const part = mat.part + (int64_t)cg * T * M;
#pragma unroll
    for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int t = 16 * tt + 4 * g + j, m = m0 + 16 * r + lm;
                if (t < T && m < M) part[(int64_t)t * M + m] = y[tt][r][j];
            }
}

template <int TT, int I>
int launch_column(const ColumnMat &m, int grid, const half_t *x, int N, int T, int K, hipStream_t s) {
    const size_t lds = CL_TABLE + 2 * (size_t)(I + TT) * CL_IMAGE;
    static bs_lds_grant granted[BS_MAX_DEVICES];
    const int st = bs_allow_lds((const void *)column_forward_kernel<TT, I>, lds, granted);
    if (st != BS_OK) return st;
    column_forward_kernel<TT, I><<<grid, 64 * CL_WAVES, lds, s>>>(m, x, N, T, K);
    BS_LAUNCH_CHECK();
    return BS_OK;
}
// Token tiles: as many as there are, from four on.  us with four, six or eight / with these: 14336 x 4096, 5 blocks, 100 tokens (7) 58.9 / 57.9, 28672 x 8192, 3, 80 (5)
// 113.4 / 109.7, 11520 x 11904, 3, 112 83.0 / 81.1, 6144 x 4096, 1, 66 21.4 / 20.7, 4096 x 4096, 6, 75 25.8 / 25.7.
// (registers: 8 per token tile and 10 per block)
constexpr int max_blocks(int token_tiles) { return token_tiles == 4 ? 8 : token_tiles <= 6 ? 7 : 6; }
template <int TT>
int launch_blocks(int I, const ColumnMat &m, int grid, const half_t *x, int N, int T, int K, hipStream_t s) {
    switch (I) {
        case 1: return launch_column<TT, 1>(m, grid, x, N, T, K, s);
        case 2: return launch_column<TT, 2>(m, grid, x, N, T, K, s);
        case 3: return launch_column<TT, 3>(m, grid, x, N, T, K, s);
        case 4: return launch_column<TT, 4>(m, grid, x, N, T, K, s);
        case 5: return launch_column<TT, 5>(m, grid, x, N, T, K, s);
        case 6: return launch_column<TT, 6>(m, grid, x, N, T, K, s);
        case 7: if constexpr (max_blocks(TT) >= 7) return launch_column<TT, 7>(m, grid, x, N, T, K, s); break;
        case 8: if constexpr (max_blocks(TT) >= 8) return launch_column<TT, 8>(m, grid, x, N, T, K, s); break;
    }
    return BS_ERR_SHAPE;
}
int token_tiles(int T) { return T <= 64 ? 4 : (int)bs_cdiv(T, 16); }
int launch_tokens(const ColumnMat &m, int I, int grid, const half_t *x, int N, int T, int K, hipStream_t s) {
    switch (token_tiles(T)) {
        case 4: return launch_blocks<4>(I, m, grid, x, N, T, K, s);
        case 5: return launch_blocks<5>(I, m, grid, x, N, T, K, s);
        case 6: return launch_blocks<6>(I, m, grid, x, N, T, K, s);
        case 7: return launch_blocks<7>(I, m, grid, x, N, T, K, s);
        default: return launch_blocks<8>(I, m, grid, x, N, T, K, s);
    }
}

}  // namespace

#ifdef COLUMN_RANKS
int bs_launch_column_ranks(const ColumnMat &m, int I, int grid, const half_t *x, int N, int T, int K, hipStream_t s) { return launch_tokens(m, I, grid, x, N, T, K, s); }
#else
namespace {

struct ColumnPlan {
    int row_groups, spans, groups;
};
ColumnPlan make_column_plan(int M, int N) {
    ColumnPlan p;
    p.row_groups = (int)bs_cdiv(M, CL_ROWS);
    const int all = (int)bs_cdiv(N, 256);
    int groups = 256 / p.row_groups;                // one workgroup per CU
    if (groups > all) groups = all;
    if (groups < 1) groups = 1;
    p.spans = (int)bs_cdiv(all, groups);
    p.groups = (int)bs_cdiv(all, p.spans);
    return p;
}

}  // namespace

// From how many weights on this kernel runs: with fewer there are 256 x 256 squares for fewer than about 3/4 of the CUs, and the start and end
// of a workgroup (10 to 15 us with the summing launch) are most of it.  Measured (us, walked or panel kernel -> this one, M x N x I x T):
// 512 x 640 x 5 x 71 10.1 -> 14.3, 4893 x 384 x 2 x 109 13.0 -> 14.6, 1518 x 5760 x 2 x 117 20.7 -> 23.1, 2023 x 5376 x 2 19.4 -> 21.5;
// 1781 x 6656 x 1 x 50 17.9 -> 14.9, 16256 x 768 x 5 x 111 29.6 -> 28.5, 4480 x 3840 x 3 x 87 31.8 -> 24.2, 3712 x 8448 x 6 x 110 60.4 -> 41.4,
// 27520 x 4608 x 5 x 125 156 -> 106, 11520 x 11904 x 3 x 125 156 -> 78.
constexpr int64_t CL_MIN_WEIGHTS = 11ll << 20;

// Column groups (partial sums per output) when this kernel takes the shape, else 0.
int bs_column_partials(int I, int M, int N, int K, int T) {
    if (bs_prefill_mode() != 0 || K < 4 || K > 16 || I < 1 || T < CL_MIN_T || T > CL_MAX_T || I > max_blocks(token_tiles(T)) || M < 1 || N < SF_COLS || N % SF_COLS != 0) return 0;
    if ((int64_t)M * N < CL_MIN_WEIGHTS || (int64_t)M * (N >> 3) >= ((int64_t)1 << 32)) return 0;       // a row's signs within a 32-bit byte offset
    return make_column_plan(M, N).groups;
}

// ... and the columns of one.
int bs_column_width(int I, int M, int N, int K, int T) { return bs_column_partials(I, M, N, K, T) > 0 ? 256 * make_column_plan(M, N).spans : 0; }

int bs_launch_column(const uint8_t *packed, const half_t *u, const half_t *vt, int I, int M, float *part, const half_t *x, int N, int K, int T, hipStream_t s) {
    const int groups = bs_column_partials(I, M, N, K, T);
    if (groups == 0 || !bs_aligned(x, 16) || !bs_aligned(packed, 16) || !bs_aligned(vt, 16) || !bs_aligned(u, K == 16 ? 16 : 2)) return BS_ERR_SHAPE;
    const ColumnPlan p = make_column_plan(M, N);
    const ColumnMat m{packed, u, vt, part, M, p.row_groups, p.spans};
    const int grid = p.row_groups * p.groups;
    return K == 16 ? launch_tokens(m, I, grid, x, N, T, K, s) : bs_launch_column_ranks(m, I, grid, x, N, T, K, s);
}
#endif
