// Packed-sign GEMV for one to three tokens on gfx950's sparse matrix instruction, v_smfmac_f32_16x16x64_f16: the sign bits are its index operand.
//
//   y[t, m] = sum_i sum_r u_i[m, r] * ( sum_n s_i[m, n] * vt_i[r, n] * x[t, n] )
//
// The instruction multiplies a 16 x 64 matrix A, of which two in four neighbours are given and the others are zero, by a dense 64 x 16 matrix B; two bits
// per given element say where it stands.  Here the four rows of B that belong together are -vt[r, n], +vt[r, n], -vt[r, n'], +vt[r, n'] (r: B's 16 columns), the two given
// elements of A are x[t, n] and x[t, n'], the same in all of its 16 rows, and their places are s[m, n] and 2 + s[m, n']: every product is x * (+-vt), exact in fp32 as
// the halves it is made of, and D[m, r] is the inner sum.  Nothing is rounded before y: error against float64 ahead of that rounding 1e-7 to 4e-7 (drawn factors; the
// kernels that round vt * x or the weight to fp16: 2 to 3e-4).
//
// Operands.  The index of 32 columns takes two VALU instructions per 16 signs and row tile and no table: a word of 32 signs has every second bit where an index has its low bit,
// (w & 0x55555555) | 0x88888888 serves the odd columns, the same of w >> 1 the even ones, 16 of them per half of the word (the instruction picks the half).  A lane loads the
// 16 sign bytes of 128 columns of its row: 16 operands per unit of 512 columns.  B goes through LDS once per workgroup as the pairs (-v, +v) in operand order.  x: lane j
// of every row of 16 lanes holds operand j's elements, which v_mov_b32_dpp row_newbcast hands to the others; tokens share everything else.
//
// Units are (block, row tile of 128 R rows, 512 columns), the column chunk fastest; partition over one workgroup of 8 waves per CU, partial sums and summing launch as gemv.hip has
// them.  Signs, vt and x are requested one unit ahead; the two register sets of the signs take turns without being copied (a copy at the end of a unit waits for the
// requests it is there to overlap: 43.0 against 41.0 us on 16 blocks of 4096 x 14336).  u comes by way of LDS while the last unit of a row of units is multiplied.  Columns beyond
// N have x = 0 and vt = 0 (0 times an infinity further left would be NaN); rows beyond M and ranks beyond K repeat the last one and are left out at the end.
//
// What bounds it: with four row tiles a unit is 128 matrix instructions per SIMD, 8.9 ns each on their own and 10.3 with three VALU instructions between them, and 256 KB of B out
// of LDS, a us as well: 2.0 us measured where units follow each other (4.2 TB/s), of which the multiplication takes 1.5 with the signs in L2.  A call with one unit per workgroup
// takes 4 to 7 us: 1.5 until vt has arrived, 0.7 until everybody's has, the unit, 0.7 for u and the sums, and the launch.  us in a replayed graph, tile kernel / this, one token: 4096 x 11008, 4 blocks
// 25.7 / 17.7, 8 39.3 / 25.6 (other shapes at sparse_plan).  Measured and not kept: the pairs made from single halves in registers, half the LDS traffic for two VALU
// instructions per product (42.3 -> 45.3 us on 16 blocks of 4096 x 14336); eight row tiles (64 KB per unit arrive too late: 41.6, and 16.1 instead of 13.7 on 4096 x 11008); both
// 64-byte halves of a line of sign bytes requested together, 1024 columns ahead (44.0, 15.3); operands of B two ahead and of x one ahead (42.2, 14.6 against 43.8, 15.0 in that run).
#include "common.h"
#include "gemv_shared.h"

#include <type_traits>
#include <utility>

namespace {

typedef _Float16 half16_t __attribute__((ext_vector_type(16)));

template <class F, int... Is>
__device__ __forceinline__ void sp_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void sp_for(F &&f) {
    sp_for_impl(f, std::make_integer_sequence<int, N>{});
}

constexpr int SP_WAVES = 8, SP_THREADS = 64 * SP_WAVES;

// raw buffer descriptor from a pointer: no stride, no range limit short of 4 GiB (every offset used with it is checked
// by construction: rows clamped to M, columns to N; vt's ends with the block, what lies beyond reads as zeros)
__device__ __forceinline__ __amdgpu_buffer_rsrc_t sp_rsrc(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, -1, 0x00020000);
}

// a barrier that waits for this wave's LDS accesses, not for what it has requested from memory
__device__ __forceinline__ void sp_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (0 << 8));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}

// the sum over the 16 lanes that share lane / 16, in every one of them
__device__ __forceinline__ float sp_row_sum(float v) {
    auto add = [&](auto ctrl) {
        v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), decltype(ctrl)::value, 0xF, 0xF, true));
    };
    add(std::integral_constant<int, 0xB1>{});        // quad_perm 1 0 3 2
    add(std::integral_constant<int, 0x4E>{});        // quad_perm 2 3 0 1
    add(std::integral_constant<int, 0x141>{});       // row_half_mirror
    add(std::integral_constant<int, 0x140>{});       // row_mirror
    return v;
}

template <int R, int T>
struct SparseKernel {
    static constexpr int RW = SP_WAVES * R * 16;                                   // rows per workgroup
    static constexpr int VT = 32 * 1024, X = T * 1024, U = RW * 32;                // bytes of LDS: each twice
    static constexpr int LDS = 2 * (VT + X + U);
};

template <int R, int T>
__global__ __launch_bounds__(SP_THREADS, 2) void gemv_sparse_kernel(const GemvGroup grp, const half_t *__restrict__ x, int N, int K, int n_units) {
    typedef SparseKernel<R, T> SK;
    constexpr int RW = SK::RW;
    extern __shared__ __attribute__((aligned(16))) char lds[];
    char *const vt_l = lds, *const x_l = vt_l + 2 * SK::VT, *const u_l = x_l + 2 * SK::X;

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, g = lane >> 4;

    // XCD-aware slot -> range (workgroups are dealt round-robin to the 8 XCDs; each XCD gets a
    // contiguous run of ranges), then the matrix of the group this workgroup belongs to
    int wg;
    {
        const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
        const int base = nb >> 3, rem = nb & 7;
        wg = xcd * base + min(xcd, rem) + loc;
    }
    GemvMat mat = grp.m[0];
#pragma unroll
    for (int j = 1; j < GEMV_MAX_GROUP; j++)
        if (j < grp.n && wg >= grp.m[j].first_wg) mat = grp.m[j];
    wg -= mat.first_wg;
    const uint8_t *__restrict__ packed = mat.packed;
    const half_t *__restrict__ u = mat.u;
    const half_t *__restrict__ vt = mat.vt;
    float *__restrict__ part = mat.part;
    const int M = mat.M, row_tiles = mat.row_tiles, kmax = mat.kmax;
    const Split sp = mat.sp;
    const int u_begin = sp.start(wg), u_end = sp.start(wg + 1);
    if (u_begin >= u_end) return;
    const uint32_t row_bytes = (uint32_t)N >> 3;

    // ---- requests: signs, vt and x of the step after the one being multiplied -------------------------------------------------
    uint32_t qoff[R];                                // this lane's row in each row tile of the wave
    __amdgpu_buffer_rsrc_t rq, rv;                   // signs and vt of the block
    const __amdgpu_buffer_rsrc_t rx = sp_rsrc(x);
    auto set_row = [&](int rowid) {
        const int i = rowid / row_tiles, rt = rowid - i * row_tiles;
#pragma unroll
        for (int r = 0; r < R; r++) qoff[r] = (uint32_t)min(rt * RW + (wave * R + r) * 16 + lm, M - 1) * row_bytes;
        rq = sp_rsrc(packed + (int64_t)i * M * row_bytes);
        rv = __builtin_amdgcn_make_buffer_rsrc(const_cast<half_t *>(vt + (int64_t)i * K * N), 0, K * N * 2, 0x00020000);
    };
    auto request = [&](uint4_t (&w)[R], int c) {
        const uint32_t at = min((uint32_t)c * 64u + 16u * g, row_bytes - 16u);
#pragma unroll
        for (int r = 0; r < R; r++) w[r] = __builtin_amdgcn_raw_buffer_load_b128(rq, (int)(qoff[r] + at), 0, 0);
    };
    // vt: a wave takes 64 columns, a lane 8 columns of one rank at a time; x: a thread 16 columns of one token
    half8_t pv[2], px[2];
    const uint32_t rank_at = (uint32_t)min(lm, K - 1) * (uint32_t)N * 2u;
    const bool px_mine = tid < 32 * T;
    auto request_z = [&](int c) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int col = 512 * c + 8 * (8 * wave + 4 * k + g);
            pv[k] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rv, (int)(col < N ? rank_at + 2 * col : 0x80000000u), 0, 0));
        }
        if (px_mine) {
            const int col = 512 * c + 16 * (tid & 31), at = 2 * ((tid >> 5) * N + min(col, N - 16));
            px[0] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rx, at, 0, 0));
            px[1] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rx, at + 16, 0, 0));
            if (col >= N) px[0] = px[1] = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
        }
    };
    half2_t minus_plus = {(half_t)-1, (half_t)1};
    asm("" : "+v"(minus_plus));
    auto leave_z = [&](int buf) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int piece = 8 * wave + 4 * k + g, p = piece & 63, s = (p & 15) >> 1, half = p >> 5, to_g = 2 * ((p >> 4) & 1) + (p & 1);
            char *to = vt_l + buf * SK::VT + s * 4096 + half * 1024 + (16 * to_g + lm) * 16;
#pragma unroll
            for (int e = 0; e < 2; e++) {            // odd columns, even columns
                half8_t o;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const half_t val = pv[k][7 - 2 * j - e];
                    const half2_t pair = (half2_t){val, val} * minus_plus;
                    o[2 * j] = pair[0];
                    o[2 * j + 1] = pair[1];
                }
                *reinterpret_cast<half8_t *>(to + e * 2048) = o;
            }
        }
        if (px_mine) {
            const int j = tid & 31, gg = j >> 3, op = j & 7;
            char *to = x_l + buf * SK::X + (tid >> 5) * 1024 + op * 128 + gg * 16;
            const half8_t a = px[0], b = px[1];
            *reinterpret_cast<half8_t *>(to) = (half8_t){a[7], a[5], a[3], a[1], b[7], b[5], b[3], b[1]};
            *reinterpret_cast<half8_t *>(to + 64) = (half8_t){a[6], a[4], a[2], a[0], b[6], b[4], b[2], b[0]};
        }
    };

    constexpr int SETS = R * T <= 2 ? 2 : 1;         // (few accumulators: odd and even columns apart)
    float4_t acc[SETS][R][T];
    auto clear_acc = [&]() {
#pragma unroll
        for (int s = 0; s < SETS; s++)
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < T; t++) acc[s][r][t] = (float4_t){0.f, 0.f, 0.f, 0.f};
    };
    clear_acc();

    // ---- one unit: sixteen operands of 32 columns ------------------------------------------------------------------------------
    uint32_t even_bits = 0x55555555u, index_base = 0x88888888u;
    asm("" : "+s"(even_bits));
    asm("" : "+v"(index_base));
    auto consume = [&](const uint4_t (&w)[R], int buf) {
        const char *vb = vt_l + buf * SK::VT + lane * 16;
        half8_t v[2][2];
        uint4_t xs[T];                               // lane lm of a row of 16: operand lm of x
#pragma unroll
        for (int t = 0; t < T; t++) xs[t] = *reinterpret_cast<const uint4_t *>(x_l + buf * SK::X + t * 1024 + lm * 64 + g * 16);
        auto fetch = [&](auto oc) {                  // operand o = 4 p + 2 h + e
            constexpr int o = decltype(oc)::value;
            v[o & 1][0] = *reinterpret_cast<const half8_t *>(vb + o * 2048);
            v[o & 1][1] = *reinterpret_cast<const half8_t *>(vb + o * 2048 + 1024);
        };
        uint32_t idx[2][R];
        fetch(std::integral_constant<int, 0>{});
        sp_for<16>([&](auto oc) {
            constexpr int o = decltype(oc)::value, p = o >> 2, h = (o >> 1) & 1, e = o & 1;
            if constexpr (o + 1 < 16) fetch(std::integral_constant<int, (o + 1) & 15>{});
            if constexpr (h == 0) {
#pragma unroll
                for (int r = 0; r < R; r++) idx[e][r] = ((w[r][p] >> e) & even_bits) | index_base;
            }
            half16_t b;
#pragma unroll
            for (int k = 0; k < 16; k++) b[k] = v[o & 1][k >> 3][k & 7];
            half8_t xa[T];
#pragma unroll
            for (int t = 0; t < T; t++) {
                uint4_t all;
#pragma unroll
                for (int k = 0; k < 4; k++) all[k] = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)xs[t][k], 0x150 + o, 0xF, 0xF, true);      // row_newbcast
                xa[t] = __builtin_bit_cast(half8_t, all);
            }
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < T; t++)
                    acc[e % SETS][r][t] = __builtin_amdgcn_smfmac_f32_16x16x64_f16(xa[t], b, acc[e % SETS][r][t], (int)idx[e][r], 0, h);
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < T; t++) asm volatile("" : "+v"(acc[e % SETS][r][t]));
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // ---- u of a row of units: requested while its last step is multiplied, by way of LDS -----------------------------------
    constexpr int UQ = RW * 4 / SP_THREADS;          // pieces of four ranks per thread
    half4_t pu[UQ];
    auto request_u = [&](int rowid) {
        const int i = rowid / row_tiles, rt = rowid - i * row_tiles;
#pragma unroll
        for (int k = 0; k < UQ; k++) {
            const int q = tid + k * SP_THREADS, row = min(rt * RW + (q >> 2), M - 1), r0 = 4 * (q & 3);
            const half_t *up = u + ((int64_t)i * M + row) * K;
            if (K == 16) {
                pu[k] = *reinterpret_cast<const half4_t *>(up + r0);
            } else {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const half_t val = up[min(r0 + e, K - 1)];
                    pu[k][e] = r0 + e < K ? val : (half_t)0;
                }
            }
        }
    };
    auto leave_u = [&](int parity) {
#pragma unroll
        for (int k = 0; k < UQ; k++) *reinterpret_cast<half4_t *>(u_l + parity * SK::U + (tid + k * SP_THREADS) * 8) = pu[k];
    };
    // D[row 4 g + j, rank lm]: times u, added over the ranks
    auto flush = [&](int rowid, bool row_done, int parity) {
        const int i = rowid / row_tiles, rt = rowid - i * row_tiles;
        const int slot = wg - sp.owner(rowid * n_units);
        const half_t *ub = reinterpret_cast<const half_t *>(u_l + parity * SK::U) + (wave * R * 16 + 4 * g) * 16 + lm;
        constexpr int Q = (R + 3) / 4;               // lanes take over four tiles' rows at a time: lane (g, lm) row 4 g + lm % 4 of tile lm / 4
        float own[Q][T];
#pragma unroll
        for (int r = 0; r < R; r++)
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const float uv = (float)ub[(r * 16 + j) * 16];
#pragma unroll
                for (int t = 0; t < T; t++) {
                    float d = acc[0][r][t][j];
                    if (SETS == 2) d += acc[SETS - 1][r][t][j];
                    const float sum = sp_row_sum(lm < K ? d * uv : 0.f);     // (lanes beyond K repeat rank K - 1)
                    if (r % 4 == 0 && j == 0) own[r / 4][t] = sum;
                    else own[r / 4][t] = lm == 4 * (r % 4) + j ? sum : own[r / 4][t];
                }
            }
        const int tile = lm >> 2;
#pragma unroll
        for (int q = 0; q < Q; q++) {
            const int row = rt * RW + (wave * R + 4 * q + tile) * 16 + 4 * g + (lm & 3);
            if ((R % 4 != 0 && 4 * q + tile >= R) || row >= M) continue;
#pragma unroll
            for (int t = 0; t < T; t++) {
                float *to = part + (((int64_t)i * kmax + slot) * T + t) * M + row;
                *to = own[q][t];
                // the workgroup that finishes a row of units zero-fills the slots above its own (nobody writes
                // them): the summing kernel adds all kmax slots blindly
                if (row_done)
                    for (int dead = slot + 1; dead < kmax; dead++) {
                        to += (int64_t)T * M;
                        *to = 0.f;
                    }
            }
        }
        clear_acc();
    };

    int rowid = u_begin / n_units, c = u_begin % n_units, left = u_end - u_begin, parity = 0;
    set_row(rowid);
    uint4_t even[R], odd[R];
    // a unit that is not the last: w is multiplied, the next one requested into `to`
    auto unit = [&](const uint4_t (&w)[R], uint4_t (&to)[R], int buf) {
        const bool crossing = c + 1 == n_units;      // the next unit starts another row of units
        c = crossing ? 0 : c + 1;
        if (crossing) {
            request_u(rowid);
            set_row(rowid + 1);
        }
        request_z(c);
        request(to, c);
        __builtin_amdgcn_sched_barrier(0);
        consume(w, buf);
        __builtin_amdgcn_sched_barrier(0);
        leave_z(buf ^ 1);
        if (crossing) leave_u(parity);
        sp_barrier();
        if (crossing) {
            flush(rowid, true, parity);
            parity ^= 1;
            rowid++;
        }
    };
    auto last = [&](const uint4_t (&w)[R], int buf) {
        request_u(rowid);
        __builtin_amdgcn_sched_barrier(0);
        consume(w, buf);
        leave_u(parity);
        sp_barrier();
        flush(rowid, u_end % n_units == 0, parity);
    };
    request_z(c);
    request(even, c);
    leave_z(0);
    sp_barrier();
    while (true) {
        if (left == 1) {
            last(even, 0);
            break;
        }
        unit(even, odd, 0);
        if (left == 2) {
            last(odd, 1);
            break;
        }
        unit(odd, even, 1);
        left -= 2;
    }
}

template <int R, int T>
int launch_sparse(int grid, const GemvGroup &grp, const half_t *x, int N, int K, int n_units, hipStream_t s) {
    const size_t lds = SparseKernel<R, T>::LDS;
    static bs_lds_grant granted[BS_MAX_DEVICES];
    const int st = bs_allow_lds((const void *)gemv_sparse_kernel<R, T>, lds, granted);
    if (st != BS_OK) return st;
    gemv_sparse_kernel<R, T><<<grid, SP_THREADS, lds, s>>>(grp, x, N, K, n_units);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

}  // namespace

// Whole 128-column groups, one to three tokens; rows per workgroup 128 R.  (A block of vt, and x, lie within 31-bit byte offsets.)
bool bs_gemv_sparse_takes(int N, int K, int R, int T) {
    return N >= 128 && N % 128 == 0 && K >= 1 && K <= 16 && T >= 1 && T <= 3 && (R == 1 || R == 2 || R == 4) && (int64_t)(K > T ? K : T) * N * 2 < ((int64_t)1 << 31);
}

int bs_launch_gemv_sparse(int R, int T, int grid, const GemvGroup &grp, const half_t *x, int N, int K, int n_units, hipStream_t s) {
    if (!bs_gemv_sparse_takes(N, K, R, T) || n_units != (int)bs_cdiv(N, 512)) return BS_ERR_SHAPE;
    switch (10 * T + R) {
#define SP_CASE(t, r) case 10 * t + r: return launch_sparse<r, t>(grid, grp, x, N, K, n_units, s);
        SP_CASE(1, 1) SP_CASE(1, 2) SP_CASE(1, 4)
        SP_CASE(2, 1) SP_CASE(2, 2) SP_CASE(2, 4)
        SP_CASE(3, 1) SP_CASE(3, 2) SP_CASE(3, 4)
#undef SP_CASE
        default: return BS_ERR_SHAPE;
    }
}
