// Dense fp16 contraction y[T, M] = x[T, N] @ w[M, N]^T (+ bias) on gfx950 MFMA.
//
// Both operands are contiguous along the contracted index N, which is what
// v_mfma_f32_32x32x16_f16 wants: a lane supplies eight consecutive k of one
// row (A = tokens) or one column (B = features), i.e. one 16-byte read per
// fragment.
//
// With N a multiple of 64, every tile behind a rebuilt weight from 33 tokens on is gemm_pipe.hip's, and of bs_linear_f16's those of 128 x 128 and more and
// most of 64 x 64; this file holds the others and the choice.  linear_f16_kernel: WT x WF waves of AT x AF MFMA tiles each, k-steps of GK columns through two
// LDS buffers; rows are padded by 8 halves so that the lanes served per LDS cycle hit disjoint banks.  Four shapes:
// 256 x 256 (8 waves of 128 x 64, GK = 32, three register sets of pieces in flight), 128 x 256 (8 waves of 64 x 64) and
// 128 x 128 (4 waves) for N % 64 != 0, and 64 x 64 (4 waves, two workgroups per CU, GK = 128: half as many barriers) for
// problems too small to fill the chip with anything larger (N % 64 == 0: see pipe_64).
// The loop is software-pipelined at three levels, all through registers:
//   - global requests run NS k-steps ahead through NS register sets (four where the registers allow it: the
//     kernel waits for requests more than for anything else, and a fourth set is worth 3 to 13 %; five and six were
//     no better), all of them unconditional buffer loads: descriptor,
//     32-bit lane offset, scalar k offset;
//   - the LDS writes of step s + 1 and the requests of step s + NS are cut into one
//     portion per MFMA group instead of one burst per step;
//   - MFMA fragments are read from LDS one group ahead of use, the first group of the
//     next step right behind the barrier.
// One barrier per step.  On this part LDS takes b128 reads at about 460 B/ns per CU
// and b128 writes at about 165 B/ns (independent of the lane-to-address map as long as
// rows are padded), global requests at 64 B per clock: with 64 x 64 per-wave tiles the
// LDS time equals the MFMA time, which is what the larger tiles are for.  Measured dead
// ends: 128 x 128 per-wave tiles with one wave per SIMD (nothing covers a wait), a
// per-workgroup rotation of the k order (less sharing in L2), 16-wave workgroups, requests
// that write LDS directly (global_load_lds_dwordx4: same time per step).
// 33..128 tokens use narrower workgroups of the same kernel (more workgroups for
// the few token rows); up to 32 tokens: linear_skinny_kernel (below).
#include "common.h"
#include <type_traits>
#include <utility>

namespace {

// Compile-time loop (the index is a constant expression inside the body).
template <class F, int... Is>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// LDS rows of a k-step.  GK = 32: 64-byte rows with no padding, the four 16-byte pieces of a
// row XOR-ed with bits 2..3 of the row number - staging writes (four lanes per row, rows 64 bytes
// apart) and fragment reads (sixteen rows, one piece each) then both spread over all banks;
// with padded rows the writes of the 256 x 256 kernel conflicted (SQ_LDS_BANK_CONFLICT about a
// tenth of its cycles).  Wider steps: rows padded by 8 halves (no conflicts measured).
__host__ __device__ constexpr bool lds_swizzled(int gk) { return gk == 32; }
__host__ __device__ constexpr int lds_stride(int gk) { return lds_swizzled(gk) ? gk : gk + 8; }

template <int WT, int WF, int AT, int AF, int GK, bool KTAIL, int NS = 3>
__global__ __launch_bounds__(64 * WT * WF) void linear_f16_kernel(
    const half_t *__restrict__ x, const half_t *__restrict__ w, const half_t *__restrict__ bias,
    half_t *__restrict__ y, int T, int M, int N) {
    constexpr int THREADS = 64 * WT * WF;
    constexpr int BT = WT * AT * 32, BF = WF * AF * 32;      // workgroup tile: tokens x features
    constexpr int ROWS = BT + BF;                            // LDS rows per buffer (x rows, then w rows)
    constexpr int PPR = GK / 8;                              // 16-byte pieces per row and k-step
    constexpr int LSTRIDE = lds_stride(GK);                  // halves per LDS row
    constexpr bool SWZ = lds_swizzled(GK);
    constexpr int JX = BT * PPR / THREADS, JW = BF * PPR / THREADS;   // pieces per thread: x rows, w rows
    static_assert(BT * PPR % THREADS == 0 && BF * PPR % THREADS == 0, "every thread stages whole pieces");
    constexpr int PER_THREAD = JX + JW;
    extern __shared__ __attribute__((aligned(16))) half_t lds_raw[];
    half_t (*lds)[ROWS * LSTRIDE] = reinterpret_cast<half_t (*)[ROWS * LSTRIDE]>(lds_raw);

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int t0 = blockIdx.y * BT, m0 = blockIdx.x * BF;
    const int wt = (wave / WF) * (AT * 32), wf = (wave % WF) * (AF * 32);
    const int l32 = lane & 31, kh = lane >> 5;

    // Loader role.  Piece j of a thread is row tid / PPR + (THREADS / PPR) * j of the x
    // tile (j < JX) or of the w tile, 16-byte piece tid % PPR.  Addresses are a
    // workgroup-uniform pointer (tile origin + k-step, scalar registers) plus a 32-bit
    // per-thread byte offset; rows beyond T or M repeat the last row (their outputs are
    // never stored), so no load in the main loop is conditional.
    const char *xt = reinterpret_cast<const char *>(x + (int64_t)t0 * N);
    const char *wt_ = reinterpret_cast<const char *>(w + (int64_t)m0 * N);
    const int lrow = tid / PPR, lpiece = tid % PPR;
    // raw buffer descriptors over the two tile origins (no stride, no range limit short of 4 GiB: offsets are checked
    // by construction - rows are clamped to the tile, k-steps to the contracted range)
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)xt, 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)wt_, 0, -1, 0x00020000);
    uint32_t off[PER_THREAD];
    int dst[PER_THREAD];
#pragma unroll
    for (int j = 0; j < PER_THREAD; j++) {
        const bool isx = j < JX;
        const int r = lrow + (THREADS / PPR) * (isx ? j : j - JX);
        const int rr = isx ? min(r, T - 1 - t0) : min(r, M - 1 - m0);
        off[j] = (uint32_t)rr * (uint32_t)N * 2u + 16u * lpiece;
        dst[j] = ((isx ? 0 : BT) + r) * LSTRIDE + 8 * (SWZ ? (lpiece ^ ((r >> 2) & 3)) : lpiece);
    }

    float16_t acc[AT][AF];
#pragma unroll
    for (int a = 0; a < AT; a++)
#pragma unroll
        for (int b = 0; b < AF; b++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[a][b][v] = 0.f;

    const int steps = (N + GK - 1) / GK;
    // NS register sets: while step s is multiplied, the pieces of step s + 1 are in one set
    // (landed, on their way to LDS) and those of the steps up to s + NS in flight into the others.
    // Every request is unconditional (past the end the last step is requested again), so
    // the compiler's count of outstanding loads is exact and a wait for one set never
    // drains the other.  KTAIL (N not a multiple of GK): pieces beyond column N are read
    // from column 0 instead and replaced by zeros.
    uint4_t stage[NS][PER_THREAD];
    // part `part` of `parts` of the pieces of one step (the whole step: 0 of 1)
    auto fetch = [&](auto setc, int step_, auto partc, auto partsc) {
        constexpr int set = decltype(setc)::value, part = decltype(partc)::value, parts = decltype(partsc)::value;
        constexpr int j0 = part * PER_THREAD / parts, j1 = (part + 1) * PER_THREAD / parts;
        const int step = min(step_, steps - 1);
        if constexpr (KTAIL) {
            const bool in = step * GK + 8 * lpiece < N;              // N % 8 == 0: a piece is all in or all out
            const uint32_t koff = in ? (uint32_t)step * (GK * 2) : 0u - 16u * lpiece;
#pragma unroll
            for (int j = j0; j < j1; j++) {
                const uint4_t v = *reinterpret_cast<const uint4_t *>((j < JX ? xt : wt_) + (off[j] + koff));
                stage[set][j] = in ? v : (uint4_t){0, 0, 0, 0};
            }
        } else {
            // buffer loads: descriptor (tile origin) + 32-bit lane offset + scalar k offset - no 64-bit address arithmetic
            // per request (4-7 % of the kernel's time with flat global loads)
            const int koff = step * (GK * 2);
#pragma unroll
            for (int j = j0; j < j1; j++)
                stage[set][j] = __builtin_amdgcn_raw_buffer_load_b128(j < JX ? rx : rw, (int)off[j], koff, 0);
        }
    };
    // part `part` of `parts` of a register set goes to LDS (the whole set: 0 of 1)
    auto stash = [&](auto setc, int buf, auto partc, auto partsc) {
        constexpr int set = decltype(setc)::value, part = decltype(partc)::value, parts = decltype(partsc)::value;
#pragma unroll
        for (int j = part * PER_THREAD / parts; j < (part + 1) * PER_THREAD / parts; j++)
            *reinterpret_cast<uint4_t *>(&lds[buf][dst[j]]) = stage[set][j];
    };
    // Fragments travel through two register sets as well: the LDS reads of sub-step
    // kk + 1 are issued before the MFMAs of sub-step kk, and those of the next step's
    // first sub-step right after the barrier, before the MFMAs of this step's last one
    // (whose fragments were read before the barrier, so the buffer is free to be
    // overwritten).  No MFMA waits for an LDS read issued just before it.
    constexpr int NK = GK / 16;
    static_assert(NK % 2 == 0, "the fragment sets alternate with a period of two sub-steps");
    half8_t fa[2][AT], fb[2][AF];
    const int swz = (l32 >> 2) & 3;             // wt, wf and the tile offsets are multiples of 32: only the lane's row counts
    auto load_frags = [&](auto setc, int buf, int kk) {
        constexpr int set = decltype(setc)::value;
        const half_t *xs = &lds[buf][0], *ws = &lds[buf][BT * LSTRIDE];
#pragma unroll
        for (int j = 0; j < AT; j++)
            fa[set][j] = *reinterpret_cast<const half8_t *>(xs + (wt + 32 * j + l32) * LSTRIDE + (SWZ ? 8 * ((2 * kk + kh) ^ swz) : 16 * kk + 8 * kh));
#pragma unroll
        for (int j = 0; j < AF; j++)
            fb[set][j] = *reinterpret_cast<const half8_t *>(ws + (wf + 32 * j + l32) * LSTRIDE + (SWZ ? 8 * ((2 * kk + kh) ^ swz) : 16 * kk + 8 * kh));
    };
    auto mfmas = [&](auto setc) {
        constexpr int set = decltype(setc)::value;
#pragma unroll
        for (int ai = 0; ai < AT; ai++)
#pragma unroll
            for (int bi = 0; bi < AF; bi++)
                acc[ai][bi] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[set][ai], fb[set][bi], acc[ai][bi], 0, 0, 0);
    };
    using S0 = std::integral_constant<int, 0>;
    using S1 = std::integral_constant<int, 1>;
    // step s reads LDS buffer s & 1; its pieces travelled through register set s & 1
    // Neither the requests for step s + 2 nor the LDS writes of step s + 1 (requested a
    // step ago) are issued in one burst - a wave that queues six or more 1 KB requests
    // blocks on the address unit and every wave of the workgroup does so at the same
    // time, right after the barrier, with the matrix pipe idle.  Both are cut into
    // portions, one per group of MFMAs, issued together with the fragment reads in front
    // of the group.  Nobody reads the other LDS buffer between the previous barrier and
    // the next one, so it can be written all along the step.
    using PF = std::integral_constant<int, NK>;
    using PS = std::integral_constant<int, NK - 1>;
    auto one_step = [&](auto cur, auto nxt, auto bufc, int step) {
        constexpr int buf = decltype(bufc)::value;
        static_for<NK / 2>([&](auto hc) {
            constexpr int kk = 2 * decltype(hc)::value;
            fetch(cur, step + NS, std::integral_constant<int, kk>{}, PF{});   // set `cur` was emptied into LDS a step ago
            load_frags(S1{}, buf, kk + 1);
            stash(nxt, buf ^ 1, std::integral_constant<int, kk>{}, PS{});    // after the last step: a copy nobody reads
            __builtin_amdgcn_sched_barrier(0);
            mfmas(S0{});
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (kk + 2 < NK) {
                fetch(cur, step + NS, std::integral_constant<int, kk + 1>{}, PF{});
                load_frags(S0{}, buf, kk + 2);
                stash(nxt, buf ^ 1, std::integral_constant<int, kk + 1>{}, PS{});
                __builtin_amdgcn_sched_barrier(0);
                mfmas(S1{});
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        __syncthreads();
        fetch(cur, step + NS, std::integral_constant<int, NK - 1>{}, PF{});
        load_frags(S0{}, buf ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        mfmas(S1{});
        __builtin_amdgcn_sched_barrier(0);
    };

    // step s: its pieces travel through register set s % NS and are multiplied out of LDS buffer s % 2; the loop is
    // written out over one period of both, so that every set and buffer index is a constant
    static_for<NS>([&](auto kc) { fetch(kc, decltype(kc)::value, S0{}, S1{}); });
    stash(S0{}, 0, S0{}, S1{});
    __syncthreads();
    load_frags(S0{}, 0, 0);
    constexpr int PERIOD = NS % 2 == 0 ? NS : 2 * NS;
    for (int step = 0; step < steps; step += PERIOD) {
        static_for<PERIOD>([&](auto kc) {
            constexpr int k = decltype(kc)::value;
            if (k == 0 || step + k < steps)
                one_step(std::integral_constant<int, k % NS>{}, std::integral_constant<int, (k + 1) % NS>{},
                         std::integral_constant<int, k % 2>{}, step + k);
        });
    }

    // D[token, feature]: lane holds feature l32, tokens 8 * (v / 4) + 4 * kh + v % 4
#pragma unroll
    for (int bi = 0; bi < AF; bi++) {
        const int m = m0 + wf + 32 * bi + l32;
        if (m >= M) continue;
        const float bv = bias ? (float)bias[m] : 0.f;
#pragma unroll
        for (int ai = 0; ai < AT; ai++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int t = t0 + wt + 32 * ai + 8 * (v >> 2) + 4 * kh + (v & 3);
                if (t < T) y[(int64_t)t * M + m] = (half_t)(acc[ai][bi][v] + bv);
            }
    }
}

// Few tokens (<= 32): the job is to stream w once at memory speed, so nothing is shared through LDS.  A workgroup owns 16 F features; its 8 waves split the contracted
// range, each reading its fragments of v_mfma_f32_16x16x32_f16 straight from global memory, whole 128-byte lines (the two halves of one back to back), AHEAD
// lines of 16 F rows in flight, TB blocks of 16 tokens against them.  The waves' sums are added through LDS in a fixed order.  N % 8 == 0: pieces beyond the last
// column, or the wave's last line, are asked for beyond the end of the buffer, which reads as zeros.  Every feature is summed in the same order, so equal rows of w
// (words that share an embedding) have equal outputs.  Workgroups that start at places of their own along the rows ask different memory channels and are faster where rows are 4, 8 or
// 16 KB (us, this / so: 32000 x 8192, 8 tokens 98.3 / 90.8; 32000 x 4096, one 52.8 / 48.7; 14336 x 4096, 8 27.0 / 24.1; 32000 x 5120, 8 62.0 / 61.7), but then the order depends on the
// workgroup; two or four parts whose sums commute, walked in orders of their own, are not (97 and 102 on the first).
// What bounds it: memory (32000 x 8192, one token: 5.6 TB/s), with 16 tokens and more the reads of x, as many bytes per workgroup as T / (16 F) of w.  us, the kernel
// before (v_mfma_f32_32x32x16_f16, half a line's quarter per request, N % 16 == 0 only, otherwise the tiled kernel) / this: 32000 x 4096, one token 55.7 / 48.7, 8 tokens
// 63.9 / 49.3, 32 tokens 89.1 / 56.8; 32000 x 8192, 8 tokens 123.9 / 92.5; 4096 x 4104, 8 tokens 26.0 / 8.1; 512 x 6008 27.5 / 8.1.  Fewer parts of the contracted range and more features side by
// side (4, 2, 1 parts): slower from 4096 columns on, level below.
constexpr int SKINNY_WAVES = 8, SKINNY_LINE = 64;               // columns of a line
template <int TB, int F, int AHEAD>
__global__ __launch_bounds__(64 * SKINNY_WAVES, 4) void linear_skinny_kernel(
    const half_t *__restrict__ x, const half_t *__restrict__ w, const half_t *__restrict__ bias,
    half_t *__restrict__ y, int T, int M, int N) {
    __shared__ float4_t red[SKINNY_WAVES][TB * F][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lm = lane & 15, g = lane >> 4;
    const int m0 = blockIdx.x * (16 * F);
    const int lines = (N + SKINNY_LINE - 1) / SKINNY_LINE, per = (lines + SKINNY_WAVES - 1) / SKINNY_WAVES;
    const int begin = wave * per, end = min(begin + per, lines), limit = min(end * SKINNY_LINE, N);     // (no branch around a product: its loads would move into it)
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)(w + (int64_t)m0 * N), 0, (int)((uint32_t)min(16 * F, M - m0) * (uint32_t)N * 2u), 0x00020000);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)x, 0, (int)((uint32_t)T * (uint32_t)N * 2u), 0x00020000);
    uint32_t off_w[F], off_x[TB];
#pragma unroll
    for (int f = 0; f < F; f++) off_w[f] = (uint32_t)(16 * f + lm) * (uint32_t)N * 2u + 16u * g;
#pragma unroll
    for (int b = 0; b < TB; b++) off_x[b] = (uint32_t)min(16 * b + lm, T - 1) * (uint32_t)N * 2u + 16u * g;

    float4_t acc[TB][F];
#pragma unroll
    for (int b = 0; b < TB; b++)
#pragma unroll
        for (int f = 0; f < F; f++) acc[b][f] = (float4_t){0.f, 0.f, 0.f, 0.f};
    for (int at = begin; at < end; at += AHEAD) {
        half8_t wf[AHEAD][2][F], xf[AHEAD][2][TB];
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
            const int col = (at + q) * SKINNY_LINE;
#pragma unroll
            for (int f = 0; f < F; f++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    wf[q][h][f] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rw, (int)(col + 32 * h + 8 * g < limit ? off_w[f] + 64u * h : 0x80000000u), 2 * col, 0));
#pragma unroll
            for (int b = 0; b < TB; b++)
#pragma unroll
                for (int h = 0; h < 2; h++)
                    xf[q][h][b] = __builtin_bit_cast(half8_t, __builtin_amdgcn_raw_buffer_load_b128(rx, (int)(col + 32 * h + 8 * g < limit ? off_x[b] + 64u * h : 0x80000000u), 2 * col, 0));
        }
        __builtin_amdgcn_sched_barrier(0);                               // (all of them on their way before the first is waited for)
#pragma unroll
        for (int q = 0; q < AHEAD; q++) {
#pragma unroll
            for (int h = 0; h < 2; h++)
#pragma unroll
                for (int b = 0; b < TB; b++)
#pragma unroll
                    for (int f = 0; f < F; f++) acc[b][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[q][h][b], wf[q][h][f], acc[b][f], 0, 0, 0);
        }
    }
#pragma unroll
    for (int b = 0; b < TB; b++)
#pragma unroll
        for (int f = 0; f < F; f++) red[wave][b * F + f][lane] = acc[b][f];
    __syncthreads();
    // D[token, feature]: lane 16 g + lm holds tokens 4 g .. 4 g + 3 of feature lm
    for (int o = tid; o < TB * F * 256; o += 64 * SKINNY_WAVES) {
        const int f = (o >> 4) % F, t = o / (16 * F), m = m0 + o % (16 * F);
        float sum = 0.f;
#pragma unroll
        for (int k = 0; k < SKINNY_WAVES; k++) sum += red[k][(t >> 4) * F + f][16 * ((t >> 2) & 3) + (o & 15)][t & 3];
        if (m < M && t < T) y[(int64_t)t * M + m] = (half_t)(sum + (bias ? (float)bias[m] : 0.f));
    }
}

// Shapes the tiled kernel does not take (N % 8 != 0 or unaligned buffers).
__global__ __launch_bounds__(256) void linear_generic_kernel(
    const half_t *__restrict__ x, const half_t *__restrict__ w, const half_t *__restrict__ bias,
    half_t *__restrict__ y, int T, int M, int N) {
    // one wave per output element, lanes stride over n
    const int lane = threadIdx.x & 63;
    int64_t o = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t total = (int64_t)T * M;
    const int64_t stride = ((int64_t)gridDim.x * blockDim.x) >> 6;
    for (; o < total; o += stride) {
        const int t = (int)(o / M), m = (int)(o % M);
        float acc = 0.f;
        for (int n = lane; n < N; n += 64)
            acc = __builtin_fmaf((float)x[(int64_t)t * N + n], (float)w[(int64_t)m * N + n], acc);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
        if (lane == 0) y[o] = (half_t)(acc + (bias ? (float)bias[m] : 0.f));
    }
}

// NS: register sets of pieces in flight.  WHOLE: also instantiate the kernel for a contracted range without a partial last
// k-step (false: the caller only comes with N % GK != 0).
template <int WT, int WF, int AT, int AF, int GK, int NS = 3, bool WHOLE = true>
int launch_tiled(const half_t *x, const half_t *w, const half_t *bias, half_t *y, int T, int M, int N,
                 hipStream_t s) {
    constexpr int BT = WT * AT * 32, BF = WF * AF * 32;
    constexpr size_t lds = (size_t)2 * (BT + BF) * lds_stride(GK) * sizeof(half_t);
    static bs_lds_grant granted[2][BS_MAX_DEVICES];
    const dim3 grid((unsigned)bs_cdiv(M, BF), (unsigned)bs_cdiv(T, BT));
    if (N % GK != 0) {
        const int st = bs_allow_lds((const void *)linear_f16_kernel<WT, WF, AT, AF, GK, true, NS>, lds, granted[1]);
        if (st != BS_OK) return st;
        linear_f16_kernel<WT, WF, AT, AF, GK, true, NS><<<grid, 64 * WT * WF, lds, s>>>(x, w, bias, y, T, M, N);
        return BS_OK;
    }
    if constexpr (WHOLE) {
        const int st = bs_allow_lds((const void *)linear_f16_kernel<WT, WF, AT, AF, GK, false, NS>, lds, granted[0]);
        if (st != BS_OK) return st;
        linear_f16_kernel<WT, WF, AT, AF, GK, false, NS><<<grid, 64 * WT * WF, lds, s>>>(x, w, bias, y, T, M, N);
        return BS_OK;
    }
    return BS_ERR_SHAPE;
}

}  // namespace

// Which kernel bs_linear_f16 runs for these dimensions: tokens x features per workgroup (0 x 0 for the
// one-wave-per-output kernel), and whether the contracted range ends in a partial k-step.
struct LinearTile { int bt, bf, gk; };
static LinearTile linear_tile(int T, int M, int N, bool aligned) {
    if (!(N % 8 == 0 && aligned) || N >= (1 << 23)) return {0, 0, 0};     // (a tile's rows stay within 32-bit byte offsets)
    // linear_skinny_kernel: the more features a workgroup has, the less x it reads, but what counts is the rounds of 256 workgroups, each of which takes about as long
    // half empty: 16 features while one round holds them, 64 where they take less than 4/7 of the rounds of 32.  us, 16 / 32 / 64 features, 4096 columns: 8 tokens, 4096 rows
    // 8.8 / 11.4 / 18.4, 4189 15.2 / 11.5 / 18.5, 8192 15.8 / 14.7 / 18.6, 8400 21.8 / 22.2 / 18.6, 17129 34.8 / 34.5 / 38.5, 24600 47.0 / 39.9 / 39.6, 33000 61.1 / 54.0 /
    // 57.3; 32 tokens, 4189 23.3 / 16.6 / 24.1, 8400 33.6 / 32.0 / 23.9.  Below 1024 columns 32 and 64 are closer (720, 8 tokens: 4189 rows 4.2 / 2.9 / 3.7, 12288
    // 5.6 / 3.8 / 3.9, 17129 8.4 / 5.1 / 5.8), and from 960 on 16 are kept to 5119 rows, where the kernel's tests have them.
    if (T <= 32 && N >= 1024) return {32, M <= 4096 ? 16 : 7 * bs_cdiv(M, 256 * 64) < 4 * bs_cdiv(M, 256 * 32) ? 64 : 32, 0};
    if (T <= 32) return {32, M >= 12288 ? 64 : M > (N < 960 ? 4096 : 5119) ? 32 : 16, 0};
    if (T <= 128) return M >= 8192 ? LinearTile{128, 64, 64} : LinearTile{128, 32, 128};
    // The largest tile whose grid still covers most of the 256 CUs: 256 x 256 and
    // 128 x 256 move the fewest bytes per flop; 128 x 128 and 64 x 64
    // keep a small problem spread over the chip.
    const auto wgs = [&](int bt, int bf) { return bs_cdiv(T, bt) * bs_cdiv(M, bf); };
    return wgs(256, 256) >= 160 ? LinearTile{256, 256, N % 64 == 0 ? 64 : 32} :
           wgs(128, 256) >= 160 ? LinearTile{128, 256, 64} :
           wgs(128, 128) >= 160 ? LinearTile{128, 128, 64} : LinearTile{64, 64, 128};
}

// Which kernel has the 64 x 64 tiles where N % 64 == 0.  While a CU has one workgroup linear_pipe_kernel (us, linear_f16_kernel / linear_pipe_kernel: 190 tokens on 5000 x 2048 15.1 / 12.0, 256
// on 4096 x 4096 23.6 / 21.2).  Beyond that linear_f16_kernel is ahead where the tiles of features are a multiple of 8: a tile's features are then on one XCD for all tokens, which reads them once
// (256 on 5120 x 3072 23.8 / 29.2, x 8192 54.5 / 63.8, 6656 x 4096 33.9 / 35.8, 320 on 5600 x 5120 43.0 / 48.1; up to 1280 columns it is behind, 140 on 6144 x 1024 10.0 / 8.3); elsewhere it is
// behind (200 on 7600 x 4096 42.8 / 32.3, 320 on 5152 x 1792 19.6 / 16.1), but for long rows of up to 384 workgroups, where neither is (160 on 5870 x 4096 29.3 / 32.3, 400 on 2447 32.6 / 25.6) and it stays.
// Of 130 drawn products of 257 to 620 workgroups 3 are 2 to 7 % slower so than on linear_f16_kernel throughout, 0.956 of its time on average; by workgroups and columns alone 20 were, up to 15 %.
static bool pipe_64(const LinearTile &tile, int T, int M, int N) {
    const int64_t rows = bs_cdiv(M, 64), wg = bs_cdiv(T, 64) * rows;
    return tile.bt == 64 && tile.bf == 64 && (wg <= 256 || N <= 1280 || (rows % 8 != 0 && (wg > 384 || N <= 3072)));
}

// whether linear_pipe_kernel has this tile of bs_linear_f16's
static bool on_pipe(const LinearTile &tile, int T, int M, int N) { return N % 64 == 0 && (tile.bf >= 128 || pipe_64(tile, T, M, N)); }

// The tile behind a rebuilt weight, where scratch for partial sums can be had too.  splits > 1: the contracted range is
// cut into that many parts, whose sums a second kernel adds up: a few tokens on a large weight are a handful of large
// tiles, which leave most of the chip idle, or many small ones, which move the most bytes per flop (509 tokens on
// 4096 x 14336: 114 us with 64 x 64 tiles, 68 with 32 tiles of 256 x 256 in 8 parts each).
struct LinearChoice { int bt, bf, splits; };      // bt == 0: as bs_linear_f16

// The tiles of gemm_pipe.hip, and in us what a k-step of 64 columns and the start and end of a workgroup take: while a CU has one workgroup, and (step_two > 0) a pair of
// workgroups that share one.  A fit to the times of every tile on 256 products, 40 to 3300 tokens on 14 matrices from 600 x 512 to 28672 x 8192: the choice
// made with it is 1.0 % from the best tile on average, 25 at worst.  Four entries were further off and are set by whole calls, 22 to 50 drawn ones each, on the tile and on the one that the new
// estimate takes: 256 x 192 (1.336: 1.025 of the other's time on average, 2254 tokens on 4592 x 2176 59.1 us, on 192 x 256 55.7), two workgroups per CU of 160 x 128 (1.189: 1.046, 3120 on 3188 x 24576
// 510 / 450), of 64 x 64 (0.440: 1.17, 1994 on 545 x 9088 62.2 / 52.6) and, on rows of more than 8192 columns, of 64 x 128 (1.10, 313 on 11067 x 17664 356 / 302; shorter rows are as estimated).
// What the sums cost: whole calls cut and not, 98 of 132 to 1400 tokens on 12 matrices, and 132 drawn ones of 129 to 4100 on
// weights of 64 to 380 MiB: beyond 64 MiB of sums 0.5 us more per MiB than up to there (2515 tokens on 9480 x 12800, 182 MiB, 597 us in two parts, 540 in one; 2735 on 7320 x 25216, 305 MiB,
// 1001 in four, 1011).  Where the estimates are level the cut is 3 to 20 % behind (6936 x 22272, 1722 tokens 585 / 493, 8824 x 17408, 1362 480 / 427), and the calls that it is ahead on (4096 x
// 14336, 1400 tokens 186 / 211, 509 123 / 149) are clear of that line.
struct PipeTile { int bt, bf; double step, start, step_two, start_two; };
static const PipeTile pipe_tiles[] = {
    {256, 256, 1.604, 4.1, 0, 0}, {224, 256, 1.471, 3.5, 0, 0}, {192, 256, 1.358, 2.6, 0, 0}, {256, 192, 1.385, 2.9, 0, 0},
    {160, 256, 1.143, 3.1, 0, 0}, {192, 192, 0.966, 3.1, 0, 0}, {256, 128, 0.970, 2.6, 0, 0}, {128, 256, 0.930, 2.3, 0, 0},
    {224, 128, 0.862, 2.2, 0, 0}, {192, 128, 0.758, 1.9, 0, 0}, {128, 192, 0.777, 2.1, 0, 0}, {160, 128, 0.760, 1.3, 1.330, 4.8},
    {128, 128, 0.620, 1.2, 1.034, 3.0}, {96, 128, 0.540, 1.1, 0.922, 1.6}, {64, 128, 0.433, 0.8, 0.688, 1.8}, {64, 64, 0.250, 1.1, 0.484, 0.9}};

// Time in us that a tile is expected to take: rounds of workgroups over the chip, the last one shorter while part of it is idle (power, and memory to itself), plus the sums.
static double linear_cost(const PipeTile &t, int splits, int T, int M, int N) {
    const int64_t all = bs_cdiv(N, 64), steps = bs_cdiv(all, splits), parts = bs_cdiv(all, steps);
    const int64_t wg = bs_cdiv(T, t.bt) * bs_cdiv(M, t.bf) * parts;
    const bool two = t.step_two > 0 && wg > 256;
    const int64_t slots = two ? 512 : 256, rounds = bs_cdiv(wg, slots);
    const double step = !two ? t.step : N > 8192 && t.bt == 64 && t.bf == 128 ? 1.1 * t.step_two : t.step_two;
    double us = (rounds - 0.43 * (rounds - (double)wg / slots)) * steps * step + rounds * (two ? t.start_two : t.start) + 2.0;
    // (sums beyond 64 MiB no longer stay in the cache between the two kernels)
    const double sums = (double)parts * T * M, cached = 1 << 24;
    if (parts > 1) us += 3.0 + 0.5e-6 * sums + (sums > cached ? 2e-6 * (sums - cached) : 0.);
    return us;
}

static LinearChoice linear_choice(int T, int M, int N) {
    if (N % 64 != 0 || N >= (1 << 23)) return {0, 0, 1};
    // Partial sums only behind a weight that is beyond the static scratch by itself (a call that fits the static scratch
    // is never refused, or run differently, for their sake; smaller weights gain little), never more of them than weight,
    // and where a row of y can be written 16 bytes at a time.
    const int64_t weight = (int64_t)M * N * 2;
    const bool may_split = weight > (int64_t)BS_STATIC_SCRATCH_BYTES && M % 8 == 0;
    if (T <= 32 && !may_split) return {0, 0, 1};
    static const int cuts[] = {2, 3, 4, 6, 8, 12};
    LinearChoice one = {0, 0, 1}, cut = {0, 0, 1};
    double one_us = 1e30, cut_us = 1e30;
    for (const PipeTile &t : pipe_tiles) {
        if (T > 32) {
            const double us = linear_cost(t, 1, T, M, N);
            if (us < one_us) one_us = us, one = {t.bt, t.bf, 1};
        }
        if (!may_split || t.bf == 64) continue;
        for (int c : cuts) {
            if ((int64_t)c * T * M * 4 > weight) break;
            const double us = linear_cost(t, c, T, M, N);
            if (us < cut_us) cut_us = us, cut = {t.bt, t.bf, c};
        }
    }
    return cut_us < one_us ? cut : one;
}
// (asked for the scratch, then for the launch: the last answer of the thread is kept)
static LinearChoice linear_choice_kept(int T, int M, int N) {
    static thread_local int kT = 0, kM = 0, kN = 0;
    static thread_local LinearChoice kept = {0, 0, 1};
    if (T != kT || M != kM || N != kN) kept = linear_choice(T, M, N), kT = T, kM = M, kN = N;
    return kept;
}

int64_t bs_linear_parts_bytes(int T, int M, int N) {
    const LinearChoice c = linear_choice_kept(T, M, N);
    return c.splits > 1 ? (int64_t)c.splits * T * M * 4 : 0;
}

int bs_launch_linear_parts(const half_t *x, const half_t *w, const half_t *bias, half_t *y, int T, int M, int N, float *part, hipStream_t s) {
    const LinearChoice c = linear_choice_kept(T, M, N);
    if (c.bt == 0) return bs_launch_linear_f16(x, w, bias, y, T, M, N, s);
    return bs_launch_linear_pipe(x, w, bias, y, T, M, N, c.bt, c.bf, c.splits, part, s);
}

int bs_launch_linear_f16(const half_t *x, const half_t *w, const half_t *bias, half_t *y,
                         int T, int M, int N, hipStream_t s) {
    const LinearTile tile = linear_tile(T, M, N, bs_aligned(x, 16) && bs_aligned(w, 16));
    int st = BS_OK;
    if (tile.bt == 0) {
        int64_t blocks = bs_cdiv((int64_t)T * M, 4);
        if (blocks > 256 * 64) blocks = 256 * 64;
        linear_generic_kernel<<<(int)blocks, 256, 0, s>>>(x, w, bias, y, T, M, N);
    } else if (tile.gk == 0) {
        const auto skinny = [&](auto kernel) { kernel<<<(int)bs_cdiv(M, tile.bf), 64 * SKINNY_WAVES, 0, s>>>(x, w, bias, y, T, M, N); };
        if (T <= 16) tile.bf == 64 ? skinny(linear_skinny_kernel<1, 4, 2>) : tile.bf == 32 ? skinny(linear_skinny_kernel<1, 2, 2>) : skinny(linear_skinny_kernel<1, 1, 6>);
        else tile.bf == 64 ? skinny(linear_skinny_kernel<2, 4, 1>) : tile.bf == 32 ? skinny(linear_skinny_kernel<2, 2, 2>) : skinny(linear_skinny_kernel<2, 1, 4>);
    } else if (on_pipe(tile, T, M, N)) {
        return bs_launch_linear_pipe(x, w, bias, y, T, M, N, tile.bt, tile.bf, 1, nullptr, s);
    } else if (tile.bt == 128 && tile.bf == 64) {
        st = launch_tiled<2, 2, 2, 1, 64>(x, w, bias, y, T, M, N, s);
    } else if (tile.bt == 128 && tile.bf == 32) {
        st = launch_tiled<4, 1, 1, 1, 128>(x, w, bias, y, T, M, N, s);
    } else if (tile.bt == 256) {
        st = launch_tiled<2, 4, 4, 2, 32>(x, w, bias, y, T, M, N, s);
    } else if (tile.bf == 256) {
        st = launch_tiled<2, 4, 2, 2, 64, 4, false>(x, w, bias, y, T, M, N, s);
    } else if (tile.bf == 128) {
        st = launch_tiled<2, 2, 2, 2, 64, 4, false>(x, w, bias, y, T, M, N, s);
    } else {
        st = launch_tiled<2, 2, 1, 1, 128, 4>(x, w, bias, y, T, M, N, s);
    }
    if (st != BS_OK) return st;
    BS_LAUNCH_CHECK();
    return BS_OK;
}

extern "C" int bs_linear_plan(int T, int M, int N, int *tile_tokens, int *tile_features, int *k_step, int *k_tail) {
    if (!tile_tokens || !tile_features || !k_step || !k_tail) return BS_ERR_NULL;
    if (T <= 0 || M <= 0 || N <= 0) return BS_ERR_SHAPE;
    LinearTile t = linear_tile(T, M, N, true);
    if (on_pipe(t, T, M, N)) t.gk = 64;                     // linear_pipe_kernel's
    *tile_tokens = t.bt;
    *tile_features = t.bf;
    *k_step = t.gk;
    *k_tail = t.gk > 0 && N % t.gk != 0;
    return BS_OK;
}

extern "C" int bs_dense_plan(int T, int M, int N, int rebuilt, int *tile_tokens, int *tile_features, int *parts, int *stages) {
    if (!tile_tokens || !tile_features || !parts || !stages) return BS_ERR_NULL;
    if (T <= 0 || M <= 0 || N <= 0) return BS_ERR_SHAPE;
    const LinearTile t = linear_tile(T, M, N, true);
    LinearChoice c = rebuilt ? linear_choice(T, M, N) : LinearChoice{0, 0, 1};
    const bool pipe = c.bt != 0 || on_pipe(t, T, M, N);
    if (c.bt == 0) c = {t.bt, t.bf, 1};
    *tile_tokens = c.bt;
    *tile_features = c.bf;
    *parts = 1;
    *stages = 0;
    return pipe ? bs_linear_pipe_plan(T, M, N, c.bt, c.bf, c.splits, parts, stages) : (int)BS_OK;
}

extern "C" int bs_linear_f16(const void *x, const void *w, const void *bias, void *y,
                             int T, int M, int N, void *stream) {
    if (T < 0 || M <= 0 || N <= 0) return BS_ERR_SHAPE;
    if (T == 0) return BS_OK;
    if (!x || !w || !y) return BS_ERR_NULL;
    if (!bs_aligned(x, 2) || !bs_aligned(w, 2) || !bs_aligned(y, 2) || !bs_aligned(bias, 2))
        return BS_ERR_ALIGN;
    return bs_launch_linear_f16((const half_t *)x, (const half_t *)w, (const half_t *)bias,
                                (half_t *)y, T, M, N, (hipStream_t)stream);
}
