// Forward for one to 48 tokens on gfx950, rank 16 (and 4 to 15: tile_ranks.hip, tile_few_ranks.hip): the weight is rebuilt in registers, 32 x 32 outputs per matrix instruction,
// and multiplied by x at once; it never goes to memory.
//
//   part[cg, t, m] = sum_{n in column group cg} x[t, n] * fp16( sum_i s_i[m, n] * sum_r u_i[m, r] * vt_i[r, n] )
//
// A workgroup is 8 waves side by side: wave w owns 32 NP columns (NP = 4: 1024 columns per workgroup, 2: 512, 1: 256) and keeps what
// belongs to them in registers - the vt fragments of ALL blocks and the x fragments - while tiles of 32 rows pass by.  Per tile the
// sign rows (whole 128 or 64-byte runs of a line, each loaded once) and u rows of all blocks are fetched by all waves together into a ring in LDS.
// Per block a wave runs NP v_mfma_f32_32x32x16_f16, D[column, row]: rank 16 is exactly their depth, so an output costs half the
// matrix time of a 16x16x16 product, and a lane gets 16 consecutive columns of one row.  The sum over the blocks is kept divided by
// the current block's sign: between two blocks it changes sign where they differ, which is one v_xor_b32 per output with a mask from a
// table in LDS (four masks per nibble of the two sign words' difference), and the matrix instruction adds the next block's product.
// Behind the last block the lane's columns, rounded to fp16 as a stored weight is, become B operands of y[token, row] += x . w
// (v_mfma_f32_16x16x32_f16).  The waves' y tiles (same rows, other columns) meet in LDS, double buffered, and are added up in wave
// order while the next tile is rebuilt: one barrier per tile, and scratch holds one partial per 256 NP columns.
//
// The rebuilt weight itself (TT = 0, in forwards above 128 tokens) is the same walk with the rounded tile stored instead of multiplied.  Whole calls of
// 130 tokens, us, reconstruct_tile_kernel / this: 14336 x 4096, 8 blocks 104 / 90, 4096 x 14336, 8 109 / 92 (the rebuild by itself, by the profiler, 82 / 63),
// 28672 x 8192, 3 310 / 241, 14336 x 4096, 5 89 / 84.
//
// What bounds it: the issue of a wave's instructions: by the counters vector instructions take 64 % of a SIMD's cycles on 28672 x 8192, 3 blocks, 8 tokens
// and 60 on 4096 x 14336, 4 blocks, 4 tokens (the matrix cores 22 and 15), where runs are short 33 (5000 x 4096, 6 blocks, 37 tokens) and waits at the
// barrier and for LDS as much, in the rebuild 51 with its stores waited for.  Simple VALU instructions (v_xor_b32, v_and_b32, v_lshrrev_b32, fp32 add, mul and FMA on
// three registers) of two waves run side by side on a SIMD, 1.0 ns each; v_fma_mix_f32, v_and_or_b32, v_bfe, v_alignbit, conversions and whatever
// has a scalar operand take 1.8 ns, and a single wave issues one instruction in 2 ns whatever it is.  A step (1024 signs: 16 v_xor, 5 for the
// table addresses, 4 lookups, one product) takes 45 ns per SIMD with two waves and 40 with four; with the signs as fp16 in v_fma_mix 46 and 42.
// About 1300 cycles per tile and wave (barrier, hand-over, rounding, second product) come on top.  The loop over the tiles has no branch around a request or a
// store: stores that have nothing to write go to an offset or a buffer that drops them, waves without columns do their work for nobody.  Where the compiler could
// not tell how many were in flight, every tile waited for the requests made right before it and for its own stores (us with such branches / without: rebuild of
// 4096 x 14336, 8 blocks 65.2 / 59.4, 14336 x 4096, 5 45.9 / 42.3; 10 blocks of 4096 x 4096, 8 tokens 23.9 / 22.5; a step of 8 sequences over two 70B-shape layers 662 / 642).  us, strip_forward_kernel / this, with the summing launch, in a
// replayed graph on rotating copies: 28672 x 8192, 3 blocks, 8 tokens 86.5 / 62.8; 14336 x 4096, 8 blocks, 8 tokens 50.0 / 42.6; 5000 x 4096, 6 blocks, 37 tokens
// 29.7 / 25.6.  (One and two tokens of larger matrices whose columns are no multiple of 512 are the sparse kernel's, see sparse_plan in gemv.hip.)
#include "common.h"
#include "rebuild_shared.h"

#include <type_traits>
#include <utility>

constexpr int TL_WAVES = 8, TL_ROWS = 32, TL_GROUP = 4, TL_MIN_RANK = 4;
struct TileMat {
    const uint8_t *packed;
    const half_t *u, *vt;
    float *part;
    half_t *w;                                      // (the rebuild: where the weight goes; part is null)
    int I, M, np, row_tiles, first_wg, wgs;         // workgroups first_wg + wgs * column group .. + wgs - 1
};
struct TileGroup {
    TileMat m[TL_GROUP];
    int n;
    float *ssq;                                     // [column groups of matrix 0][T]: sums of x^2 over the group's columns, or null
};

// The kernels for ranks 4 to 15 are the same code with a rank that is not known at compile time, in translation units of their own that include this file: tile_ranks.hip (8 to 15) and
// tile_few_ranks.hip (4 to 7).  With one kernel for all ranks rank 16 was up to 1.5 % slower (a step of eight sequences over two 70B-shape layers 620 / 628).
#ifdef TILE_RANKS
constexpr int TL_RANKS = TILE_RANKS;                // the least rank of this build
#else
constexpr int TL_RANKS = 16;
#endif
// tt: token tiles of 16, 0 for the rebuild
int bs_launch_tile_ranks(const TileGroup &grp, int grid, const half_t *x, int N, int T, int K, int tt, hipStream_t s);
int bs_launch_tile_few_ranks(const TileGroup &grp, int grid, const half_t *x, int N, int T, int K, int tt, hipStream_t s);

namespace {

constexpr int TL_TABLE = 512, TL_HALVES = 256;      // bytes: the tables of sign masks at the start of LDS, where the one for pairs of halves begins
constexpr int TL_LDS = 160 * 1024;

__device__ __forceinline__ void tl_barrier() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
// a buffer of so many bytes: what lies beyond is not written
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tl_buffer(const void *p, int bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, __builtin_amdgcn_readfirstlane(bytes), 0x00020000);
}
// wait until at most n of this wave's LDS accesses, which run in order, are to come
template <int n>
__device__ __forceinline__ void tl_wait_lds() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(15 | (3 << 14) | (7 << 4) | (n << 8));
}
template <class F, int... Is>
__device__ __forceinline__ void tl_for_impl(F &&f, std::integer_sequence<int, Is...>) {
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void tl_for(F &&f) {
    tl_for_impl(f, std::make_integer_sequence<int, N>{});
}

// A row of u has fewer than 16 ranks: its pieces are read so that they lie within it, what this leaves ahead of a piece's first rank goes, and zeros take the places of the
// ranks that do not exist.  8 to 15: the second piece of 16 bytes is the row's last 16.  4 to 7: a piece is two of 8 bytes, the row's first and its last; the second piece is nothing.
__device__ __forceinline__ uint4_t tl_ranks(const uint4_t &p, bool second, int K) {
    uint64_t lo = p[0] | (uint64_t)p[1] << 32, hi = p[2] | (uint64_t)p[3] << 32;
    if constexpr (TL_RANKS == 8) {
        int s = 16 * (16 - K);                      // bits: 16 to 128
        if (s >= 64) {
            lo = hi;
            hi = 0;
            s -= 64;
        }
        if (s > 0) {
            lo = s < 64 ? lo >> s | hi << (64 - s) : 0;
            hi = s < 64 ? hi >> s : 0;
        }
        const uint4_t q = {(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
        return second ? q : p;
    } else {
        hi = K == 4 ? 0 : hi >> (16 * (8 - K));
        const uint4_t q = {(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
        return second ? (uint4_t){0, 0, 0, 0} : q;
    }
}
// 16 bytes of a chunk; ranks 4 to 7: two of 8, the second one `apart` behind the first
__device__ __forceinline__ uint4_t tl_load(__amdgpu_buffer_rsrc_t r, int at, int apart) {
    if constexpr (TL_RANKS >= 8) return __builtin_amdgcn_raw_buffer_load_b128(r, at, 0, 0);
    else {
        const uint2_t a = __builtin_amdgcn_raw_buffer_load_b64(r, at, 0, 0), b = __builtin_amdgcn_raw_buffer_load_b64(r, at + apart, 0, 0);
        return (uint4_t){a[0], a[1], b[0], b[1]};
    }
}

typedef const __attribute__((address_space(3))) char *lds_bytes;
typedef __attribute__((address_space(3))) char *lds_bytes_rw;
typedef const __attribute__((address_space(3))) half8_t *lds_half8;
typedef __attribute__((address_space(3))) half8_t *lds_half8_rw;
typedef const __attribute__((address_space(3))) uint4_t *lds_uint4;
typedef __attribute__((address_space(3))) uint4_t *lds_uint4_rw;
typedef const __attribute__((address_space(3))) uint2_t *lds_uint2;
typedef const __attribute__((address_space(3))) uint32_t *lds_u32;
typedef const __attribute__((address_space(3))) uint16_t *lds_u16;
typedef const __attribute__((address_space(3))) float *lds_f32;
typedef __attribute__((address_space(3))) float *lds_f32_rw;
typedef __attribute__((address_space(3))) float4_t *lds_f32x4_rw;

// TT: token tiles of 16; 0: the weight itself is what is wanted, it goes to memory.
// SPLIT (few tokens): the weight is not rounded to fp16 but enters the second product as two fp16 terms.
template <int TT, int NP, bool SPLIT = false>
struct TileKernel {
    static constexpr int WC = 32 * NP, CG = WC * TL_WAVES;     // columns per wave, per workgroup
    static constexpr int SROW = CG / 8;                        // sign bytes of a row in a stage
    static constexpr int RP = SROW / 16;                       // ... in 16-byte pieces
    static constexpr int SCH = SROW * TL_ROWS / 1024;          // requests of 1 KB per block: signs; u is one more
    // what a row's pieces are XOR-ed with in a stage, so that the 32 rows a read takes fall on different banks
    static __device__ __forceinline__ int swizzle(int r) { return (r * RP / 16) % RP; }
    // LDS: the table of sign masks (at address 0: the kernel has no other LDS), an area for two y tiles of every wave or its tile of the
    // weight (and at first for the vt images), and the ring of stages
    static constexpr int AREA = TT ? 32 * 1024 * TT : TL_WAVES * TL_ROWS * WC * 2;
    static constexpr int stage_bytes(int I) { return I * (SCH + 1) * 1024; }
    static constexpr size_t lds_size(int I) { return TL_TABLE + AREA + STAGES * (size_t)stage_bytes(I); }
    static constexpr int STAGES = 3;                           // the tile in work, the next one, one that is being written
    // most blocks: LDS, and the registers of the vt fragments
    static constexpr int max_blocks() {
        int I = NP == 4 ? (TT <= 1 ? 4 : TT == 2 ? 2 : 1) : NP == 2 ? (TT <= 1 ? 10 : 8) : 16;
        while (lds_size(I) > TL_LDS) I--;
        return I;
    }

    // A lane's piece within chunk c of a tile: chunks of 1 KB, the signs of block c / SCH first, then the u rows of the blocks
    static __device__ __forceinline__ uint32_t piece_at(int c, int I, int lane, int cg, uint32_t row_bytes, int K) {
        if (c < I * SCH) {
            const int r = (c % SCH) * (64 / RP) + lane / RP, piece = (lane % RP) ^ swizzle(r);
            return (uint32_t)r * row_bytes + min((uint32_t)(cg * SROW + piece * 16), row_bytes - 16u);
        }
        return (uint32_t)(lane >> 1) * (2u * K) + (TL_RANKS >= 8 && second_half(lane) ? 2u * K - 16u : 0u);
    }
    // whether the lane's piece of a u chunk is ranks 8 to 15
    static __device__ __forceinline__ bool second_half(int lane) { return ((lane ^ (lane >> 5)) & 1) != 0; }
    // y tiles: [buffer][wave][TT token tiles][rows 0-15, 16-31][four tokens: 4][row: 16][token: 4]; floats, of wave 0
    static constexpr int Y = 16 * TT * TL_ROWS;
    static __device__ __forceinline__ int y_at(int buf, int tt, int t, int row) { return buf * (TL_WAVES * Y) + tt * 512 + row / 16 * 256 + t / 4 * 64 + row % 16 * 4 + t % 4; }

    // The waves without columns, those from `active` on: their share of walk's requests and sums, between the same barriers.  (A path of their own, one for all block
    // counts: a branch in walk's loop leaves the compiler unsure of what is in flight, and doing the others' work on the last columns, for nobody, they took its issue
    // slots from them.  us, so / this: 13888 x 128 (half of the waves have no columns), 10 blocks, 3 tokens 11.2 / 9.6; 251 x 128, 5, 44 8.7 / 8.0; 4921 x 384, 3, 38 10.0 / 9.4.)
    static __device__ __forceinline__ void walk_without_columns(const uint8_t *__restrict__ packed, const half_t *__restrict__ u, float *__restrict__ part, int I, int M, lds_bytes_rw lds,
                                                                int N, int T, int ranks, int cg, int rt0, int len, bool ssq, int wave, int active) {
        const int K = TL_RANKS == 16 ? 16 : ranks;
        constexpr int MOST = 4;                                  // (32 chunks at most: 16 blocks of one patch)
        const int tid = threadIdx.x, lane = tid & 63, chunks = I * (SCH + 1), stage_size = stage_bytes(I), my_t = tid >> 5, my_row = tid & 31;
        const uint32_t row_bytes = (uint32_t)N >> 3;
        lds_bytes_rw area = lds + TL_TABLE, ring = area + AREA;
        uint4_t ahead[2][MOST];
        auto request = [&](int k, int n) {                       // tile n, or the last one
            const int rt = rt0 + min(n, len - 1);
            const uint32_t rows = min(M - rt * TL_ROWS, TL_ROWS);
#pragma unroll
            for (int q = 0; q < MOST; q++) {
                const int c = wave + TL_WAVES * q;
                if (c >= chunks) break;
                const bool signs = c < I * SCH;
                const char *from = signs ? reinterpret_cast<const char *>(packed) + (int64_t)(c / SCH) * M * row_bytes : reinterpret_cast<const char *>(u) + (int64_t)(c - I * SCH) * M * (2 * K);
                const uint32_t pitch = signs ? row_bytes : 2u * K;
                ahead[k][q] = tl_load(tl_buffer(from + (int64_t)(rt * TL_ROWS) * pitch, (int)(rows * pitch)), (int)piece_at(c, I, lane, cg, row_bytes, K), signs ? 8 : 2 * K - 8);
            }
        };
        auto write = [&](int k, int stage) {
#pragma unroll
            for (int q = 0; q < MOST; q++) {
                if (TL_RANKS < 16 && wave + TL_WAVES * q >= I * SCH) ahead[k][q] = tl_ranks(ahead[k][q], second_half(lane), K);
                if (wave + TL_WAVES * q < chunks) ((lds_uint4_rw)(ring + stage * stage_size + (wave + TL_WAVES * q) * 1024))[lane] = ahead[k][q];
            }
        };
        auto sums = [&](int n) {                                 // tile n, in walk's order
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                if (16 * tt + my_t >= T || (rt0 + n) * TL_ROWS + my_row >= M) continue;
                lds_f32 red = (lds_f32)(area) + y_at(n & 1, tt, my_t, my_row);
                float sum = red[0];
                for (int w = 1; w < active; w++) sum += red[w * Y];
                part[((int64_t)cg * T + 16 * tt + my_t) * M + (rt0 + n) * TL_ROWS + my_row] = sum;
            }
        };
        request(0, 0);
        request(1, 1);
        write(0, 0);
        write(1, 1);
        request(0, 2);
        if (ssq) {
            __syncthreads();
            __syncthreads();
        }
        tl_wait_lds<0>();
        tl_barrier();                                            // the first tile is here
        for (int n = 0; n < len; n++) {
            tl_wait_lds<0>();
            tl_barrier();                                        // tile n + 1 and the y tiles of n - 2 are in LDS, the stage of n - 1 is free
            write(0, (n + 2) % STAGES);
            request(0, n + 3);
            if (n >= 2) sums(n - 2);
        }
        tl_wait_lds<0>();
        if (len > 2) tl_barrier();
        tl_barrier();
        for (int n = max(len - 2, 0); n < len; n++) sums(n);
    }

    // One run of row tiles [rt0, rt0 + len) of column group cg of one matrix.
    template <int I>
    static __device__ __forceinline__ void walk(const uint8_t *__restrict__ packed, const half_t *__restrict__ u, const half_t *__restrict__ vt,
                                                float *__restrict__ part, half_t *__restrict__ w, int M, lds_bytes_rw lds, const half_t *__restrict__ x,
                                                int N, int T, int ranks, int cg, int rt0, int len, float *ssq) {
        const int K = TL_RANKS == 16 ? 16 : ranks;
        constexpr int STAGE = stage_bytes(I);
        constexpr int CHUNKS = I * (SCH + 1), PER = CHUNKS / TL_WAVES, MORE = CHUNKS % TL_WAVES, MOST = PER + (MORE != 0);
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));                           // (what follows from it is not shared between the block counts: registers)
        const int lane = tid & 63;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
        const int row = lane & 31, h = lane >> 5;               // in the rebuild
        const int lm = lane & 15, g = lane >> 4;                // in the second product
        const uint32_t row_bytes = (uint32_t)N >> 3;
        lds_bytes_rw area = lds + TL_TABLE, ring = area + AREA;
        // Waves whose columns exist (all or none of a wave's).  The others are in walk_without_columns, or (TT = 0, where all of them wait for the stores) do the
        // same work on the last columns, for nobody.
        const int active = min(TL_WAVES, (N - cg * CG) / WC);
        const int n0 = min(cg * CG + wave * WC, N - WC);

        // ---- requests ----------------------------------------------------------------------------------------------------
        // Wave w takes chunks w, w + 8, ...; one that is short of a chunk takes the last one too.
        const char *from[MOST];                                  // row 0 of the next tile to be requested
        uint32_t pitch[MOST], offset[MOST];                      // the lane's piece within a tile
        auto chunk_of = [&](int k) { return MORE == 0 || k < PER ? wave + TL_WAVES * k : min(wave + TL_WAVES * k, CHUNKS - 1); };
#pragma unroll
        for (int k = 0; k < MOST; k++) {
            const int c = chunk_of(k);
            const bool signs = c < I * SCH;
            from[k] = signs ? reinterpret_cast<const char *>(packed) + (int64_t)(c / SCH) * M * row_bytes : reinterpret_cast<const char *>(u) + (int64_t)(c - I * SCH) * M * (2 * K);
            pitch[k] = signs ? row_bytes : 2u * K;
            from[k] += (int64_t)(rt0 * TL_ROWS) * pitch[k];
            offset[k] = piece_at(c, I, lane, cg, row_bytes, K);
        }
        // A tile's pieces travel through registers: requested three tiles ahead, written to LDS at the end of the tile two ahead of it.
        int asked = rt0;                                         // the row tile `from` stands at
        const int last_rt = rt0 + len - 1;
        uint4_t pieces[MOST], pieces_1[MOST];                    // (pieces_1: only of the run's second tile)
        // (Behind the last tile that one is requested again.  A tile is a buffer that ends with the matrix's last row; rows beyond it read as zeros.)
        auto request_next = [&](uint4_t (&to)[MOST]) {
            const uint32_t rows = min(M - asked * TL_ROWS, TL_ROWS);
#pragma unroll
            for (int k = 0; k < MOST; k++) {
                to[k] = tl_load(tl_buffer(from[k], (int)(rows * pitch[k])), (int)offset[k], chunk_of(k) < I * SCH ? 8 : 2 * K - 8);
                __builtin_amdgcn_sched_barrier(0);               // (in the same order wherever they are issued: the waits count on it)
            }
            if (asked < last_rt) {
                asked++;
#pragma unroll
                for (int k = 0; k < MOST; k++) from[k] += pitch[k] * (uint32_t)TL_ROWS;
            }
        };
        auto write_tile = [&](int stage, uint4_t (&p)[MOST]) {
            if constexpr (TL_RANKS < 16) {
#pragma unroll
                for (int k = 0; k < MOST; k++)
                    if (chunk_of(k) >= I * SCH) p[k] = tl_ranks(p[k], second_half(lane), K);
            }
#pragma unroll
            for (int k = 0; k < MOST; k++) ((lds_uint4_rw)(ring + stage * STAGE + chunk_of(k) * 1024))[lane] = p[k];
        };
#pragma unroll
        for (int k = 0; k < MOST; k++) pieces[k] = pieces_1[k] = (uint4_t){0, 0, 0, 0};
        request_next(pieces);
        if constexpr (NP < 4) request_next(pieces_1);

        // ---- this wave's vt and x fragments -----------------------------------------------------------------------
        // vt: a lane takes 8 columns x 8 ranks of one block, turns them in registers and leaves them as [column][rank] in the wave's own
        // part of the area; the fragments are read back from there.  (The columns of a group of eight are XOR-ed with the group's
        // number: the groups lie a whole turn of the banks apart.)
        half8_t vf[I][NP];
        constexpr int TX = TT ? TT : 1;
        half8_t xf[TX][NP];
        {
            constexpr int PIECES = WC / 8, BP = 32 / PIECES, PASSES = (I + BP - 1) / BP, IMAGE = WC * 32;   // BP blocks per pass of loads
            constexpr int ROOM = (AREA / TL_WAVES < 8192 ? AREA / TL_WAVES : 8192), SB = ROOM / IMAGE;      // SB of them fit the image
            lds_bytes_rw img = area + wave * ROOM;
            const int piece = lane % PIECES, kh = (lane / PIECES) & 1, bl = lane / (2 * PIECES);
            const int col = 16 * NP * ((row >> 2) & 1) + 4 * (row >> 3) + (row & 3);
            half8_t v[PASSES][8];
#pragma unroll
            for (int pass = 0; pass < PASSES; pass++) {
                const half_t *src = vt + (int64_t)min(pass * BP + bl, I - 1) * K * N + n0 + 8 * piece;
#pragma unroll
                for (int r = 0; r < 8; r++) v[pass][r] = *reinterpret_cast<const half8_t *>(src + (int64_t)min(8 * kh + r, K - 1) * N);
            }
            if constexpr (TL_RANKS < 16) {           // (ranks that do not exist)
#pragma unroll
                for (int pass = 0; pass < PASSES; pass++)
#pragma unroll
                    for (int r = 0; r < 8; r++)
                        if (8 * kh + r >= K) v[pass][r] = (half8_t){0, 0, 0, 0, 0, 0, 0, 0};
            }
            // x: the columns whose weights lane group g holds when the rows are sorted out for the second product (see there)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                const half_t *xr = x + (int64_t)min(tt * 16 + lm, T - 1) * N + n0 + 16 * NP * (g >> 1) + 8 * (g & 1);   // (rows beyond T: outputs nobody stores)
#pragma unroll
                for (int p = 0; p < NP; p++) xf[tt][p] = *reinterpret_cast<const half8_t *>(xr + 16 * p);
            }
#pragma unroll
            for (int pass = 0; pass < PASSES; pass++)
#pragma unroll
                for (int sub = 0; sub < BP / SB; sub++) {
                    if (BP == SB || bl / SB == sub) {
#pragma unroll
                        for (int e = 0; e < 8; e++) {
                            half8_t o;
#pragma unroll
                            for (int r = 0; r < 8; r++) o[r] = v[pass][r][e];
                            *(lds_half8_rw)(img + (bl % SB) * IMAGE + (8 * piece + (e ^ (piece & 7))) * 32 + 16 * kh) = o;
                        }
                    }
                    asm volatile("" ::: "memory");   // (a wave's LDS accesses run in order, but the lanes read what others wrote)
#pragma unroll
                    for (int b = 0; b < SB; b++)
                        if (pass * BP + sub * SB + b < I)
#pragma unroll
                            for (int p = 0; p < NP; p++)
                                vf[pass * BP + sub * SB + b][p] = *(lds_half8)(img + b * IMAGE + ((col + 16 * p) ^ (((col + 16 * p) >> 3) & 7)) * 32 + 16 * h);
                    asm volatile("" ::: "memory");
                }
        }
        write_tile(0, pieces);
        if constexpr (NP < 4) write_tile(1, pieces_1);
        request_next(pieces);
        if (TT > 0 && ssq) {          // sums of squares of x over the group's columns
            lds_f32_rw sums = (lds_f32_rw)area;
            __syncthreads();                         // (the area holds the vt images)
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                float q = 0.f;
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int k = 0; k < 8; k++) q += (float)xf[tt][p][k] * (float)xf[tt][p][k];
                q += __shfl_xor(q, 16, 64);
                q += __shfl_xor(q, 32, 64);
                if (g == 0) sums[wave * (16 * TT) + tt * 16 + lm] = q;
            }
            __syncthreads();
            if (tid < T) {
                float q = 0.f;
                for (int w = 0; w < active; w++) q += sums[w * (16 * TT) + tid];
                ssq[cg * T + tid] = q;
            }
        }

        // ---- y tiles ---------------------------------------------------------------------------------------------------------
        // Pass tt of a hand-over is one output per thread: this thread's of every wave, added in wave order.  The reads are issued ahead of
        // where they are added up.
        const int my_t = tid >> 5, my_row = tid & 31;
        const uint32_t my_out = (uint32_t)(my_t * M + my_row) * 4u;
        float *const out = part + (int64_t)cg * T * M;
        // (a wave's two tokens of pass tt)
        auto takes = [&](int tt) { return 16 * tt + 2 * wave < T; };
        auto collect = [&](int buf, int tt, float (&v)[TL_WAVES]) {
            lds_f32 red = (lds_f32)(area) + y_at(buf, tt, my_t, my_row);
            if (takes(tt)) {
#pragma unroll
                for (int w = 0; w < TL_WAVES; w++) v[w] = red[w * Y];
            }
        };
        auto hand_over = [&](int rt, int tt, const float (&v)[TL_WAVES], bool valid) {
            float sum = 0.f;
            if (takes(tt)) {
                sum = v[0];
                if (active == TL_WAVES) {
#pragma unroll
                    for (int w = 1; w < TL_WAVES; w++) sum += v[w];
                } else {
#pragma unroll
                    for (int w = 1; w < TL_WAVES; w++)
                        if (w < active) sum += v[w];
                }
            }
            // (Always issued, to an offset or a buffer of no size that drops it where there is nothing to write: with a store that may or may not be on
            // its way the wait for the requests behind it is a wait for everything.)
            const uint32_t at = 16 * tt + my_t < T && rt * TL_ROWS + my_row < M ? my_out : 0xFFFFFFFFu;
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, sum), tl_buffer(out + ((int64_t)(16 * tt) * M + rt * TL_ROWS), valid ? -1 : 0), (int)at, 0, 0);
        };
        // the second product's result: rows 0-15 ([tt][0]) and 16-31 ([tt][1]) of a tile, D[token 4 g + j, row lm] of each
        float4_t y[TX][2];
        auto leave = [&](int buf) {
            lds_f32x4_rw red = (lds_f32x4_rw)(area + (buf * TL_WAVES + wave) * (Y * 4)) + lane;
#pragma unroll
            for (int tt = 0; tt < TT; tt++)
#pragma unroll
                for (int r = 0; r < 2; r++) red[128 * tt + 64 * r] = y[tt][r];
        };
#pragma unroll
        for (int tt = 0; tt < TT; tt++) y[tt][0] = y[tt][1] = (float4_t){0.f, 0.f, 0.f, 0.f};

        // ---- the rebuild ------------------------------------------------------------------------------------------------
        // Steps s = NP i + p: ahead of block i (i = I: behind the last) the sums of patch p change sign where blocks i - 1 and i differ, then the
        // matrix instruction adds block i's product: the sum so far is kept divided by the block's sign, and a change of sign is exact, so
        // this is the fp32 sum over the blocks for one operation per sign.  The table turns a nibble of the two sign words' difference
        // into four masks; they are looked up LOOK steps ahead, u rows and sign words SETS - 1 blocks ahead, across the end of a tile: the barrier
        // that opens tile n also says that tile n + 1 is in LDS.  The fences keep the compiler from moving the lookups of many steps
        // ahead, for which there are no registers.
        constexpr int STEPS = (I + 1) * NP, SETS = NP == 4 ? 2 : NP == 2 ? 3 : 4, LOOK = NP == 1 || (NP == 2 && I <= 8) ? 2 : 1;
        const int mine_at = wave * (WC / 8) + h * (WC / 16);     // byte of a sign row: this lane's WC / 2 columns
        const int sread = row * SROW + ((mine_at >> 4) ^ swizzle(row)) * 16 + (mine_at & 15);
        const int uread = I * SCH * 1024 + row * 32 + 16 * (h ^ ((row >> 4) & 1));
        float16_t acc[NP];
        uint4_t mask[LOOK + 1][4];
        uint2_t pair_mask[LOOK + 1][4];                          // behind the last block: of rounded pairs
        uint4_t wt[NP][2];                                       // the rounded tile (not SPLIT): this lane's columns 8 e .. + 7 of patch p
        half8_t uf[SETS];
        constexpr int WORDS = NP == 4 ? 2 : 1;
        uint32_t sw[SETS][WORDS], flip[WORDS], flip4[WORDS];
        auto fetch = [&](lds_bytes st, auto ic) {
            constexpr int i = decltype(ic)::value;
            uf[i % SETS] = *(lds_half8)(st + uread + i * 1024);
            lds_bytes at = st + sread + i * (SCH * 1024);
            if constexpr (NP == 4) {
                const uint2_t two = *(lds_uint2)at;
                sw[i % SETS][0] = two[0];
                sw[i % SETS][1] = two[1];
            } else
                sw[i % SETS][0] = NP == 2 ? *(lds_u32)at : *(lds_u16)at;
        };
        auto look_up = [&](auto sc) {
            constexpr int s = decltype(sc)::value, i = s / NP, p = s % NP;
            if constexpr (s < STEPS) {
                constexpr int word = p / 2;
                if constexpr (p == 0) {
#pragma unroll
                    for (int k = 0; k < WORDS; k++) {
                        flip[k] = i < I ? sw[(i + SETS - 1) % SETS][k] ^ sw[i % SETS][k] : ~sw[(i + SETS - 1) % SETS][k];
                        flip4[k] = flip[k] << 4;
                        asm("" : "+v"(flip4[k]));
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    // nibble q of the patch: byte 2 p + q / 2, its upper half first; times 16 it is the place of its masks
                    const uint32_t at = ((q & 1 ? flip4[word] : flip[word]) >> (8 * (2 * (p % 2) + (q >> 1)))) & 0xF0u;
                    if constexpr (i < I || SPLIT) mask[s % (LOOK + 1)][q] = *(lds_uint4)(uintptr_t)at;
                    else pair_mask[s % (LOOK + 1)][q] = *(lds_uint2)(uintptr_t)(at + TL_HALVES);
                }
            }
        };
        auto fetch_first = [&](lds_bytes st) { tl_for<(I < SETS ? I : SETS)>([&](auto ic) { fetch(st, ic); }); };
        auto first_block = [&]() {
#pragma unroll
            for (int p = 0; p < NP; p++)
                acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[0][p], uf[0], (float16_t){0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
            tl_for<LOOK>([&](auto k) { look_up(std::integral_constant<int, NP + decltype(k)::value>{}); });
        };
        tl_wait_lds<0>();
        tl_barrier();                                // the first tile is here, everybody is done with the images
        fetch_first(ring);
        first_block();
        if constexpr (NP == 4) {                     // (no registers for two tiles' pieces)
            write_tile(1, pieces);
            request_next(pieces);
        }
        // ---- the weight's way to memory (TT = 0) --------------------------------------------------------------------------
        // By way of LDS (the wave's own part; the 16-byte chunks XOR-ed with the row) a store instruction writes whole lines; the stores
        // of a tile are issued between the steps of the next one, all at once they would be waited for.
        constexpr int CH = 4 * NP, STORES = TL_ROWS * CH / 64;       // chunks per row, store instructions per tile
        const auto place = [&](int r, int c) { return (lds_half8_rw)(area + wave * (TL_ROWS * WC * 2) + r * (WC * 2) + ((c ^ (r * CH / 16)) % CH) * 16); };
        const uint32_t w_lane = ((uint32_t)(lane / CH) * (uint32_t)N + n0 + 8 * (lane % CH)) * 2u;
        // (the tile as a buffer that ends with the last row: rows beyond it, and all of them where there is no tile, are dropped)
        auto tile_of = [&](int rt, bool valid) { return tl_buffer(w + (int64_t)(rt * TL_ROWS) * N, valid ? min(TL_ROWS, M - rt * TL_ROWS) * N * 2 : 0); };
        auto store_to = [&](__amdgpu_buffer_rsrc_t tile, int k, const half8_t &o) {
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, o), tile, (int)(w_lane + (uint32_t)(k * (64 / CH)) * (uint32_t)N * 2u), 0, 0);
        };
        auto chunk = [&](int k) { return *place(k * (64 / CH) + lane / CH, lane % CH); };
        if constexpr (TT == 0 && NP == 4) {          // (as many stores, all dropped, behind the requests as there are at the end of the loop: the wait counts both)
#pragma unroll
            for (int c = 0; c < STORES; c++) store_to(tile_of(rt0, false), c, (half8_t){0, 0, 0, 0, 0, 0, 0, 0});
        }
        if constexpr (NP == 4) tl_wait_lds<0>();     // (tile 1, written just now with nothing behind it: the loop's wait would let it pass the first barrier unfinished)
        int stage = 0;
#pragma clang loop unroll(disable)
        for (int n = 0; n < len; n++) {
            __builtin_amdgcn_s_setprio(0);
            tl_wait_lds<4>();                        // (a wave's last LDS writes have four lookups or more behind them, or have been waited for)
            tl_barrier();                            // tile n + 1 and the y tiles of n - 2 are in LDS, the stage of n - 1 is free
            const int free_stage = stage == 0 ? STAGES - 1 : stage - 1;
            lds_bytes st = ring + stage * STAGE;
            if (++stage == STAGES) stage = 0;
            lds_bytes st_next = ring + stage * STAGE;
            // Three tiles are in work: tile n is rebuilt, the product of n - 1 is on its way to LDS, and the waves' results of n - 2 are
            // added up between the first steps.
            const int before = (n & 1) ^ 1, oldest = n & 1;
            auto pass_on = [&]() {                   // tile n + 2 into LDS, tile n + 3 requested
                write_tile(free_stage, pieces);
                request_next(pieces);
            };
            if constexpr (NP == 4) pass_on();        // (at the end it would take eight registers more than there are)
            float v[TL_WAVES];
            [[maybe_unused]] const __amdgpu_buffer_rsrc_t last_tile = tile_of(rt0 + n - 1, TT == 0 && n > 0 && wave < active);
            tl_for<STEPS - NP>([&](auto sc) {
                constexpr int k = decltype(sc)::value, s = k + NP, i = s / NP, p = s % NP;
                // (of the two waves of a SIMD the older one goes first; so that both come to the barrier together, the younger one does in the
                // second half)
                if constexpr (k == (STEPS - NP) / 2)
                    if (wave >= TL_WAVES / 2) __builtin_amdgcn_s_setprio(1);
                look_up(std::integral_constant<int, s + LOOK>{});
                if constexpr (p == 0 && i < I && i + SETS - 1 < I) fetch(st, std::integral_constant<int, i + SETS - 1>{});
                if constexpr (s == STEPS - NP) fetch_first(st_next);
                if constexpr (k % 2 == 0 && k / 2 >= 1 && k / 2 <= TT) hand_over(rt0 + n - 2, k / 2 - 1, v, n >= 2);
                if constexpr (k % 2 == 0 && k / 2 < TT) collect(oldest, k / 2, v);
                // (the weight's stores C .. D - 1 of the last tile go with this step)
                constexpr int C = TT ? 0 : (STORES * k + STEPS - NP - 1) / (STEPS - NP), D = TT ? 0 : (STORES * (k + 1) + STEPS - NP - 1) / (STEPS - NP);
                half8_t out[D > C ? D - C : 1];
#pragma unroll
                for (int c = C; c < D; c++) out[c - C] = chunk(c);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (i < I || SPLIT) {
                    asm volatile("" : "+v"(mask[s % (LOOK + 1)][0]), "+v"(mask[s % (LOOK + 1)][1]), "+v"(mask[s % (LOOK + 1)][2]), "+v"(mask[s % (LOOK + 1)][3]));   // (one wait for the four)
#pragma unroll
                    for (int q = 0; q < 4; q++)
#pragma unroll
                        for (int j = 0; j < 4; j++) {
                            const float sum = acc[p][4 * q + j];
                            const uint32_t m = mask[s % (LOOK + 1)][q][j];
                            acc[p][4 * q + j] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, sum) ^ m);
                        }
                    if constexpr (i < I)
                        acc[p] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[i][p], uf[i % SETS], acc[p], 0, 0, 0);
                    asm volatile("" : "+v"(acc[p]));
                } else {
                    // Behind the last block the sums are rounded first, once, to fp16 as a stored weight is, and the sign changed on the rounded pairs: half the
                    // operations, and the same bits.  Of the time with the change in fp32, 100 calls of 8 to 48 tokens: 0.992, none more than 1 % behind (14336 x 4096, 2 blocks, 37 tokens 34.4 /
                    // 33.4 us, 5000 x 4096, 6, 37 26.75 / 26.55); in the rebuild level at 1 to 16 blocks (4096 x 4096, 8 blocks 18.96 / 18.97, 14336 x 4096, 8 47.45 / 47.47).
                    asm volatile("" : "+v"(pair_mask[s % (LOOK + 1)][0]), "+v"(pair_mask[s % (LOOK + 1)][1]), "+v"(pair_mask[s % (LOOK + 1)][2]), "+v"(pair_mask[s % (LOOK + 1)][3]));
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const half2_t two = {(half_t)acc[p][2 * k], (half_t)acc[p][2 * k + 1]};
                        wt[p][k / 4][k % 4] = __builtin_bit_cast(uint32_t, two) ^ pair_mask[s % (LOOK + 1)][k / 2][k % 2];
                    }
                    asm volatile("" : "+v"(wt[p][0]), "+v"(wt[p][1]));
                }
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (D > C) {
#pragma unroll
                    for (int c = C; c < D; c++) store_to(last_tile, c, out[c - C]);
                }
                if constexpr (TT > 0 && k == (STEPS - NP > 1 ? 1 : 0)) leave(before);
            });
            // (the passes for which there were not enough steps)
            constexpr int COLLECTED = (STEPS - NP + 1) / 2 < TT ? (STEPS - NP + 1) / 2 : TT, HANDED = (STEPS - NP - 1) / 2 < TT ? (STEPS - NP - 1) / 2 : TT;
            if constexpr (HANDED < COLLECTED) hand_over(rt0 + n - 2, COLLECTED - 1, v, n >= 2);
            tl_for<TT - COLLECTED>([&](auto k) {
                collect(oldest, COLLECTED + decltype(k)::value, v);
                hand_over(rt0 + n - 2, COLLECTED + decltype(k)::value, v, n >= 2);
            });
            if constexpr (NP < 4) pass_on();
            if constexpr (TT == 0) {
                // A lane holds columns 16 NP h .. + 16 NP - 1 of row l % 32
#pragma unroll
                for (int p = 0; p < NP; p++)
#pragma unroll
                    for (int e = 0; e < 2; e++) *place(row, 2 * NP * h + 2 * p + e) = __builtin_bit_cast(half8_t, wt[p][e]);
                asm volatile("" ::: "memory");               // (the stores' lanes read what others wrote)
                first_block();                               // of tile n + 1
            } else if constexpr (SPLIT) {
                // Two terms per weight: rounded towards zero, and 2^18 times what that leaves, in sums of its own, so that it is no subnormal number where
                // the weight is small (lost: 2^-21 of a weight, 2^-12 of one below 2^-24, and never less than 2^-44).  The lanes trade places as below.
                constexpr float UP = 262144.f;
                float4_t rest[2];
#pragma unroll
                for (int r = 0; r < 2; r++) y[0][r] = rest[r] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    half2_t t[2][8];
#pragma unroll
                    for (int k = 0; k < 8; k++) {
                        const float a = acc[p][2 * k], b = acc[p][2 * k + 1];
                        t[0][k] = __builtin_bit_cast(half2_t, __builtin_amdgcn_cvt_pkrtz(a, b));
                        t[1][k] = (half2_t){(half_t)__builtin_fmaf((float)t[0][k][0], -UP, UP * a), (half_t)__builtin_fmaf((float)t[0][k][1], -UP, UP * b)};
                    }
#pragma unroll
                    for (int term = 1; term >= 0; term--) {
                        uint4_t lo, hi;
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const half2_t a = t[term][k], b = t[term][4 + k];
                            const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
                            lo[k] = r[0];
                            hi[k] = r[1];
                        }
                        float4_t (&sum)[2] = term == 0 ? y[0] : rest;
                        sum[0] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][p], __builtin_bit_cast(half8_t, lo), sum[0], 0, 0, 0);
                        sum[1] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[0][p], __builtin_bit_cast(half8_t, hi), sum[1], 0, 0, 0);
                    }
                }
                // A weight that the terms cannot hold (from about 256 on, where 2^18 * 2^-10 of it is beyond fp16, or infinite) leaves an infinity or
                // a NaN in the second one, whatever its sign, and so in every y of its row.  Such y come from the fp32 weights instead.
                float any = 0.f;
#pragma unroll
                for (int r = 0; r < 2; r++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        any += rest[r][j];
                        y[0][r][j] = __builtin_fmaf(rest[r][j], 1.f / UP, y[0][r][j]);
                    }
                if (__builtin_expect(__builtin_amdgcn_ballot_w64(!__builtin_isfinite(any)) != 0, 0)) {
                    float4_t full[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
                    for (int p = 0; p < NP; p++)
#pragma unroll
                        for (int k = 0; k < 8; k++) {
                            const float a = acc[p][k], b = acc[p][8 + k];
                            const auto w = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b), false, false);
                            const uint32_t lo = w[0], hi = w[1];
                            full[0] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)xf[0][p][k], __builtin_bit_cast(float, lo), full[0], 0, 0, 0);
                            full[1] = __builtin_amdgcn_mfma_f32_16x16x4f32((float)xf[0][p][k], __builtin_bit_cast(float, hi), full[1], 0, 0, 0);
                        }
#pragma unroll
                    for (int r = 0; r < 2; r++)
#pragma unroll
                        for (int j = 0; j < 4; j++)
                            if (!__builtin_isfinite(y[0][r][j])) y[0][r][j] = full[r][j];
                }
                first_block();                   // of tile n + 1
            } else {
                // A lane holds columns 16 NP h + 16 p .. + 15 of row l % 32; lanes 16-31 and 48-63
                // trade their first eight columns for the last eight of lanes 0-15 and 32-47, so that every lane group g has eight columns
                // (16 NP (g / 2) + 16 p + 8 (g % 2) .. + 7) of rows 0-15 in one register set and of rows 16-31 in the other: B operands of
                // v_mfma_f32_16x16x32_f16.
                half8_t wf[NP][2];
#pragma unroll
                for (int p = 0; p < NP; p++) {
                    uint4_t lo, hi;
#pragma unroll
                    for (int k = 0; k < 4; k++) {
                        const auto r = __builtin_amdgcn_permlane16_swap(wt[p][0][k], wt[p][1][k], false, false);
                        lo[k] = r[0];
                        hi[k] = r[1];
                    }
                    wf[p][0] = __builtin_bit_cast(half8_t, lo);
                    wf[p][1] = __builtin_bit_cast(half8_t, hi);
                }
                first_block();                       // of tile n + 1
#pragma unroll
                for (int tt = 0; tt < TT; tt++)
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        y[tt][r] = (float4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                        for (int p = 0; p < NP; p++) y[tt][r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xf[tt][p], wf[p][r], y[tt][r], 0, 0, 0);
                    }
            }
        }
        if (TT == 0) {
#pragma unroll
            for (int c = 0; c < STORES; c++) store_to(tile_of(last_rt, wave < active), c, chunk(c));
            return;
        }
        // the last two tiles
        if (len > 2) tl_barrier();                   // (everybody has collected the tile whose place this is)
        leave((len & 1) ^ 1);
        tl_wait_lds<0>();
        tl_barrier();
#pragma unroll
        for (int n = 0; n < 2; n++) {
            if (len + n < 2) continue;
#pragma unroll
            for (int tt = 0; tt < TT; tt++) {
                float v[TL_WAVES];
                collect((len + n) & 1, tt, v);
                hand_over(rt0 + len + n - 2, tt, v, true);
            }
        }
    }
};

template <int TT, bool SPLIT>
__global__ __launch_bounds__(64 * TL_WAVES, 2) void tile_forward_kernel(const TileGroup grp_, const half_t *__restrict__ x, int N, int T, int K) {
    extern __shared__ __attribute__((aligned(1024))) char tl_lds[];
    lds_bytes_rw lds = (lds_bytes_rw)tl_lds;
    // nibble v, column j of its four (first in the top bit): the sign bit of an fp32 where the bit is set (visible behind walk's first barrier)
    // and behind it the sign bits of two pairs of fp16
    if (threadIdx.x < 64) {
        const uint32_t v = threadIdx.x >> 2, j = threadIdx.x & 3, first = v >> (3 - 2 * (j & 1)) & 1, second = v >> (2 - 2 * (j & 1)) & 1;
        ((__attribute__((address_space(3))) uint32_t *)lds)[threadIdx.x] = v >> (3 - j) & 1 ? 0x80000000u : 0u;
        ((__attribute__((address_space(3))) uint32_t *)lds)[TL_HALVES / 4 + threadIdx.x] = first << 15 | second << 31;
    }
    // (the argument block itself, so that a matrix is picked by its number with scalar loads)
    typedef const __attribute__((address_space(4))) TileGroup *kernarg_group;
    const kernarg_group grp = (kernarg_group)__builtin_amdgcn_kernarg_segment_ptr();
    // Workgroups are dealt round-robin to the 8 XCDs: each XCD takes a contiguous run of (matrix, column group, run of row tiles), so that
    // workgroups with the same slices of x and vt, and column groups that share lines of sign bytes, meet in one L2.
    const int nb = gridDim.x, xcd = blockIdx.x & 7, loc = blockIdx.x >> 3, base = nb >> 3, rem = nb & 7;
    const int v = xcd * base + min(xcd, rem) + loc;
    int j = 0;
    while (j + 1 < grp->n && v >= grp->m[j + 1].first_wg) j++;
    const int r = v - grp->m[j].first_wg, wgs = grp->m[j].wgs, tiles = grp->m[j].row_tiles, cg = r / wgs, run = r - cg * wgs;
    const int rt = (int)((int64_t)tiles * run / wgs), len = (int)((int64_t)tiles * (run + 1) / wgs) - rt;
    float *ssq = j == 0 && run == 0 ? grp->ssq : nullptr;
    if constexpr (TT > 0) {
        const int np = grp->m[j].np, patches = N / 32 - cg * TL_WAVES * np;      // from the group's first column on
        if (patches < TL_WAVES * np) {
            const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), active = patches >> (np >> 1);
            if (wave >= active) {
                auto rest = [&](auto k) {
                    TileKernel<TT, decltype(k)::value, SPLIT>::walk_without_columns(grp->m[j].packed, grp->m[j].u, grp->m[j].part, grp->m[j].I, grp->m[j].M, lds, N, T, K, cg, rt, len, ssq != nullptr, wave, active);
                };
                if (np == 4) rest(std::integral_constant<int, 4>{});
                else if (np == 2) rest(std::integral_constant<int, 2>{});
                else rest(std::integral_constant<int, 1>{});
                return;
            }
        }
    }
    auto walk = [&](auto np, auto blocks) {
        typedef TileKernel<TT, decltype(np)::value, SPLIT> TK;
        if constexpr (decltype(blocks)::value <= TK::max_blocks())
            TK::template walk<decltype(blocks)::value>(grp->m[j].packed, grp->m[j].u, grp->m[j].vt, grp->m[j].part, grp->m[j].w, grp->m[j].M, lds, x, N, T, K, cg, rt, len, ssq);
    };
    // (the narrower widths serve what the wider ones cannot hold, and short runs)
    switch (grp->m[j].np * 32 + grp->m[j].I) {
#define TL_CASE(np, k) \
    case np * 32 + k: walk(std::integral_constant<int, np>{}, std::integral_constant<int, k>{}); break;
        TL_CASE(4, 1) TL_CASE(4, 2) TL_CASE(4, 3) TL_CASE(4, 4)
        TL_CASE(2, 1) TL_CASE(2, 2) TL_CASE(2, 3) TL_CASE(2, 4) TL_CASE(2, 5) TL_CASE(2, 6) TL_CASE(2, 7) TL_CASE(2, 8) TL_CASE(2, 9) TL_CASE(2, 10)
        TL_CASE(1, 1) TL_CASE(1, 2) TL_CASE(1, 3) TL_CASE(1, 4) TL_CASE(1, 5) TL_CASE(1, 6) TL_CASE(1, 7) TL_CASE(1, 8)
        TL_CASE(1, 9) TL_CASE(1, 10) TL_CASE(1, 11) TL_CASE(1, 12) TL_CASE(1, 13) TL_CASE(1, 14) TL_CASE(1, 15) TL_CASE(1, 16)
#undef TL_CASE
    }
}

template <int TT, bool SPLIT = false>
int launch_tile(const TileGroup &grp, int grid, const half_t *x, int N, int T, int K, hipStream_t s) {
    size_t lds = 0;
    for (int j = 0; j < grp.n; j++) {
        const int np = grp.m[j].np, I = grp.m[j].I;
        const size_t b = np == 4 ? TileKernel<TT, 4>::lds_size(I) : np == 2 ? TileKernel<TT, 2>::lds_size(I) : TileKernel<TT, 1>::lds_size(I);
        if (b > lds) lds = b;
    }
    static bs_lds_grant granted[BS_MAX_DEVICES];
    const int st = bs_allow_lds((const void *)tile_forward_kernel<TT, SPLIT>, lds, granted);
    if (st != BS_OK) return st;
    tile_forward_kernel<TT, SPLIT><<<grid, 64 * TL_WAVES, lds, s>>>(grp, x, N, T, K);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

#ifndef TILE_RANKS
// Per matrix the width of its column groups (256 np columns) and how many workgroups share the row tiles of one.  The estimate behind it
// (cycles): a tile costs 1300 + 250 per block and np (with one patch per wave, a chain of mask, product, mask, 420 per block), a
// workgroup's start 2000 + 560 per block and np.
struct TilePlan {
    int grid;                                       // 0: not taken
    double cost;
    int np[TL_GROUP], groups[TL_GROUP], wgs[TL_GROUP];
};
int tile_limit(int np, int T) {
    const int tt = (T + 15) / 16;
    if (tt == 0) return np == 4 ? TileKernel<0, 4>::max_blocks() : np == 2 ? TileKernel<0, 2>::max_blocks() : TileKernel<0, 1>::max_blocks();
    return tt == 1 ? (np == 4 ? TileKernel<1, 4>::max_blocks() : np == 2 ? TileKernel<1, 2>::max_blocks() : TileKernel<1, 1>::max_blocks())
           : tt == 2 ? (np == 4 ? TileKernel<2, 4>::max_blocks() : np == 2 ? TileKernel<2, 2>::max_blocks() : TileKernel<2, 1>::max_blocks())
                     : (np == 4 ? TileKernel<3, 4>::max_blocks() : np == 2 ? TileKernel<3, 2>::max_blocks() : TileKernel<3, 1>::max_blocks());
}
double tile_cost(int np, int I) { return 1300 + (np == 1 ? 420 : 250 * np) * I; }
double start_cost(int np, int I) { return 2000 + 560 * np * I; }
// the plan in which every matrix takes the widest groups up to `widest` that its blocks allow
TilePlan tile_plan_up_to(int widest, const int *I, const int *M, int n, int N, int T) {
    TilePlan p;
    p.grid = 0;
    double work[TL_GROUP], all = 0;
    int tiles[TL_GROUP];
    for (int j = 0; j < n; j++) {
        p.np[j] = widest;
        while (p.np[j] > 1 && I[j] > tile_limit(p.np[j], T)) p.np[j] >>= 1;
        if (I[j] > tile_limit(p.np[j], T)) return p;
        p.groups[j] = (int)bs_cdiv(N, 256 * p.np[j]);
        tiles[j] = (int)bs_cdiv(M[j], TL_ROWS);
        work[j] = p.groups[j] * (tiles[j] * tile_cost(p.np[j], I[j]) + start_cost(p.np[j], I[j]));
        all += work[j];
    }
    // workgroups (one per CU) in proportion to the work, the rest to whoever takes longest
    auto run = [&](int j) { return bs_cdiv(tiles[j], p.wgs[j]) * tile_cost(p.np[j], I[j]) + start_cost(p.np[j], I[j]); };
    int grid = 0;
    for (int j = 0; j < n; j++) {
        const int w = (int)(256 * work[j] / all / p.groups[j]);
        p.wgs[j] = w < 1 ? 1 : w > tiles[j] ? tiles[j] : w;
        grid += p.wgs[j] * p.groups[j];
    }
    int worst;
    while (true) {
        worst = 0;
        for (int j = 1; j < n; j++)
            if (run(j) > run(worst)) worst = j;
        if (grid + p.groups[worst] > 256 || p.wgs[worst] >= tiles[worst]) break;
        p.wgs[worst]++;
        grid += p.groups[worst];
    }
    p.grid = grid;
    p.cost = run(worst) * bs_cdiv(grid, 256);
    return p;
}
TilePlan make_tile_plan(const int *I, const int *M, int n, int N, int K, int T) {
    TilePlan best;
    best.grid = 0;
    for (int widest = 4; widest >= 1; widest >>= 1) {
        const TilePlan p = tile_plan_up_to(widest, I, M, n, N, T);
        if (p.grid != 0 && (best.grid == 0 || p.cost < best.cost)) best = p;
    }
    // Against the strip kernel's steps (128 rows x 128 columns on the busiest CU).  With one patch per wave it is the better one where its
    // rows and strips happen to fill the chip; us strip / this: 7286 x 1024, 11 blocks (2 steps, runs of 4) 18.6 / 21.2, 3328 x 1664, 16 (2, 3) 20.3 / 23.7,
    // 3366 x 2688, 11 (4, 5) 25.6 / 23.1, 2440 x 1536, 14 (2, 2) 20.4 / 17.0, 20191 x 256, 11 (6, 3) 29.4 / 15.5.  And where either does one tile or step of
    // one or two blocks: the hand-over between the waves is half a us (896 x 2176, 1 block 6.8 / 7.5; 643 x 896, 2 blocks 8.4 / 8.9; from 3 blocks
    // on level or ahead; with two patches per wave the one tile is the longer chain: 2668 x 896, 5 blocks 8.4 / 9.9, 3345 x 640, 3 7.8 / 8.6, 2019 x 1664, 3
    // 8.0 / 8.6, against two steps 4398 x 1536, 4 13.1 / 10.2.  Not for three and four tokens at N % 512 == 0, where a decode kernel is the other one).
    // (The line for one patch per wave is asked there too, although it compares with the strip kernel: of 4,200 drawn shapes that it turns away the factor-through
    // kernel's time is 1.05 of this one's at three tokens, 0.73 to 1.67, and 1.22 at four.)
    if (T > 0 && n == 1 && best.grid != 0) {
        const int64_t tiles = bs_cdiv(bs_cdiv(M[0], TL_ROWS), best.wgs[0]);
        const bool wide = best.np[0] == 2 && (T > 4 || N % 512 != 0);
        const long steps = best.np[0] == 1 || I[0] <= 2 || wide ? bs_strip_steps(I[0], M[0], N, T) : 0;
        if ((best.np[0] == 1 && tiles * 0.75 > (double)steps) || ((I[0] <= 2 || wide) && tiles == 1 && steps == 1)) best.grid = 0;
        // (below rank 8 one tile of three blocks is behind too: 2675 x 768, 5 tokens, rank 4 8.3 / 9.1, 414 x 768, 48, rank 5 8.5 / 9.1, 930 x 384, 24, rank 5 7.9 / 8.1; of 150 drawn calls
        // of ranks 4 to 15, up to 9000 x 7680, the others are at most 5 % behind, 6 % ahead on average)
        if (K < 8 && I[0] <= 3 && tiles == 1) best.grid = 0;
    }
    // Several matrices.  When not even one workgroup each fits the chip at once, the second round is the whole call again (10, 9, 1 and 3 blocks of 733, 968, 7844
    // and 215 x 19456, 40 tokens, us strip / this 126 / 253; 118 such groups of 26,000 drawn ones: 0.74 of the strip kernel's rate).  With one patch per
    // wave the strip kernel is ahead where its steps, weighed by their blocks, are few for this plan's cycles: up to three steps (2 x 3072 rows of 1024
    // columns, 4 and 9 blocks, 16 tokens 16.0 / 17.6) from 1180 cycles per step and block on (0.96; below 1.06), beyond them 1030 at 17 to 32 tokens (0.95; below
    // 1.08; up to 16 tokens 1.14 at any ratio), and 900 from 33 tokens on, where y tiles of three token tiles are handed over (4096 + 2 x 1024 rows of 4096, 8 blocks, 48
    // tokens 37 / 43; 0.96, below 1.07).  Of the 26,000 groups 10 % were more than 5 % behind the strip kernel, 4 % more than 10 %; with these lines 5 and 2 %.
    // (Not for three and four tokens at N % 512 == 0, where a decode kernel is the other one.)
    if (T > 0 && n > 1 && best.grid != 0) {
        int np = 4;
        long steps = 0;
        double weighed = 0;
        for (int j = 0; j < n; j++) {
            const long each = T > 4 || N % 512 != 0 ? bs_strip_steps(I[j], M[j], N, T) : 0;
            steps += each;
            weighed += each * (I[j] + 0.6);
            if (best.np[j] < np) np = best.np[j];
        }
        const double line = T > 32 ? 900. : steps <= 3 ? 1180. : T > 16 ? 1030. : 1e9;
        if (best.grid > 256 || (np == 1 && steps > 0 && best.cost > line * weighed)) best.grid = 0;
    }
    // The rebuild's start costs 1.2 us more than reconstruct_tile_kernel's (226 x 896, 1 block 3.6 / 5.1; 1270 x 2688, 2 blocks 5.8 / 6.4), which a single tile
    // does not win back up to a dozen blocks (556 x 384, 9 blocks 7.8 / 8.7; 257 x 384, 16 10.8 / 9.7), nor two tiles of up to four blocks (2304 x 2048, 3,
    // with its product of 775 tokens 30.4 / 31.4; 768 x 7296, 4, 1104 tokens 37.7 / 39.4) or, one patch per wave, of a dozen (748 x 4352, 9, 656 tokens
    // 29.2 / 30.4; 567 x 4608, 8, 144 tokens 28.4 / 28.6); more work per workgroup does (6144 x 4096, 3 blocks, runs of 3, 18.9 / 16.5; 2623 x 2944, 5
    // blocks, 144 tokens, runs of 2, 28.1 / 26.3).  And with five to eight strips of 128 columns reconstruct_tile_kernel has one strip per XCD and is the
    // faster one for a few blocks until a workgroup here has about ten patches per wave (144 tokens: 10743 x 896, 2 blocks 22.5 / 27.2, 17030 x 768,
    // 3 blocks 26.3 / 29.8, 20000 x 896, 2 blocks, 425 tokens 35.3 / 39.0; beyond: 22638 x 896, 2 blocks 30.3 / 28.2; 4 strips: 17030 x 512, 2 blocks 22.0 / 19.8;
    // 9 strips: 10505 x 1152, 2 blocks 32.5 / 29.3).
    if (T == 0 && best.grid != 0) {
        int64_t longest = 0;
        int most = 0, np = 0;
        double patches = 0;                          // per wave of the busiest matrix's workgroups, on average
        for (int j = 0; j < n; j++) {
            const int64_t tiles = bs_cdiv(M[j], TL_ROWS), run = bs_cdiv(tiles, best.wgs[j]);
            if (run > longest) longest = run;
            if (I[j] > most) most = I[j];
            if (best.np[j] > np) np = best.np[j];
            const double each = (double)tiles * best.np[j] / best.wgs[j];
            if (each > patches) patches = each;
        }
        const int64_t strips = N / SF_COLS;
        if ((longest == 1 && most <= 12) || (longest == 2 && (most <= 4 || (np == 1 && most <= 12))) || (strips > 4 && strips <= 8 && most <= 3 && patches <= 10.))
            best.grid = 0;
    }
    return best;
}

TilePlan checked_plan(const int *I, const int *M, int n, int N, int K, int T) {
    TilePlan none;
    none.grid = 0;
    if (n < 1 || n > TL_GROUP || K < TL_MIN_RANK || K > 16 || T < 0 || T > 48 || N < SF_COLS || N % SF_COLS != 0) return none;
    for (int j = 0; j < n; j++)
        // a block's sign and u rows, and 16 tokens of partial sums, lie within 32-bit byte offsets
        if (I[j] < 1 || M[j] < 1 || (int64_t)M[j] * (N >> 3) >= ((int64_t)1 << 32) || (int64_t)M[j] * 64 >= ((int64_t)1 << 32)) return none;
    return bs_cdiv(N, 256) <= 1024 ? make_tile_plan(I, M, n, N, K, T) : none;
}
#endif

}  // namespace

#ifdef TILE_RANKS
int TILE_LAUNCH(const TileGroup &grp, int grid, const half_t *x, int N, int T, int K, int tt, hipStream_t s) {
    return tt == 0 ? launch_tile<0>(grp, grid, x, N, T, K, s) : tt == 1 ? launch_tile<1>(grp, grid, x, N, T, K, s)
           : tt == 2 ? launch_tile<2>(grp, grid, x, N, T, K, s) : launch_tile<3>(grp, grid, x, N, T, K, s);
}
#else

// Column groups (partial sums per output) of every matrix, if this kernel takes them; cycles: of its busiest workgroup, by the plan's estimate.
bool bs_tile_partials(const int *I, const int *M, int n, int N, int K, int T, int *groups, double *cycles) {
    if (T < 1) return false;
    if (T > 48) return n == 1 && (groups[0] = bs_column_partials(I[0], M[0], N, K, T)) > 0;
    const TilePlan p = checked_plan(I, M, n, N, K, T);
    for (int j = 0; p.grid != 0 && j < n; j++) groups[j] = p.groups[j];
    if (cycles) *cycles = p.cost;
    return p.grid != 0;
}

// Columns per workgroup of every matrix where this kernel takes them (T = 0: their rebuild), else false.
bool bs_tile_columns(const int *I, const int *M, int n, int N, int K, int T, int *columns) {
    if (T > 48) return n == 1 && (columns[0] = bs_column_width(I[0], M[0], N, K, T)) > 0;
    const TilePlan p = checked_plan(I, M, n, N, K, T);
    for (int j = 0; p.grid != 0 && j < n; j++) columns[j] = 256 * p.np[j];
    return p.grid != 0;
}

int bs_launch_tile_group(int n, const uint8_t *const *packed, const half_t *const *u, const half_t *const *vt, const int *I, const int *M,
                         float *const *part, float *ssq, const half_t *x, int N, int K, int T, bool split, hipStream_t s) {
    if (T > 48) return n == 1 && !ssq && !split ? bs_launch_column(packed[0], u[0], vt[0], I[0], M[0], part[0], x, N, K, T, s) : BS_ERR_SHAPE;
    const TilePlan p = checked_plan(I, M, n, N, K, T);
    if (p.grid == 0 || T < 1 || (split && T > 16) || !bs_aligned(x, 16)) return BS_ERR_SHAPE;
    TileGroup grp;
    grp.n = n;
    grp.ssq = ssq;
    int first = 0;
    for (int j = 0; j < n; j++) {
        if (!bs_aligned(packed[j], 16) || !bs_aligned(vt[j], 16) || !bs_aligned(u[j], K == 16 ? 16 : 2)) return BS_ERR_SHAPE;
        grp.m[j] = TileMat{packed[j], u[j], vt[j], part[j], nullptr, I[j], M[j], p.np[j], (int)bs_cdiv(M[j], TL_ROWS), first, p.wgs[j]};
        first += p.wgs[j] * p.groups[j];
    }
    for (int j = n; j < TL_GROUP; j++) grp.m[j] = grp.m[0];
    if (K != 16) return split ? BS_ERR_SHAPE : (K < 8 ? bs_launch_tile_few_ranks : bs_launch_tile_ranks)(grp, p.grid, x, N, T, K, (int)bs_cdiv(T, 16), s);
    if (split) return launch_tile<1, true>(grp, p.grid, x, N, T, K, s);
    return T <= 16 ? launch_tile<1>(grp, p.grid, x, N, T, K, s) : T <= 32 ? launch_tile<2>(grp, p.grid, x, N, T, K, s) : launch_tile<3>(grp, p.grid, x, N, T, K, s);
}

// The weights of n <= 4 matrices with the same columns, w[j] f16 [M[j], N]; BS_ERR_SHAPE: not taken, nothing was enqueued.
int bs_launch_tile_rebuild(int n, const uint8_t *const *packed, const half_t *const *u, const half_t *const *vt, const int *I, const int *M,
                           half_t *const *w, int N, int K, hipStream_t s) {
    for (int j = 0; j < n && j < TL_GROUP; j++)
        if (!bs_aligned(packed[j], 16) || !bs_aligned(vt[j], 16) || !bs_aligned(u[j], K == 16 ? 16 : 2) || !bs_aligned(w[j], 16)) return BS_ERR_SHAPE;
    const TilePlan p = checked_plan(I, M, n, N, K, 0);
    if (p.grid == 0) return BS_ERR_SHAPE;
    TileGroup grp;
    grp.n = n;
    grp.ssq = nullptr;
    int first = 0;
    for (int j = 0; j < n; j++) {
        grp.m[j] = TileMat{packed[j], u[j], vt[j], nullptr, w[j], I[j], M[j], p.np[j], (int)bs_cdiv(M[j], TL_ROWS), first, p.wgs[j]};
        first += p.wgs[j] * p.groups[j];
    }
    for (int j = n; j < TL_GROUP; j++) grp.m[j] = grp.m[0];
    return K == 16 ? launch_tile<0>(grp, p.grid, nullptr, N, 0, K, s) : (K < 8 ? bs_launch_tile_few_ranks : bs_launch_tile_ranks)(grp, p.grid, nullptr, N, 0, K, 0, s);
}
#endif
