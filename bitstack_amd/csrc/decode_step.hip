// The two steps of a decoder layer that sit between the compressed linears at
// decode time: RMSNorm, and one position of rotary grouped-query attention over a
// static KV cache.  Small, latency-bound kernels; their point is to replace a
// dozen framework launches per layer by two.
#include "common.h"

namespace {

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// One workgroup per row; the row stays in registers between the two passes.  ADD: the row is fp16(x + add), which is written
// too (sum may be x or add: a thread reads what it overwrites).
constexpr int RMS_THREADS = 256, RMS_MAX_CHUNKS = 8;   // 256 * 8 * 8 halves = 16384 columns

template <bool ADD>
__global__ __launch_bounds__(RMS_THREADS) void rmsnorm_kernel(const half_t *x, const half_t *add, half_t *sum,
                                                              const half_t *__restrict__ weight,
                                                              half_t *__restrict__ y, int H, float eps) {
    __shared__ float wsum[RMS_THREADS / 64];
    const int tid = threadIdx.x;
    const half_t *xr = x + (int64_t)blockIdx.x * H;
    half_t *yr = y + (int64_t)blockIdx.x * H;
    half8_t v[RMS_MAX_CHUNKS];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < RMS_MAX_CHUNKS; c++) {
        const int col = (c * RMS_THREADS + tid) * 8;
        if (col < H) {
            v[c] = *reinterpret_cast<const half8_t *>(xr + col);
            if (ADD) {
                v[c] += *reinterpret_cast<const half8_t *>(add + (int64_t)blockIdx.x * H + col);
                *reinterpret_cast<half8_t *>(sum + (int64_t)blockIdx.x * H + col) = v[c];
            }
#pragma unroll
            for (int e = 0; e < 8; e++) ss += (float)v[c][e] * (float)v[c][e];
        }
    }
    ss = wave_sum(ss);
    if ((tid & 63) == 0) wsum[tid >> 6] = ss;
    __syncthreads();
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < RMS_THREADS / 64; w++) total += wsum[w];
    const float r = rsqrtf(total / (float)H + eps);
#pragma unroll
    for (int c = 0; c < RMS_MAX_CHUNKS; c++) {
        const int col = (c * RMS_THREADS + tid) * 8;
        if (col < H) {
            const half8_t w8 = *reinterpret_cast<const half8_t *>(weight + col);
            half8_t o;
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = (half_t)((float)(half_t)((float)v[c][e] * r) * (float)w8[e]);
            *reinterpret_cast<half8_t *>(yr + col) = o;
        }
    }
}

// One position of attention: a workgroup serves HP query heads of one KV head and sequence, its waves walk the cache in
// tiles of 16 positions (tile = wave, wave + WAVES, ...) with a running (max, sum, weighted v) per wave, merged through LDS.
//
// Both products run on the matrix cores, the heads as columns (HP of 16 used):
//   scores  S[position, head] = K q     16x16x32, K rows as loaded (a lane: position l % 16, dimensions 32 c + 8 (l / 16) ..)
//   output  O[dim, head] += V^T P       16x16x32, four positions twice: P is split into two fp16 terms, p = hi + lo to 2^-22,
//                                       and the eight k slots of a lane hold {hi, lo} against {v, v}, so the weights keep the
//                                       precision they had as fp32 numbers; where an infinite v makes NaN of that, the wave
//                                       goes over its positions again with fp32 weights (the check: 0.1 us)
// A lane of the scores holds positions 4 (l / 16) + i of head l % 16, which is what the second product wants of P; V needs no
// transposition either: a lane loads dimensions 8 r .. 8 r + 7 (r = l % 16) of its four positions, and product number j takes
// half j of each, so that its row r is dimension 8 r + j.  K of the next tile is requested behind the scores, V behind the
// output product.
//
// What bounds it: the fetches, and below about a thousand positions the chain position -> first tile -> merge.  Folding
// position by position on the VALU (32 instructions per position and head) took 46 us
// on 8 sequences x 64 heads (8 KV heads) at position 2100 where this takes 22.5 (69 MB: 3.1 TB/s), 18.7 / 8.8 on 16 x 32 at 300,
// 8.2 / 6.9 on 1 x 32 at 384.
constexpr int ATT_D = 128, ATT_MAX_LEN = 8192, ATT_TILE = 16, ATT_WHOLE = 512, ATT_MAX_SPLITS = 16, ATT_PART = ATT_D + 4;

template <int HP, int WAVES, bool SPLIT>
__global__ __launch_bounds__(WAVES * 64) void attention_decode_kernel(
    const half_t *__restrict__ qkv, half_t *__restrict__ kcache, half_t *__restrict__ vcache,
    const half_t *__restrict__ cosv, const half_t *__restrict__ sinv, const int64_t *__restrict__ pos_ptr,
    half_t *__restrict__ out, float *__restrict__ part, int B, int heads, int kv_heads, int max_len) {
    constexpr int THREADS = WAVES * 64;
    __shared__ __attribute__((aligned(16))) half_t qrot[HP][ATT_D];            // rotated queries
    __shared__ __attribute__((aligned(16))) half_t knew[ATT_D], vnew[ATT_D];   // this position's rotated k and v
    __shared__ float wm[HP][WAVES], wl[HP][WAVES];                             // per wave: running max, sum of exp
    __shared__ __attribute__((aligned(16))) float wacc[HP][WAVES][ATT_D];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, r16 = lane & 15, g = lane >> 4;
    // The workgroups of one KV head read the same rows: on one XCD (workgroups are dealt to the eight in turn) they share them
    // in its L2.
    const int rep = heads / kv_heads, share = rep / HP, pairs = B * kv_heads;
    const int id = blockIdx.x;
    const bool dealt = pairs % 8 == 0;
    const int pair = dealt ? (id & 7) + 8 * (id / (8 * share)) : id / share, sub = dealt ? (id >> 3) % share : id % share;
    const int b = pair / kv_heads, hk = pair % kv_heads, head0 = hk * rep + sub * HP;
    const int row = (heads + 2 * kv_heads) * ATT_D;
    const half_t *qh = qkv + (int64_t)b * row + (int64_t)head0 * ATT_D;        // the HP query heads, contiguous
    const half_t *kn = qkv + (int64_t)b * row + (heads + hk) * ATT_D;
    const half_t *vn = qkv + (int64_t)b * row + (heads + kv_heads + hk) * ATT_D;
    half_t *orow = out + ((int64_t)b * heads + head0) * ATT_D;
    // Work items of the set-up: HP * 64 query pairs, 64 key pairs (dimension i and i + 64 rotate together), 128 values.  What
    // does not depend on the position is fetched before the position is known.
    constexpr int QP = HP * 64, ITEMS = QP + 64 + ATT_D;
    static_assert(ITEMS <= THREADS, "one set-up item per thread");
    float fa = 0.f, fb = 0.f;
    if (tid < QP) {
        const int h = tid >> 6, i = tid & 63;
        fa = (float)qh[h * ATT_D + i]; fb = (float)qh[h * ATT_D + i + 64];
    } else if (tid < QP + 64) {
        fa = (float)kn[tid - QP]; fb = (float)kn[tid - QP + 64];
    } else if (tid < ITEMS) {
        fa = (float)vn[tid - QP - 64];
    }
    const int64_t pos64 = *pos_ptr;
    if (pos64 < 0 || pos64 >= max_len) {         // nothing sensible to do: defined output, no access outside the cache
        if (!SPLIT)
            for (int it = tid; it < HP * ATT_D; it += THREADS) orow[it] = (half_t)0;
        return;
    }
    // With the positions split, workgroup y of gridDim.y takes every gridDim.y-th round of tiles; up to ATT_WHOLE positions
    // the first takes them all and writes the result itself (two rounds are shorter than the way through the second launch).
    const bool split = SPLIT && pos64 > ATT_WHOLE;
    if (SPLIT && !split && blockIdx.y > 0) return;
    const int pos = (int)pos64, tiles = (pos + ATT_TILE - 1) / ATT_TILE;
    half_t *kc = kcache + ((int64_t)b * kv_heads + hk) * max_len * ATT_D;
    half_t *vc = vcache + ((int64_t)b * kv_heads + hk) * max_len * ATT_D;

    half8_t k8[4], v8[4];
    auto fetch_k = [&](int t) {                  // rows past the last are the last again; their scores are masked
        const half_t *p = kc + (int64_t)min(t * ATT_TILE + r16, pos - 1) * ATT_D + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; c++) k8[c] = *reinterpret_cast<const half8_t *>(p + 32 * c);
    };
    auto fetch_v = [&](int t) {
#pragma unroll
        for (int i = 0; i < 4; i++)
            v8[i] = *reinterpret_cast<const half8_t *>(vc + (int64_t)min(t * ATT_TILE + 4 * g + i, pos - 1) * ATT_D + 8 * r16);
    };
    const int step = split ? WAVES * (int)gridDim.y : WAVES;
    const int first = SPLIT ? wave + WAVES * (int)blockIdx.y : wave;
    int t = first;
    const bool own = t == tiles % step;          // the wave whose turn is next takes this step's own position
    if (t < tiles) { fetch_k(t); fetch_v(t); }

    if (tid < QP + 64) {
        const int i = tid & 63;
        const float c = (float)cosv[(int64_t)pos * (ATT_D / 2) + i], sn = (float)sinv[(int64_t)pos * (ATT_D / 2) + i];
        const half_t lo = (half_t)(fa * c - fb * sn), hi = (half_t)(fb * c + fa * sn);
        half_t *to = tid < QP ? qrot[tid >> 6] : knew;
        to[i] = lo; to[i + 64] = hi;
    } else if (tid < ITEMS) {
        vnew[tid - QP - 64] = (half_t)fa;
    }
    __syncthreads();
    if (sub == 0 && blockIdx.y == 0 && tid < ATT_D) {               // one workgroup of the KV head appends this position to the cache
        kc[(int64_t)pos * ATT_D + tid] = knew[tid];
        vc[(int64_t)pos * ATT_D + tid] = vnew[tid];
    }

    half8_t q8[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        q8[c] = r16 < HP ? *reinterpret_cast<const half8_t *>(&qrot[r16 < HP ? r16 : 0][32 * c + 8 * g]) : (half8_t)(half_t)0;
    const float scale2 = 0.08838834764831845f * 1.4426950408889634f;    // 1 / sqrt(128) * log2(e): the softmax runs in base 2
    float m = -INFINITY, l = 0.f;                // of head l % 16; the sum over this lane's positions only
    float4_t acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = (float4_t)0.f;
    auto scores = [&]() {
        float4_t s = (float4_t)0.f;
#pragma unroll
        for (int c = 0; c < 4; c++) s = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[c], q8[c], s, 0, 0, 0);
        return s;
    };
    auto fold = [&](const float4_t s, int valid) {                      // the tile's first `valid` positions (at least one)
        float p[4], mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p[i] = 4 * g + i < valid ? s[i] * scale2 : -INFINITY;
            mx = fmaxf(mx, p[i]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float mn = fmaxf(m, mx), r = __builtin_amdgcn_exp2f(m - mn);      // exp2(-inf) = 0 on the first tile
        m = mn;
        half8_t p8;
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            p[i] = __builtin_amdgcn_exp2f(p[i] - mn);
            sum += p[i];
            p8[i] = (half_t)p[i];
            p8[i + 4] = (half_t)(p[i] - (float)p8[i]);
        }
        l = l * r + sum;
        if (__any(r != 1.f)) {
#pragma unroll
            for (int j = 0; j < 8; j++) acc[j] *= r;
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const half8_t v = {v8[0][j], v8[1][j], v8[2][j], v8[3][j], v8[0][j], v8[1][j], v8[2][j], v8[3][j]};
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, p8, acc[j], 0, 0, 0);
        }
    };
    while (t < tiles) {
        const float4_t s = scores();
        const int next = t + step;
        if (next < tiles) fetch_k(next);
        fold(s, pos - t * ATT_TILE);
        if (next < tiles) fetch_v(next);
        t = next;
    }
    auto take_own = [&]() {                      // this step's own k and v, from LDS: a tile with one position
#pragma unroll
        for (int c = 0; c < 4; c++) {
            k8[c] = *reinterpret_cast<const half8_t *>(&knew[32 * c + 8 * g]);
            v8[c] = *reinterpret_cast<const half8_t *>(&vnew[8 * r16]);
        }
    };
    if (own) {
        take_own();
        fold(scores(), 1);
    }

    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (r16 < HP && g == 0) { wm[r16][wave] = m; wl[r16][wave] = l; }
    const float4_t sums = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
    const float sum = (sums[0] + sums[1]) + (sums[2] + sums[3]);
    if (__builtin_expect(__any(sum != sum), 0)) {
        // An infinite v: times a second term of zero or below it, or a masked weight, it is NaN in the output product.  The wave's
        // positions once more, head by head, each weight as one fp32 number: a lane owns dimensions 8 r16 .. 8 r16 + 7.
#pragma unroll 1
        for (int h = 0; h < HP; h++) {
            float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            auto add = [&](const float4_t s, int valid) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const float w = __shfl(__builtin_amdgcn_exp2f(s[i] * scale2 - m), (lane & 48) | h, 64);
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (4 * g + i < valid) o[e] += w * (float)v8[i][e];
                }
            };
            for (t = first; t < tiles; t += step) {
                fetch_k(t);
                fetch_v(t);
                add(scores(), pos - t * ATT_TILE);
            }
            if (own) {
                take_own();
                add(scores(), 1);
            }
#pragma unroll
            for (int e = 0; e < 8; e++) {
                o[e] += __shfl_xor(o[e], 16, 64);
                o[e] += __shfl_xor(o[e], 32, 64);
                if (g == 0) wacc[h][wave][8 * r16 + e] = o[e];
            }
        }
    } else if (r16 < HP) {
#pragma unroll
        for (int i = 0; i < 4; i++) {            // row 4 g + i of product j is dimension 8 (4 g + i) + j
            float *to = &wacc[r16][wave][8 * (4 * g + i)];
            *reinterpret_cast<float4_t *>(to) = (float4_t){acc[0][i], acc[1][i], acc[2][i], acc[3][i]};
            *reinterpret_cast<float4_t *>(to + 4) = (float4_t){acc[4][i], acc[5][i], acc[6][i], acc[7][i]};
        }
    }
    __syncthreads();
    for (int it = tid; it < HP * ATT_D; it += THREADS) {
        const int h = it >> 7, dim = it & (ATT_D - 1);
        float mx = wm[h][0];
#pragma unroll
        for (int w = 1; w < WAVES; w++) mx = fmaxf(mx, wm[h][w]);
        float o = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < WAVES; w++) {
            const float r = wl[h][w] != 0.f ? __builtin_amdgcn_exp2f(wm[h][w] - mx) : 0.f;    // 0: a wave that saw no position
            o += r * wacc[h][w][dim];
            den += r * wl[h][w];
        }
        if (split) {                             // part[head][split][max, sum, pad, pad, weighted v]
            float *to = part + (((int64_t)b * heads + head0 + h) * gridDim.y + blockIdx.y) * ATT_PART;
            to[4 + dim] = o;
            if (dim == 0) { to[0] = mx; to[1] = den; }
        } else {
            orow[it] = (half_t)(o / den);
        }
    }
}

// The splits of one head put together: every load is requested at once, one memory round trip.
template <int MAXS>
__global__ __launch_bounds__(ATT_D) void attention_merge_kernel(const float *__restrict__ part, const int64_t *__restrict__ pos_ptr,
                                                                half_t *__restrict__ out, int splits, int max_len) {
    const int dim = threadIdx.x;
    const float *p = part + (int64_t)blockIdx.x * splits * ATT_PART;
    const int64_t pos = *pos_ptr;
    float m[MAXS], l[MAXS], v[MAXS];
#pragma unroll
    for (int i = 0; i < MAXS; i++) {
        const float *q = p + (int64_t)(i < splits ? i : 0) * ATT_PART;
        m[i] = q[0]; l[i] = i < splits ? q[1] : 0.f; v[i] = q[4 + dim];
    }
    if (pos >= 0 && pos <= ATT_WHOLE) return;    // written by the first launch
    if (pos < 0 || pos >= max_len) {             // nothing was summed
        out[(int64_t)blockIdx.x * ATT_D + dim] = (half_t)0;
        return;
    }
    float mx = m[0], o = 0.f, den = 0.f;
#pragma unroll
    for (int i = 1; i < MAXS; i++) mx = fmaxf(mx, m[i]);
#pragma unroll
    for (int i = 0; i < MAXS; i++) {
        const float r = l[i] != 0.f ? __builtin_amdgcn_exp2f(m[i] - mx) : 0.f;
        o += l[i] != 0.f ? r * v[i] : 0.f;
        den += r * l[i];
    }
    out[(int64_t)blockIdx.x * ATT_D + dim] = (half_t)(o / den);
}

// Greedy token: index of the largest of V fp16 values per row (the lowest index among
// equals; NaN never wins), one workgroup per row.  The first one also counts the position up where one is given: a launch of its
// own for that is 4 us of a step.  6.4 us for 32000 values (four requests ahead instead of one by one: the same).
constexpr int ARG_THREADS = 1024;

__global__ __launch_bounds__(ARG_THREADS) void argmax_kernel(const half_t *__restrict__ x, int64_t *__restrict__ out, int64_t *__restrict__ pos, int V) {
    __shared__ float bv[ARG_THREADS / 64];
    __shared__ int bi[ARG_THREADS / 64];
    const int tid = threadIdx.x;
    const half_t *row = x + (int64_t)blockIdx.x * V;
    float best = -INFINITY;
    int at = 0x7fffffff;
    const int v8 = V & ~7;
    for (int c = tid * 8; c < v8; c += ARG_THREADS * 8) {       // ascending per thread: a later equal value never replaces
        const half8_t v = *reinterpret_cast<const half8_t *>(row + c);
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const float f = (float)v[e];
            if (f > best || (f == best && c + e < at)) { best = f; at = c + e; }
        }
    }
    for (int c = v8 + tid; c < V; c += ARG_THREADS) {
        const float f = (float)row[c];
        if (f > best || (f == best && c < at)) { best = f; at = c; }
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
        const float ob = __shfl_xor(best, o, 64);
        const int oa = __shfl_xor(at, o, 64);
        if (ob > best || (ob == best && oa < at)) { best = ob; at = oa; }
    }
    if ((tid & 63) == 0) { bv[tid >> 6] = best; bi[tid >> 6] = at; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < ARG_THREADS / 64; w++)
            if (bv[w] > best || (bv[w] == best && bi[w] < at)) { best = bv[w]; at = bi[w]; }
        out[blockIdx.x] = at == 0x7fffffff ? 0 : at;            // a row of NaNs / -inf: index 0
        if (pos && blockIdx.x == 0) *pos += 1;
    }
}

}  // namespace

int bs_launch_argmax(const half_t *x, int64_t *out, int64_t *pos, int B, int V, hipStream_t s) {
    argmax_kernel<<<B, ARG_THREADS, 0, s>>>(x, out, pos, V);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int bs_launch_rmsnorm(const half_t *x, const half_t *weight, half_t *y, int T, int H, float eps, hipStream_t s) {
    if (H > RMS_THREADS * RMS_MAX_CHUNKS * 8) return BS_ERR_SHAPE;
    rmsnorm_kernel<false><<<T, RMS_THREADS, 0, s>>>(x, nullptr, nullptr, weight, y, H, eps);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int bs_launch_add_rmsnorm(const half_t *x, const half_t *add, half_t *sum, const half_t *weight, half_t *y, int T, int H, float eps,
                          hipStream_t s) {
    if (H > RMS_THREADS * RMS_MAX_CHUNKS * 8) return BS_ERR_SHAPE;
    rmsnorm_kernel<true><<<T, RMS_THREADS, 0, s>>>(x, add, sum, weight, y, H, eps);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

template <int HP, int WAVES, bool SPLIT>
static void launch_attention(const half_t *qkv, half_t *kcache, half_t *vcache, const half_t *cos, const half_t *sin,
                             const int64_t *pos, half_t *out, float *part, int splits, int B, int heads, int kv_heads, int max_len,
                             hipStream_t s) {
    attention_decode_kernel<HP, WAVES, SPLIT><<<dim3((int64_t)B * heads / HP, splits), WAVES * 64, 0, s>>>(
        qkv, kcache, vcache, cos, sin, pos, out, part, B, heads, kv_heads, max_len);
}

// Parts that the positions are cut into (1: not cut).  One KV head's rows go through one CU at about 60 GB/s, so few heads over
// a long cache leave the chip idle; the parts cost a second, summing launch, and up to ATT_WHOLE positions they gain nothing.
// Only the length of the cache is known here, so the line lies where the mean over its positions is the same (us not cut / cut,
// mean of six positions from 6 to 99 % of the cache): one sequence, 32 heads on 8 KV heads 8.0 / 8.9 at a length of 896, 8.5 / 8.9 at 1024,
// 9.1 / 8.8 at 1152, 12.8 / 9.5 at 2048; 64 on 8 8.6 / 8.9, 9.2 / 8.9 at 1024 and 1152; four sequences of 32 on 8 8.9 / 9.4, 9.5 / 9.4.
// A head to a workgroup merges for less: 32 on 32 8.2 / 8.7 at 896, 8.8 / 8.6 at 1024; 8 on 8 7.9 / 8.3, 8.4 / 8.3.
constexpr int ATT_SPLIT_LEN = 1100, ATT_SPLIT_LEN_SINGLE = 1000;
static int attention_splits(int B, int heads, int kv_heads, int max_len) {
    const int rep = heads / kv_heads, hp = rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1;
    const int64_t groups = (int64_t)B * heads / hp;
    if (max_len < (hp == 1 ? ATT_SPLIT_LEN_SINGLE : ATT_SPLIT_LEN) || groups > 128 || groups < 1) return 1;
    const int64_t fill = 256 / groups, longest = bs_cdiv(max_len, 256);       // 256 positions: one tile for each of 16 waves
    const int64_t splits = fill < longest ? fill : longest;
    return splits > ATT_MAX_SPLITS ? ATT_MAX_SPLITS : (int)splits;
}

int64_t bs_attention_parts_bytes(int B, int heads, int kv_heads, int max_len) {
    const int splits = attention_splits(B, heads, kv_heads, max_len);
    return splits > 1 ? (int64_t)B * heads * splits * ATT_PART * 4 : 0;
}

int bs_launch_attention_decode(const half_t *qkv, half_t *kcache, half_t *vcache, const half_t *cos, const half_t *sin,
                               const int64_t *pos, half_t *out, int B, int heads, int kv_heads, int head_dim,
                               int max_len, float *part, hipStream_t s) {
    if (head_dim != ATT_D || max_len > ATT_MAX_LEN) return BS_ERR_SHAPE;
    const int rep = heads / kv_heads;
    const int64_t all = (int64_t)B * heads;
    const int splits = part ? attention_splits(B, heads, kv_heads, max_len) : 1;
    if (splits > 1) {
        auto *launch = rep % 4 == 0 ? launch_attention<4, 16, true> : rep % 2 == 0 ? launch_attention<2, 16, true> : launch_attention<1, 16, true>;
        launch(qkv, kcache, vcache, cos, sin, pos, out, part, splits, B, heads, kv_heads, max_len, s);
        BS_LAUNCH_CHECK();
        auto *merge = splits <= 4 ? attention_merge_kernel<4> : splits <= 8 ? attention_merge_kernel<8> : attention_merge_kernel<ATT_MAX_SPLITS>;
        merge<<<(int)all, ATT_D, 0, s>>>(part, pos, out, splits, max_len);
        BS_LAUNCH_CHECK();
        return BS_OK;
    }
    // As few heads of a KV head per workgroup as still give at most one workgroup of 16 waves per CU: a CU's time is that of
    // one KV head's rows however many heads share them, and fewer heads merge faster.  Past that, workgroups of 8 waves, two
    // on a CU.
    const int hp = rep % 4 == 0 && all > 512 ? 4 : rep % 2 == 0 && all > 256 ? 2 : 1;
    const bool wide = all / hp <= 256;
    auto *launch = hp == 4 ? (wide ? launch_attention<4, 16, false> : launch_attention<4, 8, false>)
                 : hp == 2 ? (wide ? launch_attention<2, 16, false> : launch_attention<2, 8, false>)
                           : (wide ? launch_attention<1, 16, false> : launch_attention<1, 8, false>);
    launch(qkv, kcache, vcache, cos, sin, pos, out, nullptr, 1, B, heads, kv_heads, max_len, s);
    BS_LAUNCH_CHECK();
    return BS_OK;
}
