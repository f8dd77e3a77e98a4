// What sits between the compressed linears of a decoder layer when a whole prompt goes through it: rotary embedding with the
// store of k and v to the cache, the SiLU product of the MLP, and a residual sum with the RMSNorm that follows it.  Each is one
// pass over its operands, bound by memory; as framework operations they were eleven passes and launches for the rotation and
// the two cache copies, two for the SiLU product and two for the sum and the norm, with every step rounded to fp16.  Here
// each result is computed in fp32 and rounded once.
#include "common.h"

#include <algorithm>
#include <type_traits>

namespace {

constexpr int THREADS = 256;

// One workgroup per token; an item is V dimensions of a head (for q and k together with the V that rotate against them).
// 1400 tokens, 32 + 2 * 8 heads of 128: about 115 us before, 7.4 now (23 MB read and written).
template <int V>
__global__ __launch_bounds__(THREADS) void rope_store_kernel(half_t *__restrict__ q, const half_t *__restrict__ k,
                                                             const half_t *__restrict__ v, const half_t *__restrict__ cosv,
                                                             const half_t *__restrict__ sinv, half_t *__restrict__ kcache,
                                                             half_t *__restrict__ vcache, int ldq, int ldkv, int n, int heads,
                                                             int kv_heads, int d, int max_len) {
    typedef half_t vec_t __attribute__((ext_vector_type(V)));
    const int token = blockIdx.x, b = token / n, pos = token % n, d2 = d / 2;
    const int per = d2 / V, qi = heads * per, ki = kv_heads * per;               // items of q and of k; v has 2 * ki
    q += (int64_t)token * ldq;
    k += (int64_t)token * ldkv;
    v += (int64_t)token * ldkv;
    cosv += (int64_t)pos * d2;
    sinv += (int64_t)pos * d2;
    const int64_t head_stride = (int64_t)max_len * d, at = (int64_t)b * kv_heads * head_stride + (int64_t)pos * d;
    for (int it = threadIdx.x; it < qi + 3 * ki; it += THREADS) {
        if (it >= qi + ki) {
            const int j = it - qi - ki, h = j / (2 * per), c = (j % (2 * per)) * V;
            *reinterpret_cast<vec_t *>(vcache + at + h * head_stride + c) = *reinterpret_cast<const vec_t *>(v + h * d + c);
            continue;
        }
        const bool is_q = it < qi;
        const int j = is_q ? it : it - qi, h = j / per, c = (j % per) * V;
        const half_t *from = (is_q ? q : k) + h * d + c;
        half_t *to = is_q ? q + h * d + c : kcache + at + h * head_stride + c;
        const vec_t a = *reinterpret_cast<const vec_t *>(from), e = *reinterpret_cast<const vec_t *>(from + d2);
        const vec_t cs = *reinterpret_cast<const vec_t *>(cosv + c), sn = *reinterpret_cast<const vec_t *>(sinv + c);
        vec_t lo, hi;
#pragma unroll
        for (int i = 0; i < V; i++) {
            lo[i] = (half_t)((float)a[i] * (float)cs[i] - (float)e[i] * (float)sn[i]);
            hi[i] = (half_t)((float)e[i] * (float)cs[i] + (float)a[i] * (float)sn[i]);
        }
        *reinterpret_cast<vec_t *>(to) = lo;
        *reinterpret_cast<vec_t *>(to + d2) = hi;
    }
}

// y[T, width] = silu(gate) * up, rows of gate and up ld apart; eight values per thread.  y may be gate or up (ld == width): a
// thread reads what it overwrites.  1400 x 14336: 36 us as
// two operations, 18.9 now (120 MB: 6.4 TB/s).
__global__ __launch_bounds__(THREADS) void silu_mul_kernel(const half_t *gate, const half_t *up, half_t *y, int width, int ld) {
    const int i = (blockIdx.x * THREADS + threadIdx.x) * 8, count = width;
    gate += (int64_t)blockIdx.y * ld;
    up += (int64_t)blockIdx.y * ld;
    y += (int64_t)blockIdx.y * width;
    auto one = [](float a, float b) { return (half_t)(a / (1.f + __expf(-a)) * b); };
    if (i + 8 <= count) {
        const half8_t a = *reinterpret_cast<const half8_t *>(gate + i), b = *reinterpret_cast<const half8_t *>(up + i);
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = one((float)a[e], (float)b[e]);
        *reinterpret_cast<half8_t *>(y + i) = o;
    } else {
        for (int j = i; j < count; j++) y[j] = one((float)gate[j], (float)up[j]);
    }
}

// Causal attention of a whole prompt over the cache that rope_store_kernel has filled.  A wave takes 16 QT queries of one head and
// walks the positions up to its last query 64 at a time with a running (max, sum, weighted v), which takes up 32 of them at a time.  The waves of a workgroup share a KV head: their items are (tile of
// queries, head of the group), the head fastest, so that they need the same rows.  These come to LDS a stage of 64 positions at a time, requested one stage ahead, straight from
// memory (no registers, no LDS write instructions), one barrier per stage.  The operands lie as in the decode step's attention (decode_step.hip): scores S[position, query] =
// K q, output O[dim, query] += V^T P, on 16x16x32 products whose lane layouts fit without any shuffle - a lane of the scores holds four positions of one query in each of
// two tiles of 16 positions, which are the eight k slots of the output product, and V is used as it lies, product j taking half j of a lane's 16 bytes.  The 16-byte
// pieces of a row of K are XOR-ed with the row's number: a score fragment reads one piece of 16 rows, which lie a whole turn of the banks apart.
// The weights are rounded to fp16 for the second product; their sum is that of the fp32 weights.
// What bounds it: with many queries the issue of the softmax's instructions and of the products (750 TFLOP/s of the lower triangle), with few the chain of a stage, 1.2 us.
// us, every wave reading its own rows from L2 32 positions at a time / this: 2 x 700 queries with 32 heads on 8 KV heads 39.4 / 22.7, 4 x 300 20.5 / 13.3, 100 7.3 / 5.2, 4000 301 / 174,
// 4 x 1500 with 64 on 16 345 / 219, 64 on 64 357 / 244, 8 x 2048 with 64 on 8 1211 / 736.  A stage of 64 as two steps of 32 positions: 28.5 on the first, 198 on the fourth.
// Error against float64: 2.469e-4 on the first, 2.494e-4 on 1 x 2000 with 8 on 2, as before.  One maximum for the 64 positions is 5 % faster (21.7 on the first), but fewer weights are
// then a maximum, exact when rounded: 2.483e-4 and 2.506e-4.  The rounded weights' sum, by a product with ones, is no faster than that.
constexpr int AP_D = 128, AP_WAVES = 4, AP_P = 64;       // (AP_P: positions of a stage)
constexpr int AP_CHUNKS = 2 * (AP_P / 4) / AP_WAVES;                // requests per wave and stage: of 1 KB, four rows; K, then V

typedef __attribute__((address_space(3))) void *ap_lds;

// the larger of v here and in the lane whose number differs by W (16 or 32), or (SUM) both together
template <int W, bool SUM = false>
__device__ __forceinline__ float across(float v) {
    const uint32_t u = __builtin_bit_cast(uint32_t, v);
    const auto r = W == 16 ? __builtin_amdgcn_permlane16_swap(u, u, false, false) : __builtin_amdgcn_permlane32_swap(u, u, false, false);
    const uint32_t a = r[0], b = r[1];
    return SUM ? __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b) : fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
}

template <int QT>
__global__ __launch_bounds__(AP_WAVES * 64, 2) void attention_prefill_kernel(const half_t *__restrict__ q, const half_t *__restrict__ kcache,
                                                                             const half_t *__restrict__ vcache, half_t *__restrict__ out,
                                                                             int ldq, int n, int heads, int kv_heads, int max_len, int chunks) {
    // (an array per operand and stage: the compiler then knows that a request for one does not touch the others)
    __shared__ __attribute__((aligned(1024))) half_t sk0[AP_P * AP_D], sk1[AP_P * AP_D], sv0[AP_P * AP_D], sv1[AP_P * AP_D];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
    const int group = heads / kv_heads, items = group * ((n + (16 * QT) - 1) / (16 * QT));
    const int at = (int)(blockIdx.y + blockIdx.z * gridDim.y);
    if (at >= chunks) return;
    const int first = (chunks - 1 - at) * AP_WAVES, item = min(first + wave, items - 1);     // the longest first
    const int b = blockIdx.x / kv_heads, hk = blockIdx.x - b * kv_heads, head = hk * group + item % group;
    const int q0 = item / group * (16 * QT);
    const bool mine = first + wave < items;
    const int stages = min(first + AP_WAVES - 1, items - 1) / group * (16 * QT) / AP_P + 1;       // (a tile of queries lies within a stage)
    const int64_t row = (int64_t)heads * AP_D;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc((void *)(kcache + ((int64_t)b * kv_heads + hk) * max_len * AP_D), 0, -1, 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void *)(vcache + ((int64_t)b * kv_heads + hk) * max_len * AP_D), 0, -1, 0x00020000);

    auto request = [&](auto stage, int p0) {         // (rows past the last are the last again; their scores are masked)
        half_t *const k_to = decltype(stage)::value ? sk1 : sk0, *const v_to = decltype(stage)::value ? sv1 : sv0;
#pragma unroll
        for (int j = 0; j < AP_CHUNKS / 2; j++) {
            const int r = (wave * (AP_CHUNKS / 2) + j) * 4 + g;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rk, (ap_lds)(k_to + (wave * (AP_CHUNKS / 2) + j) * 512), 16, min(p0 + r, n - 1) * (AP_D * 2) + 16 * (r16 ^ (r & 15)), 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < AP_CHUNKS / 2; j++) {
            const int r = (wave * (AP_CHUNKS / 2) + j) * 4 + g;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rv, (ap_lds)(v_to + (wave * (AP_CHUNKS / 2) + j) * 512), 16, min(p0 + r, n - 1) * (AP_D * 2) + 16 * r16, 0, 0, 0);
        }
    };
    request(std::integral_constant<int, 0>{}, 0);
    half8_t q8[QT][4];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        const half_t *p = q + ((int64_t)b * n + min(q0 + 16 * t + r16, n - 1)) * ldq + head * AP_D + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; c++) q8[t][c] = *reinterpret_cast<const half8_t *>(p + 32 * c);
    }

    const float scale2 = 0.08838834764831845f * 1.4426950408889634f;    // 1 / sqrt(128) * log2(e): the softmax runs in base 2
    float m[QT], l[QT];                          // of query r16 of a tile; l: the fp32 sum of the weights, before any is rounded, over this lane's positions
    float4_t acc[QT][8];
#pragma unroll
    for (int t = 0; t < QT; t++) {
        m[t] = -INFINITY;
        l[t] = 0.f;
#pragma unroll
        for (int j = 0; j < 8; j++) acc[t][j] = (float4_t)0.f;
    }
    // a stage: positions p0 .. p0 + 63
    constexpr int A = AP_P / 16;
    auto step = [&](const half_t *sk, const half_t *sv, int p0) __attribute__((always_inline)) {     // (a call would keep the sums in memory)
        float4_t s[QT][A];                        // [query tile][position tile]
#pragma unroll
        for (int a = 0; a < A; a++) {
            half8_t k8[4];
#pragma unroll
            for (int c = 0; c < 4; c++) k8[c] = *reinterpret_cast<const half8_t *>(sk + (16 * a + r16) * AP_D + 8 * ((4 * c + g) ^ r16));
#pragma unroll
            for (int t = 0; t < QT; t++) s[t][a] = (float4_t)0.f;
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int t = 0; t < QT; t++) s[t][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[c], q8[t][c], s[t][a], 0, 0, 0);
        }
        half8_t v8[8];
        auto fetch_v = [&](int h) {
#pragma unroll
            for (int i = 0; i < 8; i++) v8[i] = *reinterpret_cast<const half8_t *>(sv + (32 * h + 16 * (i >> 2) + 4 * g + (i & 3)) * AP_D + 8 * r16);
        };
        fetch_v(0);                              // (arrives during the softmax)
        __builtin_amdgcn_sched_barrier(0);
        if (p0 + AP_P > q0) {                    // some of the positions are behind a query
#pragma unroll
            for (int t = 0; t < QT; t++)
#pragma unroll
                for (int a = 0; a < A; a++)
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (p0 + 16 * a + 4 * g + i > q0 + 16 * t + r16) s[t][a][i] = -INFINITY;
        }
        // 32 positions at a time the running maximum, the weights, their sum and what the older sums are to be multiplied by
        float r[A / 2][QT];
        half8_t p8[A / 2][QT];
#pragma unroll
        for (int h = 0; h < A / 2; h++)
#pragma unroll
            for (int t = 0; t < QT; t++) {
                float mx = s[t][2 * h][0];
#pragma unroll
                for (int i = 1; i < 8; i++) mx = fmaxf(mx, s[t][2 * h + (i >> 2)][i & 3]);
                mx = across<32>(across<16>(mx));
                const float mn = fmaxf(m[t], mx * scale2);
                r[h][t] = __builtin_amdgcn_exp2f(m[t] - mn);
                m[t] = mn;
                float sum[2];
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    const float p = __builtin_amdgcn_exp2f(s[t][2 * h + (i >> 2)][i & 3] * scale2 - mn);
                    sum[i & 1] = i < 2 ? p : sum[i & 1] + p;
                    p8[h][t][i] = (half_t)p;
                }
                l[t] = l[t] * r[h][t] + (sum[0] + sum[1]);
            }
#pragma unroll
        for (int h = 0; h < A / 2; h++) {
            if (h > 0 && p0 + 32 * h > q0) continue;      // (32 positions behind all of the queries: an infinity in their v must not make a NaN of a weight of zero)
            if (__any(r[h][0] != 1.f || r[h][QT - 1] != 1.f)) {
#pragma unroll
                for (int t = 0; t < QT; t++)
#pragma unroll
                    for (int j = 0; j < 8; j++) acc[t][j] *= r[h][t];
            }
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const half8_t v = {v8[0][j], v8[1][j], v8[2][j], v8[3][j], v8[4][j], v8[5][j], v8[6][j], v8[7][j]};
#pragma unroll
                for (int t = 0; t < QT; t++) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, p8[h][t], acc[t][j], 0, 0, 0);
            }
            if (h + 1 < A / 2) fetch_v(h + 1);
        }
    };
    auto walk = [&](auto stage, int st) {
        // this wave's requests for the stage have landed; behind the barrier everybody's have, and nobody reads the other stage any more
        __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if (st + 1 < stages) request(std::integral_constant<int, 1 - decltype(stage)::value>{}, (st + 1) * AP_P);
        const half_t *const sk = decltype(stage)::value ? sk1 : sk0, *const sv = decltype(stage)::value ? sv1 : sv0;
        if (mine && st * AP_P <= q0) step(sk, sv, st * AP_P);
    };
    for (int st = 0; st < stages; st += 2) {
        walk(std::integral_constant<int, 0>{}, st);
        if (st + 1 < stages) walk(std::integral_constant<int, 1>{}, st + 1);
    }
    if (!mine) return;
#pragma unroll
    for (int t = 0; t < QT; t++) {
        const float total = across<32, true>(across<16, true>(l[t]));
        const int qi = q0 + 16 * t + r16;
        if (qi >= n) continue;
        const float inv = 1.f / total;
        half_t *to = out + ((int64_t)b * n + qi) * row + head * AP_D;
#pragma unroll
        for (int i = 0; i < 4; i++) {            // row 4 g + i of product j is dimension 8 (4 g + i) + j
            half8_t o;
#pragma unroll
            for (int j = 0; j < 8; j++) o[j] = (half_t)(acc[t][j][i] * inv);
            *reinterpret_cast<half8_t *>(to + 8 * (4 * g + i)) = o;
        }
    }
}

}  // namespace

int bs_launch_attention_prefill(const half_t *q, const half_t *kcache, const half_t *vcache, half_t *out, int ldq, int B, int n, int heads,
                                int kv_heads, int max_len, hipStream_t s) {
    const int per = std::max(1, (1 << 24) / kv_heads - 1);      // sequences of a launch: a grid holds 2^32 threads along x
    const auto launch = [&](auto kernel, int queries) {
        const int64_t chunks = bs_cdiv((int64_t)(heads / kv_heads) * bs_cdiv(n, queries), AP_WAVES), y = chunks < 32768 ? chunks : 32768;
        if (chunks > INT32_MAX / AP_WAVES) return BS_ERR_SHAPE;
        for (int b = 0; b < B; b += per) {
            const dim3 grid((unsigned)(std::min(per, B - b) * kv_heads), (unsigned)y, (unsigned)bs_cdiv(chunks, y));
            const int64_t cache = (int64_t)b * kv_heads * max_len * AP_D;
            kernel<<<grid, AP_WAVES * 64, 0, s>>>(q + (int64_t)b * n * ldq, kcache + cache, vcache + cache, out + (int64_t)b * n * heads * AP_D, ldq, n, heads, kv_heads, max_len, (int)chunks);
        }
        return (int)BS_OK;
    };
    // 16 queries per wave while 32 would leave the chip few workgroups: the chain of a wave's stages is what such a call takes (us, 32 / 16 queries: 2 x 700 positions with 32
    // heads on 8 KV heads, 352 workgroups, 24.4 / 19.7; 1 x 1000 with 8 on 8 28.6 / 20.0; 2 x 800, 400, 27.8 / 24.2; 4 x 400, 416, 17.8 / 17.6, 3 x 700 with 24 on 24, 432, 26.0 / 24.6; but 8 x
    // 200, 448, 13.4 / 13.9, 2 x 900, 464, 30.1 / 30.3, 2 x 1000, 512, 33.7 / 35.5, 4 x 1500 with 64 on 16, 3008, 206 / 254).
    const int64_t wgs = (int64_t)B * kv_heads * bs_cdiv((int64_t)(heads / kv_heads) * bs_cdiv(n, 32), AP_WAVES);
    const int st = wgs <= 400 ? launch(attention_prefill_kernel<1>, 16) : launch(attention_prefill_kernel<2>, 32);
    if (st != BS_OK) return st;
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int bs_launch_rope_store(half_t *q, const half_t *k, const half_t *v, const half_t *cos, const half_t *sin, half_t *kcache,
                         half_t *vcache, int ldq, int ldkv, int B, int n, int heads, int kv_heads, int d, int max_len, hipStream_t s) {
    // 16-byte pieces where every row and half row starts on 16 bytes (the pointers do)
    auto *kernel = d % 16 == 0 && ldq % 8 == 0 && ldkv % 8 == 0 ? rope_store_kernel<8> : rope_store_kernel<1>;
    kernel<<<B * n, THREADS, 0, s>>>(q, k, v, cos, sin, kcache, vcache, ldq, ldkv, n, heads, kv_heads, d, max_len);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int bs_launch_silu_mul(const half_t *gate, const half_t *up, half_t *y, int T, int width, int ld, hipStream_t s) {
    for (int t = 0; t < T; t += 65535) {         // (the grid's second dimension)
        const dim3 grid((unsigned)bs_cdiv(width, THREADS * 8), (unsigned)(T - t < 65535 ? T - t : 65535));
        silu_mul_kernel<<<grid, THREADS, 0, s>>>(gate + (int64_t)t * ld, up + (int64_t)t * ld, y + (int64_t)t * width, width, ld);
    }
    BS_LAUNCH_CHECK();
    return BS_OK;
}
