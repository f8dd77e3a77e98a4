// What sits between the compressed linears of a decoder layer when a whole prompt goes through it: rotary embedding with the
// store of k and v to the cache, the SiLU product of the MLP, and a residual sum with the RMSNorm that follows it.  Each is one
// pass over its operands, bound by memory; as framework operations they were eleven passes and launches for the rotation and
// the two cache copies, two for the SiLU product and two for the sum and the norm, with every step rounded to fp16.  Here
// each result is computed in fp32 and rounded once.
#include "common.h"

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

// Causal attention of a whole prompt over the cache that rope_store_kernel has filled.  A wave takes 32 queries of one head and
// walks the positions up to its last query 32 at a time with a running (max, sum, weighted v); the four waves of a workgroup are
// four neighbouring heads, which mostly share a KV head and then find each other's rows in the L1.  The operands lie as in the
// decode step's attention (decode_step.hip): scores S[position, query] = K q, output O[dim, query] += V^T P, on 16x16x32
// products whose lane layouts fit without any shuffle - a lane of the scores holds four positions of one query in each of
// the two tiles of 16 positions, which are the eight k slots of the output product, and V is used as loaded, product j taking
// half j of a lane's 16 bytes.  No LDS, no barrier.  The rows of a step come from the L2 while the last step is multiplied: K is
// requested behind the scores, V behind the output product.
// What bounds it: the rows (16 KB a step and wave) and, with few waves, the chain of a step.  torch's attention, all sequences in
// one call / this, us: 2 x 700 queries with 32 heads on 8 KV heads 76 / 40, 4 x 300 53 / 21, 100 15 / 8, 4000 476 / 306,
// 4 x 1500 with 64 on 16 651 / 342 (430 TFLOP/s).  16 queries per wave read the rows twice as often: 55 on the first, 639 on the last.
constexpr int AP_D = 128, AP_Q = 32, AP_WAVES = 4;

__global__ __launch_bounds__(AP_WAVES * 64, 2) void attention_prefill_kernel(const half_t *__restrict__ q, const half_t *__restrict__ kcache,
                                                                             const half_t *__restrict__ vcache, half_t *__restrict__ out,
                                                                             int ldq, int n, int heads, int kv_heads, int max_len) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
    const int quads = (heads + AP_WAVES - 1) / AP_WAVES, b = blockIdx.x / quads, head = (blockIdx.x % quads) * AP_WAVES + wave;
    if (head >= heads) return;
    const int q0 = (int)(gridDim.y - 1 - blockIdx.y) * AP_Q;             // the longest rows first
    const int hk = head / (heads / kv_heads);
    const int64_t row = (int64_t)heads * AP_D;
    const half_t *kc = kcache + ((int64_t)b * kv_heads + hk) * max_len * AP_D, *vc = vcache + ((int64_t)b * kv_heads + hk) * max_len * AP_D;

    half8_t k8[2][4], v8[8], q8[2][4];
    auto fetch_k = [&](int p0) {                 // (rows past the last are the last again; their scores are masked)
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const half_t *p = kc + (int64_t)min(p0 + 16 * a + r16, n - 1) * AP_D + 8 * g;
#pragma unroll
            for (int c = 0; c < 4; c++) k8[a][c] = *reinterpret_cast<const half8_t *>(p + 32 * c);
        }
    };
    auto fetch_v = [&](int p0) {
#pragma unroll
        for (int i = 0; i < 8; i++)
            v8[i] = *reinterpret_cast<const half8_t *>(vc + (int64_t)min(p0 + 16 * (i >> 2) + 4 * g + (i & 3), n - 1) * AP_D + 8 * r16);
    };
    fetch_k(0);
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const half_t *p = q + ((int64_t)b * n + min(q0 + 16 * t + r16, n - 1)) * ldq + head * AP_D + 8 * g;
#pragma unroll
        for (int c = 0; c < 4; c++) q8[t][c] = *reinterpret_cast<const half8_t *>(p + 32 * c);
    }
    fetch_v(0);

    const float scale2 = 0.08838834764831845f * 1.4426950408889634f;    // 1 / sqrt(128) * log2(e): the softmax runs in base 2
    float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.f, 0.f};              // of query r16 of a tile; the sum over this lane's positions
    float4_t acc[2][8];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[t][j] = (float4_t)0.f;
    for (int p0 = 0; p0 <= q0; p0 += AP_Q) {
        float4_t s[2][2];                        // [query tile][position tile]
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int a = 0; a < 2; a++) {
                s[t][a] = (float4_t)0.f;
#pragma unroll
                for (int c = 0; c < 4; c++) s[t][a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(k8[a][c], q8[t][c], s[t][a], 0, 0, 0);
            }
        if (p0 < q0) fetch_k(p0 + AP_Q);
        half8_t p8[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            float p[8], mx = -INFINITY;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                p[i] = s[t][i >> 2][i & 3] * scale2;
                if (p0 == q0 && 16 * (i >> 2) + 4 * g + (i & 3) > 16 * t + r16) p[i] = -INFINITY;      // behind the query
                mx = fmaxf(mx, p[i]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
            mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
            const float mn = fmaxf(m[t], mx), r = __builtin_amdgcn_exp2f(m[t] - mn);
            m[t] = mn;
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                p[i] = __builtin_amdgcn_exp2f(p[i] - mn);
                sum += p[i];
                p8[t][i] = (half_t)p[i];
            }
            l[t] = l[t] * r + sum;
            if (__any(r != 1.f)) {
#pragma unroll
                for (int j = 0; j < 8; j++) acc[t][j] *= r;
            }
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const half8_t v = {v8[0][j], v8[1][j], v8[2][j], v8[3][j], v8[4][j], v8[5][j], v8[6][j], v8[7][j]};
#pragma unroll
            for (int t = 0; t < 2; t++) acc[t][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(v, p8[t], acc[t][j], 0, 0, 0);
        }
        if (p0 < q0) fetch_v(p0 + AP_Q);
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        l[t] += __shfl_xor(l[t], 16, 64);
        l[t] += __shfl_xor(l[t], 32, 64);
        const int qi = q0 + 16 * t + r16;
        if (qi >= n) continue;
        const float inv = 1.f / l[t];
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
    const dim3 grid((unsigned)(B * bs_cdiv(heads, AP_WAVES)), (unsigned)bs_cdiv(n, AP_Q));
    attention_prefill_kernel<<<grid, AP_WAVES * 64, 0, s>>>(q, kcache, vcache, out, ldq, n, heads, kv_heads, max_len);
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
