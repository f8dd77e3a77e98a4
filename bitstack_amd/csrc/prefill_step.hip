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
                                                             half_t *__restrict__ vcache, int n, int heads, int kv_heads, int d,
                                                             int max_len) {
    typedef half_t vec_t __attribute__((ext_vector_type(V)));
    const int token = blockIdx.x, b = token / n, pos = token % n, d2 = d / 2;
    const int per = d2 / V, qi = heads * per, ki = kv_heads * per;               // items of q and of k; v has 2 * ki
    q += (int64_t)token * heads * d;
    k += (int64_t)token * kv_heads * d;
    v += (int64_t)token * kv_heads * d;
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

// y = silu(gate) * up; eight values per thread.  y may be gate or up: a thread reads what it overwrites.  1400 x 14336: 36 us as
// two operations, 18.9 now (120 MB: 6.4 TB/s).
__global__ __launch_bounds__(THREADS) void silu_mul_kernel(const half_t *gate, const half_t *up, half_t *y, int64_t count) {
    const int64_t i = ((int64_t)blockIdx.x * THREADS + threadIdx.x) * 8;
    auto one = [](float a, float b) { return (half_t)(a / (1.f + __expf(-a)) * b); };
    if (i + 8 <= count) {
        const half8_t a = *reinterpret_cast<const half8_t *>(gate + i), b = *reinterpret_cast<const half8_t *>(up + i);
        half8_t o;
#pragma unroll
        for (int e = 0; e < 8; e++) o[e] = one((float)a[e], (float)b[e]);
        *reinterpret_cast<half8_t *>(y + i) = o;
    } else {
        for (int64_t j = i; j < count; j++) y[j] = one((float)gate[j], (float)up[j]);
    }
}

}  // namespace

int bs_launch_rope_store(half_t *q, const half_t *k, const half_t *v, const half_t *cos, const half_t *sin, half_t *kcache,
                         half_t *vcache, int B, int n, int heads, int kv_heads, int d, int max_len, hipStream_t s) {
    // 16-byte pieces where every row and half row starts on 16 bytes (the pointers do)
    auto *kernel = d % 16 == 0 ? rope_store_kernel<8> : rope_store_kernel<1>;
    kernel<<<B * n, THREADS, 0, s>>>(q, k, v, cos, sin, kcache, vcache, n, heads, kv_heads, d, max_len);
    BS_LAUNCH_CHECK();
    return BS_OK;
}

int bs_launch_silu_mul(const half_t *gate, const half_t *up, half_t *y, int64_t count, hipStream_t s) {
    silu_mul_kernel<<<bs_cdiv(count, THREADS * 8), THREADS, 0, s>>>(gate, up, y, count);
    BS_LAUNCH_CHECK();
    return BS_OK;
}
