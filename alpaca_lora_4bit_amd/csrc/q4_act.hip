// silu(gate) * up of a gated MLP block above the decode sizes, forward and backward (HBM-bound): the two elementwise kernels of
// the block's forward (src/alpaca_lora_4bit/model_attn_mlp_patch.py:224-228) and the three of its backward in one pass each.
// The results have the bits of the separate kernels: the same fp32 expressions with the exact expf, and silu(gate), the product
// and, backward, the gradient of silu(gate) go to fp16 as they do on tensors between them.  Bytes moved per element: 6 instead of 10 forward, 10 instead of 18
// backward; 8 elements a thread, one 16-byte load per operand.  us forward / backward, separate kernels -> here, over operands that
// come from HBM: 200 x 11008 7.7 / 12.1 -> 5.4 / 7.8, 1024 x 11008 23.9 / 37.4 -> 15.6 / 24.0, 4096 x 13824 93.6 / 176 -> 60.7 / 105
// (5.6 and 5.4 TB/s); the exact exponential is 0.5 us of the first and nothing of the last.
#include "q4_common.hpp"

namespace q4 {

constexpr int kActThreads = 256;

template <int V>
struct Halves { half_t v[V]; };
template <int V>
__device__ __forceinline__ Halves<V> load_halves(const half_t* p, long i) {
    if constexpr (V == 8) return __builtin_bit_cast(Halves<8>, *reinterpret_cast<const uint4_t*>(p + 8 * i));
    else return Halves<1>{{p[i]}};
}
template <int V>
__device__ __forceinline__ void store_halves(half_t* p, long i, const Halves<V>& h) {
    if constexpr (V == 8) *reinterpret_cast<uint4_t*>(p + 8 * i) = __builtin_bit_cast(uint4_t, h);
    else p[i] = h.v[0];
}

template <int V>
__device__ __forceinline__ void silu_mul_item(const half_t* gate, const half_t* up, half_t* out, long i) {
    const Halves<V> g = load_halves<V>(gate, i), u = load_halves<V>(up, i);
    Halves<V> o;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const float x = (float)g.v[e];
        const half_t s = (half_t)(x / (1.0f + expf(-x)));
        o.v[e] = (half_t)((float)s * (float)u.v[e]);
    }
    store_halves<V>(out, i, o);
}
// 8 elements per thread, the last n % 8 one by one by the first threads
__global__ __launch_bounds__(kActThreads) void silu_mul_kernel(const half_t* __restrict__ gate, const half_t* __restrict__ up,
                                                               half_t* __restrict__ out, long n) {
    const long i = (long)blockIdx.x * kActThreads + threadIdx.x;
    if (i < n / 8) silu_mul_item<8>(gate, up, out, i);
    if (i < n % 8) silu_mul_item<1>(gate, up, out, n / 8 * 8 + i);
}

template <int V>
__device__ __forceinline__ void silu_mul_bwd_item(const half_t* dout, const half_t* gate, const half_t* up, half_t* dgate,
                                                  half_t* dup, long i) {
    const Halves<V> d = load_halves<V>(dout, i), g = load_halves<V>(gate, i), u = load_halves<V>(up, i);
    Halves<V> dg, du;
#pragma unroll
    for (int e = 0; e < V; ++e) {
        const float x = (float)g.v[e], dy = (float)d.v[e], den = 1.0f + expf(-x), sig = 1.0f / den;
        const half_t s = (half_t)(x / den);
        const half_t ds = (half_t)(dy * (float)u.v[e]);
        du.v[e] = (half_t)(dy * (float)s);
        dg.v[e] = (half_t)((float)ds * sig * fmaf(x, 1.0f - sig, 1.0f));
    }
    store_halves<V>(dgate, i, dg);
    store_halves<V>(dup, i, du);
}
__global__ __launch_bounds__(kActThreads) void silu_mul_bwd_kernel(const half_t* __restrict__ dout, const half_t* __restrict__ gate,
                                                                   const half_t* __restrict__ up, half_t* __restrict__ dgate,
                                                                   half_t* __restrict__ dup, long n) {
    const long i = (long)blockIdx.x * kActThreads + threadIdx.x;
    if (i < n / 8) silu_mul_bwd_item<8>(dout, gate, up, dgate, dup, i);
    if (i < n % 8) silu_mul_bwd_item<1>(dout, gate, up, dgate, dup, n / 8 * 8 + i);
}

inline dim3 act_grid(long n) { return dim3((unsigned)((n / 8 + kActThreads) / kActThreads)); }    // covers n / 8 and n % 8 < 8 threads

}  // namespace q4

extern "C" int q4_launch_silu_mul(const void* gate, const void* up, void* out, long n, hipStream_t stream) {
    using namespace q4;
    hipLaunchKernelGGL(silu_mul_kernel, act_grid(n), dim3(kActThreads), 0, stream, (const half_t*)gate, (const half_t*)up,
                       (half_t*)out, n);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}

extern "C" int q4_launch_silu_mul_bwd(const void* dout, const void* gate, const void* up, void* dgate, void* dup, long n,
                                      hipStream_t stream) {
    using namespace q4;
    hipLaunchKernelGGL(silu_mul_bwd_kernel, act_grid(n), dim3(kActThreads), 0, stream, (const half_t*)dout, (const half_t*)gate,
                       (const half_t*)up, (half_t*)dgate, (half_t*)dup, n);
    return hipGetLastError() == hipSuccess ? 0 : -4;
}
