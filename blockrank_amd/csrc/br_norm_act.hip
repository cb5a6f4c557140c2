// Two elementwise steps of the decoder layers around the attention, each in one pass over memory:
//   RMSNorm      y = w * (x * rsqrt(mean(x^2) + eps))   (transformers models/mistral/modeling_mistral.py,
//                MistralRMSNorm.forward; the same class in the Llama and Qwen2 model files) - there: a cast
//                to fp32, a power, a mean, an addition, a reciprocal square root, two multiplications and
//                a cast back, each a kernel over the (tokens, hidden) activations;
//   SiLU gate    y = silu(gate) * up                     (MistralMLP.forward: act_fn(gate_proj(x)) * up_proj(x)).
// The ranking forward of scripts/eval_attn.py:139-151 runs both in every decoder layer; at the Mistral-7B
// shape they take 17 % of the GPU time of a forward pass.  Rounding follows the model file's order: for bf16
// tensors the normalised value is rounded to bf16 before it is multiplied by the weight, silu(gate) is
// rounded before it is multiplied by up.
#include "br_common.h"

namespace {

struct BrNormParams {
    const void* x;
    const void* w;
    void* out;
    long long rows, sx, so;     // row strides in elements
    int hidden;
    float eps;
};

template <typename T> struct Vec16;
template <> struct Vec16<__bf16> { static constexpr int N = 8; };
template <> struct Vec16<float> { static constexpr int N = 4; };

// Pieces of 16 bytes.  NT: with the non-temporal hint - for tensors that will not be found in the caches when they are
// next asked for, so that they do not push out what will.
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
template <bool NT, typename T>
__device__ inline u32x4 get16(const T* p) {
    const u32x4* q = reinterpret_cast<const u32x4*>(p);
    if constexpr (NT) return __builtin_nontemporal_load(q);
    else return *q;
}
template <bool NT, typename T>
__device__ inline void put16(T* p, const float (&f)[Vec16<T>::N]) {
    u32x4 u;
    T* e = reinterpret_cast<T*>(&u);
#pragma unroll
    for (int i = 0; i < Vec16<T>::N; ++i) e[i] = (T)f[i];
    if constexpr (NT) __builtin_nontemporal_store(u, reinterpret_cast<u32x4*>(p));
    else *reinterpret_cast<u32x4*>(p) = u;
}
template <typename T>
__device__ inline void values16(const u32x4& u, float (&f)[Vec16<T>::N]) {
    const T* e = reinterpret_cast<const T*>(&u);
#pragma unroll
    for (int i = 0; i < Vec16<T>::N; ++i) f[i] = (float)e[i];
}

// W waves (1 or 4: a workgroup) per row; a lane keeps its C 16-byte pieces of the row in registers between the sum of
// squares and the scaling, so the row is read once.  A workgroup is done after its row: the grid is one workgroup per row
// (or four rows), which at rows of 8 KiB reaches 5.8 TB/s where a persistent grid of one wave per row reached 4.8 - and
// with the non-temporal hint 6.2 TB/s where input and output together are beyond the 256 MB that the last-level cache
// keeps (26 368 rows of 8 KiB: 90 -> 70 us); below that the hint costs 10 % (13 000 rows: 32 against 36 us).  With the
// residual addition in front, which writes x, and the one behind, which reads it again: 280 us with the hint, 294 without,
// 290 with it on the stores alone; with a projection of the result in between as well, 1291 us either way.
template <typename T, int W, int C, bool NT>
__global__ __launch_bounds__(256) void br_rmsnorm_kernel(BrNormParams p) {
    constexpr int V = Vec16<T>::N;
    __shared__ float red[4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int chunks = p.hidden / V;
    const long long row = W == 4 ? (long long)blockIdx.x : (long long)blockIdx.x * 4 + wave;
    if (W == 1 && row >= p.rows) return;
    const int first = W == 4 ? threadIdx.x : lane;
    const T* x = reinterpret_cast<const T*>(p.x) + row * p.sx;
    const T* w = reinterpret_cast<const T*>(p.w);
    u32x4 v[C], wv[C];
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int c = first + 64 * W * i, at = c < chunks ? c : 0;
        v[i] = get16<NT>(x + (long long)at * V);
        wv[i] = get16<false>(w + (long long)at * V);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < C; ++i) {
        float f[V];
        values16<T>(v[i], f);
        if (first + 64 * W * i < chunks) {
#pragma unroll
            for (int e = 0; e < V; ++e) ss += f[e] * f[e];
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off);
    if constexpr (W == 4) {
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        ss = red[0] + red[1] + red[2] + red[3];
    }
    const float r = 1.0f / sqrtf(ss * (1.0f / (float)p.hidden) + p.eps);
    T* o = reinterpret_cast<T*>(p.out) + row * p.so;
#pragma unroll
    for (int i = 0; i < C; ++i) {
        const int c = first + 64 * W * i;
        if (c >= chunks) continue;
        float f[V], g[V], y[V];
        values16<T>(v[i], f);
        values16<T>(wv[i], g);
#pragma unroll
        for (int e = 0; e < V; ++e) y[e] = g[e] * (float)(T)(f[e] * r);
        put16<NT>(o + (long long)c * V, y);
    }
}

// One 16-byte piece per thread, as many threads as there are pieces.  Three streams of which none is read twice: with the
// non-temporal hint on loads and stores 6.4 TB/s at 26 368 x 14 336 bf16 against 5.4 with four pieces per thread and plain
// accesses (417 -> 350 us; one piece per thread without the hint 386).  With the down projection that reads the result (us;
// with the hint, without it, on the loads alone): 26 368 rows 2712, 2749, 2746; 14 080 rows 1462, 1496, 1497; 3520 rows 338,
// 350, 336; 560 rows 100, 98, 99.  With the two projections that write the operands as well, 26 368 rows: 7076, 7098, 7095.
template <typename T>
__global__ __launch_bounds__(256) void br_silu_mul_kernel(const T* gate, const T* up, T* out, long long n16) {
    constexpr int V = Vec16<T>::N;
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n16) return;
    const u32x4 gv = get16<true>(gate + i * V), uv = get16<true>(up + i * V);
    float g[V], u[V], y[V];
    values16<T>(gv, g);
    values16<T>(uv, u);
#pragma unroll
    for (int e = 0; e < V; ++e) y[e] = (float)(T)(g[e] / (1.0f + __expf(-g[e]))) * u[e];
    put16<true>(out + i * V, y);
}

template <typename T, bool NT>
int launch_norm(const BrNormParams& p, hipStream_t stream) {
    const int chunks = p.hidden / Vec16<T>::N;
    const dim3 one((unsigned)((p.rows + 3) / 4)), four((unsigned)p.rows);
    // a wave per row while two pieces per lane hold it, a workgroup per row beyond
    if (chunks <= 64) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 1, 1, NT>), one, dim3(256), 0, stream, p);
    else if (chunks <= 128) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 1, 2, NT>), one, dim3(256), 0, stream, p);
    else if (chunks <= 256) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 4, 1, NT>), four, dim3(256), 0, stream, p);
    else if (chunks <= 512) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 4, 2, NT>), four, dim3(256), 0, stream, p);
    else if (chunks <= 1024) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 4, 4, NT>), four, dim3(256), 0, stream, p);
    else if (chunks <= 2048) hipLaunchKernelGGL((br_rmsnorm_kernel<T, 4, 8, NT>), four, dim3(256), 0, stream, p);
    else return -1;
    return 0;
}

}  // namespace

// dtype: 0 fp32, 1 bf16.  Returns -1 if the row is too long for the kernel (more than 2048 16-byte pieces).
int br_launch_rmsnorm(const void* x, const void* w, void* out, long long rows, int hidden, long long sx, long long so, float eps, int dtype,
                      hipStream_t stream) {
    // What the last-level cache holds (256 MB): a tensor of which nothing is left there when it is read again gains from
    // not being kept, a smaller one would lose.
    constexpr double kCacheBytes = 256e6;
    // (a launch's grid is limited to 2^32 threads, and a row takes 64 or 256 of them: more rows than that go in several)
    const size_t es = dtype == 0 ? 4 : 2;
    const long long kMaxRows = (1LL << 31) / (hidden * es / 16 <= 128 ? 64 : 256);
    const bool nt = 2.0 * (double)rows * hidden * es > kCacheBytes;
    for (long long r0 = 0; r0 < rows; r0 += kMaxRows) {
        BrNormParams p;
        p.x = static_cast<const char*>(x) + r0 * sx * es; p.w = w; p.out = static_cast<char*>(out) + r0 * so * es;
        p.rows = rows - r0 < kMaxRows ? rows - r0 : kMaxRows;
        p.sx = sx; p.so = so; p.hidden = hidden; p.eps = eps;
        const int rc = dtype == 0 ? (nt ? launch_norm<float, true>(p, stream) : launch_norm<float, false>(p, stream))
                                  : (nt ? launch_norm<__bf16, true>(p, stream) : launch_norm<__bf16, false>(p, stream));
        if (rc) return rc;
    }
    return 0;
}

void br_launch_silu_mul(const void* gate, const void* up, void* out, long long n, int dtype, hipStream_t stream) {
    const int V = dtype == 0 ? 4 : 8;
    constexpr long long kMax16 = 1LL << 30;             // pieces, a thread each, per launch: the grid is limited
    for (long long i0 = 0; i0 < n / V; i0 += kMax16) {
        const long long n16 = n / V - i0 < kMax16 ? n / V - i0 : kMax16, e0 = i0 * V;
        const dim3 grid((unsigned)((n16 + 255) / 256));
        if (dtype == 0)
            hipLaunchKernelGGL(br_silu_mul_kernel<float>, grid, dim3(256), 0, stream, static_cast<const float*>(gate) + e0,
                               static_cast<const float*>(up) + e0, static_cast<float*>(out) + e0, n16);
        else
            hipLaunchKernelGGL(br_silu_mul_kernel<__bf16>, grid, dim3(256), 0, stream, static_cast<const __bf16*>(gate) + e0,
                               static_cast<const __bf16*>(up) + e0, static_cast<__bf16*>(out) + e0, n16);
    }
}
