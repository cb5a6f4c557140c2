// Rotary position embedding of Q and K in one pass: the step in front of the attention kernel.
// out = x * cos + rotate_half(x) * sin with rotate_half(x) = (-x[D/2:], x[:D/2]) - the Hugging Face
// convention (transformers models/mistral/modeling_mistral.py: rotate_half, apply_rotary_pos_emb), which
// the models BlockRank ranks with apply to the projected Q and K before every attention call.  There it
// is four multiplications, a negation, a concatenation and two additions per tensor, each a pass over
// memory; here Q and K are read once and written once, straight into the (batch, token, head, dim)
// layout the attention kernels address through strides.  Arithmetic in fp32, one rounding at the end.
#include "br_common.h"

namespace {

struct BrRopeParams {
    const void* q;
    const void* k;
    const void* cos;
    const void* sin;
    void* q_out;
    void* k_out;
    long long sq_b, sq_h, sq_t;     // element strides of q (batch, head, token); the last dim is dense
    long long sk_b, sk_h, sk_t;
    long long sc_b, sc_t;           // of cos and sin (batch, token); a batch stride of 0 broadcasts
    int B, Nq, Nkv, S, D;
    long long token0;               // first token (of B * S) of this launch
    int tokens;                     // and how many
};

template <typename T> struct Vec16;
template <> struct Vec16<__bf16> { static constexpr int N = 8; };
template <> struct Vec16<_Float16> { static constexpr int N = 8; };
template <> struct Vec16<float> { static constexpr int N = 4; };

template <typename T>
__device__ inline void load16(const T* p, float (&f)[Vec16<T>::N]) {
    const uint4 u = *reinterpret_cast<const uint4*>(p);
    const T* e = reinterpret_cast<const T*>(&u);
#pragma unroll
    for (int i = 0; i < Vec16<T>::N; ++i) f[i] = (float)e[i];
}
template <typename T>
__device__ inline void store16(T* p, const float (&f)[Vec16<T>::N]) {
    uint4 u;
    T* e = reinterpret_cast<T*>(&u);
#pragma unroll
    for (int i = 0; i < Vec16<T>::N; ++i) e[i] = (T)f[i];
    *reinterpret_cast<uint4*>(p) = u;
}

// One thread: one 16-byte piece of the first half of a head's row and the matching piece of the second half; as many
// threads as there are such pairs (a grid of at most 32 workgroups per CU that loops was 2 % slower at 26 368 tokens, 40
// heads of 128: 76 us, 7.1 TB/s of q, k and their results).
template <typename T>
__global__ __launch_bounds__(256) void br_rope_kernel(BrRopeParams p) {
    constexpr int V = Vec16<T>::N;
    const unsigned half = p.D / 2, ppr = half / V;   // pieces per half row
    const unsigned NH = p.Nq + p.Nkv;
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < (unsigned)p.tokens * NH * ppr) {
        const int c = (int)(i % ppr);
        const unsigned r = i / ppr;
        const int h = (int)(r % NH);
        const long long bt = p.token0 + r / NH;
        const int b = (int)(bt / p.S), t = (int)(bt - (long long)b * p.S);
        const bool is_q = h < p.Nq;
        const int hh = is_q ? h : h - p.Nq;
        const T* x = is_q ? reinterpret_cast<const T*>(p.q) + b * p.sq_b + hh * p.sq_h + t * p.sq_t
                          : reinterpret_cast<const T*>(p.k) + b * p.sk_b + hh * p.sk_h + t * p.sk_t;
        T* o = is_q ? reinterpret_cast<T*>(p.q_out) + (((long long)b * p.S + t) * p.Nq + hh) * p.D
                    : reinterpret_cast<T*>(p.k_out) + (((long long)b * p.S + t) * p.Nkv + hh) * p.D;
        const T* cs = reinterpret_cast<const T*>(p.cos) + b * p.sc_b + t * p.sc_t;
        const T* sn = reinterpret_cast<const T*>(p.sin) + b * p.sc_b + t * p.sc_t;
        float x1[V], x2[V], c1[V], c2[V], s1[V], s2[V], o1[V], o2[V];
        load16(x + c * V, x1);
        load16(x + half + c * V, x2);
        load16(cs + c * V, c1);
        load16(cs + half + c * V, c2);
        load16(sn + c * V, s1);
        load16(sn + half + c * V, s2);
#pragma unroll
        for (int e = 0; e < V; ++e) {
            o1[e] = x1[e] * c1[e] - x2[e] * s1[e];
            o2[e] = x2[e] * c2[e] + x1[e] * s2[e];
        }
        store16(o + c * V, o1);
        store16(o + half + c * V, o2);
    }
}

}  // namespace

// dtype: 0 fp32, 1 bf16, 2 fp16 (q, k, cos, sin and the outputs alike).
int br_launch_rope(const void* q, const void* k, const void* cos, const void* sin, void* q_out, void* k_out, int B, int Nq, int Nkv, int S,
                   int D, const long long* sq, const long long* sk, const long long* sc, int dtype, hipStream_t stream) {
    BrRopeParams p;
    p.q = q; p.k = k; p.cos = cos; p.sin = sin; p.q_out = q_out; p.k_out = k_out;
    p.sq_b = sq[0]; p.sq_h = sq[1]; p.sq_t = sq[2];
    p.sk_b = sk[0]; p.sk_h = sk[1]; p.sk_t = sk[2];
    p.sc_b = sc[0]; p.sc_t = sc[1];
    p.B = B; p.Nq = Nq; p.Nkv = Nkv; p.S = S; p.D = D;
    const int V = dtype == 0 ? 4 : 8;
    const int per_token = (Nq + Nkv) * (D / 2 / V);
    const long long most = (1LL << 30) / per_token;          // tokens per launch: its indices are 32-bit
    for (long long t0 = 0; t0 < (long long)B * S; t0 += most) {
        p.token0 = t0;
        p.tokens = (int)((long long)B * S - t0 < most ? (long long)B * S - t0 : most);
        const dim3 grid((unsigned)(((long long)p.tokens * per_token + 255) / 256));
        if (dtype == 0) hipLaunchKernelGGL(br_rope_kernel<float>, grid, dim3(256), 0, stream, p);
        else if (dtype == 1) hipLaunchKernelGGL(br_rope_kernel<__bf16>, grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL(br_rope_kernel<_Float16>, grid, dim3(256), 0, stream, p);
    }
    return 0;
}
