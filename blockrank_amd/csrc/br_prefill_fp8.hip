// Block-sparse prefill attention with Q K^T in fp8 e4m3 and P V in bf16: the quantisation of K and the fp8
// instances of the prefill kernel (templates in br_prefill_mfma_impl.h).  Inputs stay bf16.
//
//   K   one scale per (block, kv head): br_quant_kernel reads the real tokens of a block, takes max |x| and writes
//       x / scale as e4m3 into caller-provided scratch on the same token axis, with scale the power of two that puts
//       the maximum into [128, 256) (e4m3 reaches 448; a power of two makes the division exact), and the scale into the
//       table the attention kernel reads.  K is the small operand (1/4 to 1/7 of Q's volume with grouped heads).
//   Q   never touched here: the attention kernel reads the bf16 rows it reads anyway and converts them in
//       registers, each query row with its own power-of-two scale (a lane owns a row, so the scale is a per-lane
//       factor of the softmax scale).
// The query block's items (the rows the document scores are read from) run on the bf16 Q and K: their
// logits, and so the scores, are those of the bf16 kernel.
#include "br_prefill_mfma_impl.h"

namespace {

struct BrQuantParams {
    const __bf16* k;
    const int* plan;
    unsigned char* k8;
    float* scales;       // [B][M][Nkv]: dequantisation scales
    long long sk_b, sk_h, sk_t;        // input strides (elements)
    long long k8_b, k8_h;              // output strides (bytes); token stride is D
    int B, Nkv, M;
};

__device__ inline void br_values8(const uint4& u, float (&x)[8]) {
    const unsigned w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        x[2 * j] = __uint_as_float(w[j] << 16);
        x[2 * j + 1] = __uint_as_float(w[j] & 0xffff0000u);
    }
}

// A workgroup per (block, kv head): the block's rows in registers, up to UNR 16-byte pieces per thread, all requested before the
// first is used; their maximum; the rows as e4m3.  Blocks of more rows than that (512 at head dim 128) are read twice.  The query
// block's keys are not quantised: only its own rows see them, and those are computed in bf16.
// Bound by the round trips from a kernel's start to its first rows and by the bytes: 4 x 51 blocks of 16 to 512 tokens, 4 kv
// heads (28 MB in, 14 out) 18.5 us, where the maxima of whole sequences in one kernel (17.4) and the values in another (9.0) took
// 26.4 and a launch; 256 or 1024 threads 19.6 and 19.0.
constexpr int kQuantThreads = 512;
__global__ __launch_bounds__(kQuantThreads) void br_quant_kernel(BrQuantParams p) {
    constexpr int UNR = 16, W = kQuantThreads / 64;
    __shared__ float s_red[W];
    const int b = blockIdx.x / (p.M - 1), m = blockIdx.x - b * (p.M - 1), bm = b * p.M + m, h = blockIdx.y, tid = threadIdx.x;
    const int L = p.plan[br_plan_off_len(p.B, p.M) + bm], t0 = p.plan[br_plan_off_tok(p.B, p.M) + bm];
    const __bf16* src = p.k + (long long)b * p.sk_b + (long long)h * p.sk_h + (long long)t0 * p.sk_t;
    constexpr int D = 128, c8 = D / 8;            // (the variant's only head dim)
    const int n = L * c8;
    uint4 u[UNR];
    auto load = [&](int i0) {
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int i = i0 + k * kQuantThreads;
            if (i < n) u[k] = *reinterpret_cast<const uint4*>(src + (long long)(i / c8) * p.sk_t + i % c8 * 8);
        }
    };
    float mx = 0.f;
    for (int i0 = tid; i0 < n; i0 += UNR * kQuantThreads) {
        load(i0);
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            if (i0 + k * kQuantThreads >= n) break;
            float x[8];
            br_values8(u[k], x);
#pragma unroll
            for (int j = 0; j < 8; ++j) mx = fmaxf(mx, fabsf(x[j]));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if ((tid & 63) == 0) s_red[tid >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < W; ++w) mx = fmaxf(mx, s_red[w]);
    // NaN never wins fmaxf; a non-finite maximum would make every scale useless, so keep it finite
    float sc, inv;
    br_pow2_scale(fminf(mx, 3.0e38f), sc, inv);
    if (tid == 0) p.scales[(long long)bm * p.Nkv + h] = sc;
    unsigned char* dst = p.k8 + (long long)b * p.k8_b + (long long)h * p.k8_h + (long long)t0 * D;
    for (int i0 = tid; i0 < n; i0 += UNR * kQuantThreads) {
        if (n > UNR * kQuantThreads) load(i0);
#pragma unroll
        for (int k = 0; k < UNR; ++k) {
            const int i = i0 + k * kQuantThreads;
            if (i >= n) break;
            float x[8];
            br_values8(u[k], x);
            int lo = 0, hi = 0;
#pragma unroll
            for (int j = 0; j < 8; ++j) x[j] *= inv;                 // below 256 in magnitude
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(x[0], x[1], lo, false);
            lo = __builtin_amdgcn_cvt_pk_fp8_f32(x[2], x[3], lo, true);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(x[4], x[5], hi, false);
            hi = __builtin_amdgcn_cvt_pk_fp8_f32(x[6], x[7], hi, true);
            *reinterpret_cast<int2*>(dst + (long long)i * 8) = make_int2(lo, hi);       // (rows of D bytes follow each other)
        }
    }
}

template <int D, int NW>
void launch8(const BrPrefillParams& p, int grid, hipStream_t stream) {
    hipLaunchKernelGGL((br_prefill_mfma_kernel<D, NW, true, true, false>), dim3(grid), dim3(NW * 64), 0, stream, p);
}

}  // namespace

// Quantise K of a bf16 request - all blocks but the query's - into k8 (same token axis, (heads, tokens, D) bytes per batch
// entry) and fill the scale table [B][M][Nkv].
void br_launch_quantize_fp8(const void* k, const int* plan, void* k8, float* scales, const long long* sk,
                            long long k8_b, long long k8_h, int B, int Nkv, int M, hipStream_t stream) {
    BrQuantParams p;
    p.k = static_cast<const __bf16*>(k); p.plan = plan;
    p.k8 = static_cast<unsigned char*>(k8); p.scales = scales;
    p.sk_b = sk[0]; p.sk_h = sk[1]; p.sk_t = sk[2];
    p.k8_b = k8_b; p.k8_h = k8_h;
    p.B = B; p.Nkv = Nkv; p.M = M;
    if (M > 1) hipLaunchKernelGGL(br_quant_kernel, dim3(B * (M - 1), Nkv), dim3(kQuantThreads), 0, stream, p);
}

// The prefill kernel with fp8 logits (p.k8: the quantised K, p.qk_scales: its scales) followed by
// the split merge (with the score reduction ``rank`` asks for, if any).  Returns 0 on success, -1 if (D, NW) has no
// instantiation (only D = 128 is built; nothing is launched then).
int br_launch_prefill_fp8qk(const BrPrefillParams& p, int D, int NW, int n_cu, int combine_grid, hipStream_t stream,
                            hipEvent_t ev_start, hipEvent_t ev_stop, const BrTileScoreParams* rank) {
    const int per_cu = NW <= 4 ? 2 : 1;
    const int grid = n_cu * per_cu;
    if (D != 128 || NW < 4 || NW > 8) return -1;
    if (ev_start) (void)hipEventRecord(ev_start, stream);
    switch (NW) {
        case 4: launch8<128, 4>(p, grid, stream); break;
        case 5: launch8<128, 5>(p, grid, stream); break;
        case 6: launch8<128, 6>(p, grid, stream); break;
        case 7: launch8<128, 7>(p, grid, stream); break;
        case 8: launch8<128, 8>(p, grid, stream); break;
        default: return -1;
    }
    if (ev_stop) (void)hipEventRecord(ev_stop, stream);
    br_launch_finish_scores<__bf16, 128>(p, NW, combine_grid, rank, stream);
    return 0;
}
