// Per-document relevance from the query block's attention, without materialising attention rows.
//
// Reference: compute_auxiliary_attention_loss(answer_ids=None, return_logits=True), losses.py:37-78,
// applied to the logits of blockrank_std_attention.py:233,259 (scaled q.k of chosen rows of the
// query block against every key).  For each (head, chosen row) the reference soft-maxes the logits
// over all document tokens jointly and sums the probabilities per document, then averages heads and
// rows and divides by the temperature.  Here:
//   br_doc_partial_kernel  one workgroup per (document, kv head group, sequence): logits of that
//                          document's real keys for every (head, row) of the group, reduced on the
//                          fly to (max, sum of exp) per (head, row, document);
//   br_doc_final_tiles_kernel  one workgroup per sequence: joint normalisation across documents, head /
//                          row reduction, temperature (br_score_tiles.h).
#include "br_mma.h"
#include "br_score_tiles.h"

namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

struct BrScoreParams {
    const void* q;
    const void* k;
    const int* plan;        // only the block table part is used
    const int* rows;        // (B, R) positions of the chosen rows inside the query block, 0..H-1
    float* part;            // (B, Nq, R, docs, 2): max (log2 domain) and sum of exp per document
    long long sq_b, sq_h, sq_t;
    long long sk_b, sk_h, sk_t;
    int B, Nq, Nkv, M, H, R, T;
    float scale_log2;       // softmax scale * log2(e)
};

// (max, sum of 2^(logit - max)) of a document's keys for every (query head of the kv head, chosen row): one workgroup per
// (document, kv head and group of 32 (head, row) pairs, sequence).  A wave takes 32 keys at a time: A = the keys (row = key,
// each lane the pieces of its key's row), B = the pairs' query rows, so that a lane ends up with one pair and 16 of the
// keys, and the reduction is in its registers but for one exchange with the other half of the keys.
// Bandwidth: reads the documents' K once (seven heads of 16 rows: four times, from cache).  B=8, 20 documents of 96-224
// tokens, 32/8 heads, 2 rows (54 MB of K): 13.7 us, 67 us with a key per thread on the vector ALU.
template <typename T, int D>
__global__ __launch_bounds__(256) void br_doc_partial_kernel(BrScoreParams p) {
    constexpr int NP = D / BrPiece<T>::STEP;
    __shared__ float red_m[4][32], red_s[4][32];
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.T);
    const int doc = blockIdx.x, b = blockIdx.z, docs = p.M - 2;
    const int G = p.Nq / p.Nkv, pairs = G * p.R, groups = (pairs + 31) / 32;
    const int kvh = blockIdx.y / groups, p0 = (blockIdx.y - kvh * groups) * 32;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const int bm = b * p.M, mq = bm + p.M - 1;
    const int len = pv.len[bm + doc + 1], tok = pv.tok[bm + doc + 1];
    const int st_q = pv.start[mq], len_q = pv.len[mq], tok_q = pv.tok[mq];
    const int pair = p0 + ln < pairs ? p0 + ln : pairs - 1;
    const int h = pair / p.R, r = pair - h * p.R, pos = p.rows[b * p.R + r];
    const bool row_ok = pos >= st_q && pos < st_q + len_q;
    const T* kbase = reinterpret_cast<const T*>(p.k) + (long long)b * p.sk_b + (long long)kvh * p.sk_h + (long long)tok * p.sk_t + lh * BrPiece<T>::N;
    // (of q only rows that are real tokens of the query block may be read: a pair without one takes another's place in no
    // result, its operand is zero)
    uint4 qf[NP];
    {
        const T* qrow = reinterpret_cast<const T*>(p.q) + (long long)b * p.sq_b + (long long)(kvh * G + h) * p.sq_h +
                        (long long)(tok_q + (row_ok ? pos - st_q : 0)) * p.sq_t + lh * BrPiece<T>::N;
#pragma unroll
        for (int c = 0; c < NP; ++c) qf[c] = row_ok ? *reinterpret_cast<const uint4*>(qrow + c * BrPiece<T>::STEP) : uint4{0u, 0u, 0u, 0u};
    }
    float mx = -INFINITY, sm = 0.f;
    for (int k0 = wave * 32; k0 < len; k0 += 128) {
        const int key = k0 + ln < len ? k0 + ln : len - 1;       // keys past the end repeat the last one and are masked
        const T* krow = kbase + (long long)key * p.sk_t;
        uint4 kf[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) kf[c] = *reinterpret_cast<const uint4*>(krow + c * BrPiece<T>::STEP);
        f32x16 s;
#pragma unroll
        for (int v = 0; v < 16; ++v) s[v] = 0.f;
#pragma unroll
        for (int c = 0; c < NP; ++c) s = BrPiece<T>::mma(kf[c], qf[c], s);
        float mn = mx;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            s[v] = k0 + 8 * (v >> 2) + 4 * lh + (v & 3) < len ? s[v] * p.scale_log2 : -INFINITY;
            mn = fmaxf(mn, s[v]);
        }
        const float sub = mn == -INFINITY ? 0.f : mn;
        sm *= __builtin_amdgcn_exp2f(mx - sub);
#pragma unroll
        for (int v = 0; v < 16; ++v) sm += __builtin_amdgcn_exp2f(s[v] - sub);
        mx = mn;
    }
    auto join = [&](float m2, float s2) {
        const float mn = fmaxf(mx, m2), sub = mn == -INFINITY ? 0.f : mn;
        sm = sm * __builtin_amdgcn_exp2f(mx - sub) + s2 * __builtin_amdgcn_exp2f(m2 - sub);
        mx = mn;
    };
    join(__shfl_xor(mx, 32), __shfl_xor(sm, 32));
    if (lh == 0) {
        red_m[wave][ln] = mx;
        red_s[wave][ln] = sm;
    }
    __syncthreads();
    if (threadIdx.x < 32 && p0 + ln < pairs) {
        for (int w = 1; w < 4; ++w) join(red_m[w][ln], red_s[w][ln]);
        // a padded query row sees nothing; the reduction turns this into the uniform answer
        const float2 ms = row_ok ? make_float2(mx, sm) : make_float2(-INFINITY, 0.f);
        *reinterpret_cast<float2*>(p.part + ((((long long)b * p.Nq + kvh * G + h) * p.R + r) * docs + doc) * 2) = ms;
    }
}

template <int PATH>
__global__ __launch_bounds__(1024) void br_doc_final_tiles_kernel(BrTileScoreParams p, int nwaves) {
    extern __shared__ float dyn[];
    br_doc_final_tiles_body<PATH>(p, blockIdx.x, 0, dyn, nwaves);
}

void launch_final(const BrTileScoreParams& p, int tiles, hipStream_t stream) {
    const int docs = p.M - 2, path = br_doc_final_path(docs, tiles), nwaves = br_doc_final_waves(docs, path);
    const size_t lds = br_doc_final_lds(docs, path);
    if (path == 0) hipLaunchKernelGGL((br_doc_final_tiles_kernel<0>), dim3(p.B), dim3(1024), lds, stream, p, nwaves);
    else if (path == 1) hipLaunchKernelGGL((br_doc_final_tiles_kernel<1>), dim3(p.B), dim3(1024), lds, stream, p, nwaves);
    else hipLaunchKernelGGL((br_doc_final_tiles_kernel<2>), dim3(p.B), dim3(1024), lds, stream, p, nwaves);
}

}  // namespace

// dtype: 0 fp32, 1 bf16, 2 fp16
void br_launch_doc_scores(const void* q, const void* k, const int* plan, const int* rows, float* part, float* scores,
                          float* probs, const long long* sq, const long long* sk, int B, int Nq, int Nkv, int M, int H, int D,
                          int R, int T, float scale, float out_scale, int dtype, hipStream_t stream) {
    BrScoreParams p;
    p.q = q; p.k = k; p.plan = plan; p.rows = rows; p.part = part;
    p.sq_b = sq[0]; p.sq_h = sq[1]; p.sq_t = sq[2];
    p.sk_b = sk[0]; p.sk_h = sk[1]; p.sk_t = sk[2];
    p.B = B; p.Nq = Nq; p.Nkv = Nkv; p.M = M; p.H = H; p.R = R; p.T = T;
    p.scale_log2 = scale * 1.4426950408889634f;
    const dim3 grid(M - 2, Nkv * ((Nq / Nkv * R + 31) / 32), B);
    if (dtype == 0 && D == 64) hipLaunchKernelGGL((br_doc_partial_kernel<float, 64>), grid, dim3(256), 0, stream, p);
    else if (dtype == 0) hipLaunchKernelGGL((br_doc_partial_kernel<float, 128>), grid, dim3(256), 0, stream, p);
    else if (dtype == 1 && D == 64) hipLaunchKernelGGL((br_doc_partial_kernel<__bf16, 64>), grid, dim3(256), 0, stream, p);
    else if (dtype == 1) hipLaunchKernelGGL((br_doc_partial_kernel<__bf16, 128>), grid, dim3(256), 0, stream, p);
    else if (D == 64) hipLaunchKernelGGL((br_doc_partial_kernel<_Float16, 64>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((br_doc_partial_kernel<_Float16, 128>), grid, dim3(256), 0, stream, p);
    BrTileScoreParams t;
    t.part = part; t.plan = plan; t.rows = rows; t.scores = scores; t.probs = probs;
    t.B = B; t.Nq = Nq; t.M = M; t.H = H; t.R = R; t.Rw = R; t.out_scale = out_scale; t.per_doc = 1; t.count = nullptr; t.sums = nullptr; t.chunks = 1;
    launch_final(t, M - 2, stream);
}

void br_launch_doc_scores_tiles(const float* part, const int* plan, const int* rows, float* scores, float* probs, int B, int Nq,
                                int M, int H, int R, int Rw, float out_scale, hipStream_t stream) {
    BrTileScoreParams p;
    p.part = part; p.plan = plan; p.rows = rows; p.scores = scores; p.probs = probs;
    p.B = B; p.Nq = Nq; p.M = M; p.H = H; p.R = R; p.Rw = Rw; p.out_scale = out_scale; p.per_doc = 0; p.count = nullptr; p.sums = nullptr; p.chunks = 1;
    launch_final(p, br_plan_tps(M, H), stream);
}
