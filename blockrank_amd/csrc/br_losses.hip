// The steps of compute_auxiliary_attention_loss (src/blockrank/losses.py:37-93) that follow the attention, each as one
// launch instead of the dozens of elementwise ones of the torch expressions: which rows are scored, the per-document
// scores of a dense logits tensor (training), the InfoNCE loss on them, and the gradients of the two.  All of them work
// on a few kilobytes to a few megabytes: what they cost is launches, so there is one workgroup per independent row.
#include "br_common.h"

namespace {

__device__ inline float wave_max(float x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
    return x;
}
__device__ inline float wave_sum(float x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    return x;
}
// e^(x - m), with -inf - (-inf) counted as an empty sum (a maximum of -inf may also be that of NaNs alone, which stay NaN)
__device__ inline float exp_below(float x, float m) { return x == -INFINITY && m == -INFINITY ? 0.f : expf(x - m); }

// rows[b] = {i - 1, i}, i the first of the last h1 labels of sequence b that is above -100 (0 if there is none, as argmax
// gives it); flags[0]: every row is >= 0; flags[1]: every row equals guess (0 without one).  A wave per sequence.
__global__ __launch_bounds__(256) void br_bracket_rows_kernel(const int64_t* __restrict__ labels, int64_t stride, int B, int S, int h1,
                                                              const int* __restrict__ guess, int64_t* __restrict__ rows, int* __restrict__ pos,
                                                              int pos_offset, int* flags) {
    __shared__ int s_bad, s_other;
    if (threadIdx.x == 0) s_bad = s_other = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
    for (int b = threadIdx.x >> 6; b < B; b += 4) {
        const int64_t* last = labels + b * stride + (S - h1);
        int first = 0x7fffffff;
        for (int j = lane; j < h1; j += 64)
            if (last[j] > -100 && j < first) first = j;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const int y = __shfl_xor(first, o);
            first = y < first ? y : first;
        }
        if (first == 0x7fffffff) first = 0;
        if (lane == 0) {
            if (rows) {
                rows[2 * b] = first - 1;
                rows[2 * b + 1] = first;
            }
            if (pos) {
                pos[2 * b] = first - 1 + pos_offset;
                pos[2 * b + 1] = first + pos_offset;
            }
            if (first < 1) atomicOr(&s_bad, 1);
            if (guess && (guess[2 * b] != first - 1 || guess[2 * b + 1] != first)) atomicOr(&s_other, 1);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        flags[0] = s_bad == 0;
        flags[1] = guess && s_other == 0;
        __threadfence_system();
    }
}

struct BrDenseScoreParams {
    const float* x;         // (B, N, h1, M*H) logits
    const int64_t* rows;    // (B, R) indices into the h1 rows, taken modulo h1
    float* pdoc;            // (B, N, R, docs) per-document probabilities
    float* stat;            // (B, N, R, 2): maximum, 1 / sum of exponentials
    const float* g;         // (B, docs) gradient of the scores
    float* dx;              // (B, N, h1, M*H)
    int B, N, h1, M, H, R;
    float out_scale;
};

// An index outside 0..h1-1 wraps around, as torch's take_along_dim takes it.
__device__ inline int row_of(const BrDenseScoreParams& p, int b, int r) {
    const int64_t i = p.rows[(long long)b * p.R + r];
    if (i >= 0 && i < p.h1) return (int)i;
    const int m = (int)(i % p.h1);
    return m < 0 ? m + p.h1 : m;
}

// One workgroup per (sequence, head, row): softmax over the document slots, summed per document.  A wave takes a
// document at a time and keeps its (maximum, sum); the joint maximum and sum follow from those.  Latency-bound: a document's
// slots are requested together (512 of them stay in registers for the sum), and as many documents as there are waves side by
// side (12 documents of 250 slots, 128 rows: 5 us; 9.3 with four waves that read every document twice).
__global__ __launch_bounds__(1024) void br_dense_doc_probs_kernel(BrDenseScoreParams p) {
    extern __shared__ float dyn[];                         // [docs] maxima, [docs] sums
    __shared__ float red[16];
    const int docs = p.M - 2, b = blockIdx.y, n = blockIdx.x / p.R, r = blockIdx.x - n * p.R;
    float* dm = dyn;
    float* dsum = dyn + docs;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int row = row_of(p, b, r);
    const float* x = p.x + (((long long)b * p.N + n) * p.h1 + row) * p.M * p.H + p.H;
    constexpr int K = 8;
    for (int d = wave; d < docs; d += waves) {
        const float* xd = x + (long long)d * p.H;
        float v[K], m = -INFINITY;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int j = lane + 64 * k;
            v[k] = j < p.H ? xd[j] : -INFINITY;
        }
#pragma unroll
        for (int k = 0; k < K; ++k) m = fmaxf(m, v[k]);
        for (int j = lane + 64 * K; j < p.H; j += 64) m = fmaxf(m, xd[j]);
        m = wave_max(m);
        float s = 0.f;
#pragma unroll
        for (int k = 0; k < K; ++k)
            if (lane + 64 * k < p.H) s += exp_below(v[k], m);
        for (int j = lane + 64 * K; j < p.H; j += 64) s += exp_below(xd[j], m);
        s = wave_sum(s);
        if (lane == 0) {
            dm[d] = m;
            dsum[d] = s;
        }
    }
    __syncthreads();
    float m = -INFINITY;
    for (int d = threadIdx.x; d < docs; d += blockDim.x) m = fmaxf(m, dm[d]);
    m = wave_max(m);
    if (lane == 0) red[wave] = m;
    __syncthreads();
    m = red[0];
    for (int w = 1; w < waves; ++w) m = fmaxf(m, red[w]);
    __syncthreads();
    float z = 0.f;
    for (int d = threadIdx.x; d < docs; d += blockDim.x) {
        const float s = dsum[d] * exp_below(dm[d], m);
        dsum[d] = s;
        z += s;
    }
    z = wave_sum(z);
    if (lane == 0) red[wave] = z;
    __syncthreads();
    z = red[0];
    for (int w = 1; w < waves; ++w) z += red[w];
    const float inv = 1.f / z;
    const long long at = ((long long)b * p.N + n) * p.R + r;
    for (int d = threadIdx.x; d < docs; d += blockDim.x) p.pdoc[at * docs + d] = dsum[d] * inv;
    if (threadIdx.x == 0) {
        p.stat[2 * at] = m;
        p.stat[2 * at + 1] = inv;
    }
}

// scores[b][d] = out_scale * sum over heads and rows; a thread per document, consecutive documents side by side.
__global__ __launch_bounds__(256) void br_dense_doc_sum_kernel(const float* __restrict__ pdoc, float* __restrict__ scores, int docs, int NR,
                                                               float out_scale) {
    __shared__ float red[4][64];
    const int b = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, d = blockIdx.x * 64 + lane;
    float s = 0.f;
    if (d < docs)
        for (int i = wave; i < NR; i += 4) s += pdoc[((long long)b * NR + i) * docs + d];
    red[wave][lane] = s;
    __syncthreads();
    if (wave == 0 && d < docs) scores[(long long)b * docs + d] = (red[0][lane] + red[1][lane] + red[2][lane] + red[3][lane]) * out_scale;
}

struct BrInfoNceParams {
    const float* logits;     // (B, docs)
    const int64_t* answers;  // (B, A): document indices, negative ones (and docs, one past the last) are padding
    float* loss;             // 1
    float* accuracy;         // 1
    float* lse;              // (B, 2): log-sum-exp over the answers, over all documents
    const float* g;          // gradient of the loss (1)
    float* dlogits;          // (B, docs)
    int B, docs, A;
    int* in_range;           // 1: no answer is beyond docs (may be null; device or pinned host memory)
};

__device__ inline bool is_answer(const BrInfoNceParams& p, int b, int d) {
    for (int a = 0; a < p.A; ++a)
        if (p.answers[(long long)b * p.A + a] == d) return true;
    return false;
}

// Gradient of the InfoNCE loss with respect to the score of document d of sequence b
__device__ inline float infonce_gradient(const BrInfoNceParams& p, int b, int d) {
    const float x = p.logits[(long long)b * p.docs + d];
    float v = expf(x - p.lse[2 * b + 1]);
    if (is_answer(p, b, d)) v -= expf(x - p.lse[2 * b]);
    return v * *p.g / (float)p.B;
}

// dx of one (sequence, head, row of the h1): p * (g_document - sum over documents of p_document g_document) where the row
// is one of the scored ones (once for each time it is named), zero everywhere else.  g: the gradient of the scores (p.g) and
// what comes through the loss (q.g), either of them may be null.
__global__ __launch_bounds__(256) void br_dense_doc_probs_bwd_kernel(BrDenseScoreParams p, BrInfoNceParams q) {
    extern __shared__ float g[];                           // [docs]
    __shared__ float red[4];
    const int docs = p.M - 2, b = blockIdx.y, n = blockIdx.x / p.h1, row = blockIdx.x - n * p.h1;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int S = p.M * p.H;
    const long long base = (((long long)b * p.N + n) * p.h1 + row) * S;
    bool first = true;
    for (int r = 0; r < p.R; ++r) {
        if (row_of(p, b, r) != row) continue;
        const long long at = ((long long)b * p.N + n) * p.R + r;
        float t = 0.f;
        for (int d = threadIdx.x; d < docs; d += 256) {    // (each thread reads back its own elements only, here too)
            if (first) g[d] = (p.g ? p.g[(long long)b * docs + d] : 0.f) + (q.g ? infonce_gradient(q, b, d) : 0.f);
            t += p.pdoc[at * docs + d] * g[d];
        }
        t = wave_sum(t);
        __syncthreads();
        if (lane == 0) red[wave] = t;
        __syncthreads();
        const float dot = red[0] + red[1] + red[2] + red[3];
        const float m = p.stat[2 * at], inv = p.stat[2 * at + 1];
        for (int j = threadIdx.x; j < S; j += 256) {
            const int d = j / p.H - 1;
            float v = 0.f;
            if (d >= 0 && d < docs) v = expf(p.x[base + j] - m) * inv * (g[d] - dot) * p.out_scale;
            p.dx[base + j] = first ? v : p.dx[base + j] + v;     // (each thread reads back its own elements only)
        }
        first = false;
    }
    if (!first) return;
    if ((S & 3) == 0 && (reinterpret_cast<uintptr_t>(p.dx) & 15) == 0) {
        for (int j = 4 * threadIdx.x; j < S; j += 1024) *reinterpret_cast<float4*>(p.dx + base + j) = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
        for (int j = threadIdx.x; j < S; j += 256) p.dx[base + j] = 0.f;
    }
}

// The order torch's argmax has: the first NaN, else the first largest.
__device__ inline bool ahead(float x, int i, float y, int j) {
    if (isnan(x) || isnan(y)) return isnan(x) && (!isnan(y) || i < j);
    return x > y || (x == y && i < j);
}

// loss = -mean over sequences of (log-sum-exp of the answers' logits - log-sum-exp of all), accuracy = how often the first
// largest logit is an answer's; both NaN where an answer is beyond the documents.  One workgroup of sixteen waves, a wave per
// sequence: the whole input is a few kilobytes.
__device__ inline void infonce(const BrInfoNceParams& p) {
    __shared__ float s_loss[16], s_acc[16];
    __shared__ int s_beyond;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_beyond = 0;
    __syncthreads();
    for (long long i = threadIdx.x; i < (long long)p.B * p.A; i += 1024)
        if (p.answers[i] > p.docs) s_beyond = 1;
    float loss = 0.f, acc = 0.f;
    for (int b = wave; b < p.B; b += 16) {
        const float* x = p.logits + (long long)b * p.docs;
        float m = -INFINITY, mp = -INFINITY;
        int am = 0x7fffffff;
        for (int d = lane; d < p.docs; d += 64) {
            if (ahead(x[d], d, m, am)) {
                m = x[d];
                am = d;
            }
            if (is_answer(p, b, d)) mp = fmaxf(mp, x[d]);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) {
            const float y = __shfl_xor(m, o);
            const int i = __shfl_xor(am, o);
            if (ahead(y, i, m, am)) {
                m = y;
                am = i;
            }
        }
        mp = wave_max(mp);
        float s = 0.f, sp = 0.f;
        for (int d = lane; d < p.docs; d += 64) {
            s += exp_below(x[d], m);
            if (is_answer(p, b, d)) sp += exp_below(x[d], mp);
        }
        s = wave_sum(s);
        sp = wave_sum(sp);
        const float all = m + logf(s), pos = mp + logf(sp);
        loss += all - pos;
        acc += am < p.docs && is_answer(p, b, am) ? 1.f : 0.f;
        if (lane == 0) {
            p.lse[2 * b] = pos;
            p.lse[2 * b + 1] = all;
        }
    }
    if (lane == 0) {
        s_loss[wave] = loss;
        s_acc[wave] = acc;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float l = 0.f, a = 0.f;
        for (int w = 0; w < 16; ++w) {
            l += s_loss[w];
            a += s_acc[w];
        }
        *p.loss = s_beyond ? NAN : l / (float)p.B;
        *p.accuracy = s_beyond ? NAN : a / (float)p.B;
        if (p.in_range) {
            *p.in_range = s_beyond == 0;
            __threadfence_system();
        }
    }
}

__global__ __launch_bounds__(1024) void br_infonce_kernel(BrInfoNceParams p) { infonce(p); }

// The sums of br_dense_doc_sum_kernel - four waves to 64 documents, in the same order - and the loss on them, in one workgroup.
// (64 rows of 2 x 12 documents: 5.7 us; 4.5 + 4.0 in two launches, and their gap)
__global__ __launch_bounds__(1024) void br_doc_sum_infonce_kernel(const float* __restrict__ pdoc, float* scores, int NR, float out_scale, BrInfoNceParams p) {
    __shared__ float red[16][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, cols = (p.docs + 63) / 64;
    for (int c0 = 0; c0 < p.B * cols; c0 += 4) {
        const int c = c0 + (wave >> 2), b = c / cols, d = (c - b * cols) * 64 + lane;
        const bool on = b < p.B && d < p.docs;
        float s = 0.f;
        if (on)
#pragma unroll 4
            for (int i = wave & 3; i < NR; i += 4) s += pdoc[((long long)b * NR + i) * p.docs + d];
        red[wave][lane] = s;
        __syncthreads();
        if ((wave & 3) == 0 && on) scores[(long long)b * p.docs + d] = (red[wave][lane] + red[wave + 1][lane] + red[wave + 2][lane] + red[wave + 3][lane]) * out_scale;
        __syncthreads();
    }
    infonce(p);
}

__global__ __launch_bounds__(256) void br_infonce_bwd_kernel(BrInfoNceParams p) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= p.B * p.docs) return;
    const int b = i / p.docs;
    p.dlogits[i] = infonce_gradient(p, b, i - b * p.docs);
}

}  // namespace

void br_launch_bracket_rows(const int64_t* labels, int64_t stride, int B, int S, int h1, const int* guess, int64_t* rows, int* pos, int pos_offset,
                            int* flags, hipStream_t stream) {
    hipLaunchKernelGGL(br_bracket_rows_kernel, dim3(1), dim3(256), 0, stream, labels, stride, B, S, h1, guess, rows, pos, pos_offset, flags);
}

static void launch_probs(const BrDenseScoreParams& p, hipStream_t stream) {
    // a wave per document, of four at least and sixteen at most - four where more would take the launch beyond 2^32 threads
    const int docs = p.M - 2, waves = docs < 4 || (long long)p.N * p.R >= 1 << 22 ? 4 : (docs < 16 ? docs : 16);
    hipLaunchKernelGGL(br_dense_doc_probs_kernel, dim3(p.N * p.R, p.B), dim3(64 * waves), 2 * docs * sizeof(float), stream, p);
}
static void launch_sum(const float* pdoc, float* scores, int B, int docs, int NR, float out_scale, hipStream_t stream) {
    hipLaunchKernelGGL(br_dense_doc_sum_kernel, dim3((docs + 63) / 64, B), dim3(256), 0, stream, pdoc, scores, docs, NR, out_scale);
}

void br_launch_dense_doc_scores(const float* x, const int64_t* rows, float* pdoc, float* stat, float* scores, int B, int N, int h1, int M, int H,
                                int R, float out_scale, hipStream_t stream) {
    const BrDenseScoreParams p = {x, rows, pdoc, stat, nullptr, nullptr, B, N, h1, M, H, R, out_scale};
    launch_probs(p, stream);
    launch_sum(pdoc, scores, B, M - 2, N * R, out_scale, stream);
}

void br_launch_dense_doc_scores_bwd(const float* x, const int64_t* rows, const float* pdoc, const float* stat, const float* g, float* dx, int B,
                                    int N, int h1, int M, int H, int R, float out_scale, hipStream_t stream) {
    const BrDenseScoreParams p = {x, rows, const_cast<float*>(pdoc), const_cast<float*>(stat), g, dx, B, N, h1, M, H, R, out_scale};
    const BrInfoNceParams q = {};
    hipLaunchKernelGGL(br_dense_doc_probs_bwd_kernel, dim3(N * h1, B), dim3(256), (M - 2) * sizeof(float), stream, p, q);
}

// The scores and the loss on them; and both's gradient (g_loss or g_scores may be null).
void br_launch_ranking_loss(const float* x, const int64_t* rows, const int64_t* answers, float* pdoc, float* stat, float* scores, float* loss,
                            float* accuracy, float* lse, int* in_range, int B, int N, int h1, int M, int H, int R, int A, float out_scale,
                            hipStream_t stream) {
    const int docs = M - 2;
    const BrDenseScoreParams p = {x, rows, pdoc, stat, nullptr, nullptr, B, N, h1, M, H, R, out_scale};
    const BrInfoNceParams q = {scores, answers, loss, accuracy, lse, nullptr, nullptr, B, docs, A, in_range};
    launch_probs(p, stream);
    // (one workgroup sums four times 64 documents at a time: beyond a few rounds of that the sums have the chip to themselves)
    if ((long long)B * ((docs + 63) / 64) <= 16) {
        hipLaunchKernelGGL(br_doc_sum_infonce_kernel, dim3(1), dim3(1024), 0, stream, pdoc, scores, N * R, out_scale, q);
    } else {
        launch_sum(pdoc, scores, B, docs, N * R, out_scale, stream);
        hipLaunchKernelGGL(br_infonce_kernel, dim3(1), dim3(1024), 0, stream, q);
    }
}

void br_launch_ranking_loss_bwd(const float* x, const int64_t* rows, const int64_t* answers, const float* pdoc, const float* stat, const float* scores,
                                const float* lse, const float* g_loss, const float* g_scores, float* dx, int B, int N, int h1, int M, int H, int R,
                                int A, float out_scale, hipStream_t stream) {
    const BrDenseScoreParams p = {x, rows, const_cast<float*>(pdoc), const_cast<float*>(stat), g_scores, dx, B, N, h1, M, H, R, out_scale};
    const BrInfoNceParams q = {scores, answers, nullptr, nullptr, const_cast<float*>(lse), g_loss, nullptr, B, M - 2, A, nullptr};
    hipLaunchKernelGGL(br_dense_doc_probs_bwd_kernel, dim3(N * h1, B), dim3(256), (M - 2) * sizeof(float), stream, p, q);
}

void br_launch_infonce(const float* logits, const int64_t* answers, float* loss, float* accuracy, float* lse, int* in_range, int B, int docs,
                       int A, hipStream_t stream) {
    BrInfoNceParams p = {logits, answers, loss, accuracy, lse, nullptr, nullptr, B, docs, A, in_range};
    hipLaunchKernelGGL(br_infonce_kernel, dim3(1), dim3(1024), 0, stream, p);
}

void br_launch_infonce_bwd(const float* logits, const int64_t* answers, const float* lse, const float* g, float* dlogits, int B, int docs, int A,
                           hipStream_t stream) {
    BrInfoNceParams p = {logits, answers, nullptr, nullptr, const_cast<float*>(lse), g, dlogits, B, docs, A, nullptr};
    hipLaunchKernelGGL(br_infonce_bwd_kernel, dim3((B * docs + 255) / 256), dim3(256), 0, stream, p);
}
