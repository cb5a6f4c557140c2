// Per-document scores from score partials - (max, sum of 2^(logit - max)) pairs per (head, row, key tile or document): the
// parameter block and the workgroup-level reduction, shared by the stand-alone kernel (br_scores.hip) and the kernel that
// runs it next to the merge of the prefill kernel's split partials (br_finish.h).
#pragma once
#include "br_common.h"

// The partials the prefill kernel leaves for the query block's last Rw rows: part[b][n][r][tile], tiles in the order of
// the sequence's tile descriptors (document d owns tiles tbase[d+1] .. + ceil(len/64)).  per_doc: part[b][n][r][document]
// instead (one pair per document, r the index into rows; what br_doc_partial_kernel leaves).
struct BrTileScoreParams {
    const float* part;
    const int* plan;
    const int* rows;        // (B, R) indices into the last Rw positions of the query block
    float* scores;          // (B, docs)
    float* probs;           // optional (B, Nq, R, docs)
    int* count;             // [B] and
    float* sums;            // [B][chunks][docs]: where the workgroups of a sequence meet (chunks > 1 workgroups per sequence)
    int B, Nq, M, H, R, Rw;
    float out_scale;
    int per_doc;
    int chunks;             // workgroups per sequence: 1, or one per BR_SCORE_PAIRS (head, row) pairs
};

#define BR_SCORE_PAIRS 16          // pairs whose probabilities are added up before they join a sequence's sum

// PATH of the reduction (picked on the host): 0 - at most 64 documents and 128 tiles, 1 - at most 256 and 768, 2 - any.
// Each is compiled on its own so that none carries the registers of the others.
__host__ __device__ inline int br_doc_final_path(int docs, int tiles) {
    if (docs > 256 || tiles > 768) return 2;
    return docs <= 64 && tiles <= 128 ? 0 : 1;
}
#define BR_SCORE_DOC_CHUNK 8192     // PATH 2: documents whose sums are in LDS at a time (more go in several passes)
// Floats of LDS per wave: the tiles' masses and, PATH 0, four pairs' probabilities (PATH 1: one pair's, where its masses were);
// PATH 2: a sum per document.
__host__ __device__ inline int br_doc_final_per_wave(int docs, int path) {
    return path == 0 ? 128 + 4 * 64 : (path == 1 ? 768 : (docs < BR_SCORE_DOC_CHUNK ? docs : BR_SCORE_DOC_CHUNK));
}
// Waves that work on pairs: a workgroup's sixteen, or as many as the sums leave room for.
__host__ __device__ inline int br_doc_final_waves(int docs, int path) {
    if (path < 2) return BR_SCORE_PAIRS;
    const int n = 62 * 1024 / (4 * br_doc_final_per_wave(docs, path));
    return n < 1 ? 1 : (n > 16 ? 16 : n);
}
__host__ __device__ inline size_t br_doc_final_lds(int docs, int path) {
    return (size_t)br_doc_final_waves(docs, path) * br_doc_final_per_wave(docs, path) * 4;
}
// Workgroups per sequence of the launch that has a place for them to meet.  (The meeting is three round trips through memory:
// 28 pairs, two to a wave, are done in 5.6 us by one workgroup and in 6.3 by two; 64 pairs in 10.3 and, by four, 8.5.)
__host__ __device__ inline int br_doc_final_chunks(int Nq, int R, int path) {
    if (path == 0 && Nq * R <= 2 * BR_SCORE_PAIRS) return 1;
    return path < 2 ? (Nq * R + BR_SCORE_PAIRS - 1) / BR_SCORE_PAIRS : 1;
}

namespace {

struct BrScoreSeq {
    const BrTileScoreParams& p;
    const int *len, *tbase;
    int b, docs, tps, lo, hi, st_q, len_q;
    // document d's tiles, first and count; all documents' tiles are [lo, hi) of a row's partials
    __device__ void range(int d, int& t0, int& nt) const {
        t0 = p.per_doc ? d : tbase[b * p.M + d + 1];
        nt = p.per_doc ? 1 : (len[b * p.M + d + 1] + BR_BN - 1) / BR_BN;
    }
    __device__ BrScoreSeq(const BrTileScoreParams& p_, int b_) : p(p_), b(b_) {
        const int* start = p.plan + br_plan_off_start();
        len = p.plan + br_plan_off_len(p.B, p.M);
        tbase = p.plan + br_plan_off_tbase(p.B, p.M);
        docs = p.M - 2;
        tps = p.per_doc ? docs : br_plan_tps(p.M, p.H);
        st_q = start[b * p.M + p.M - 1];
        len_q = len[b * p.M + p.M - 1];
        int n;
        range(0, lo, n);
        range(docs - 1, hi, n);
        hi += n;
    }
    // the document tiles' partials of pair j; false: a padded row, whose partials were never written
    __device__ bool row(int j, const float2*& base) const {
        const int n = j / p.R, r = j - n * p.R;
        int rr = r;
        bool ok = hi > lo;
        if (!p.per_doc) {
            rr = p.rows[b * p.R + r];
            rr = rr < 0 ? 0 : (rr >= p.Rw ? p.Rw - 1 : rr);
            const int pos = p.H - p.Rw + rr;
            ok = ok && pos >= st_q && pos < st_q + len_q;
        }
        base = reinterpret_cast<const float2*>(p.part) + (((long long)b * p.Nq + n) * (p.per_doc ? p.R : p.Rw) + rr) * tps + lo;
        return ok;
    }
};

// Maximum and sum over a wave's lanes, in every lane: four steps inside rows of sixteen lanes, two across rows, all in the
// vector ALU (an exchange through the LDS crossbar, __shfl_xor, is a round trip of a hundred clocks for each).
template <int CTRL>
__device__ inline float br_dpp(float x, float otherwise) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(__float_as_uint(otherwise), __float_as_uint(x), CTRL, 0xf, 0xf, false));
}
__device__ inline float br_wave_max(float x) {
    x = fmaxf(x, br_dpp<0x111>(x, -INFINITY));       // from the lane one before in the row, two, four, eight
    x = fmaxf(x, br_dpp<0x112>(x, -INFINITY));
    x = fmaxf(x, br_dpp<0x114>(x, -INFINITY));
    x = fmaxf(x, br_dpp<0x118>(x, -INFINITY));
    x = fmaxf(x, br_dpp<0x142>(x, -INFINITY));       // a row's last lane to the next row, then the first half's to the second
    x = fmaxf(x, br_dpp<0x143>(x, -INFINITY));
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 63));
}
__device__ inline float br_wave_sum(float x) {
    x += br_dpp<0x111>(x, 0.f);
    x += br_dpp<0x112>(x, 0.f);
    x += br_dpp<0x114>(x, 0.f);
    x += br_dpp<0x118>(x, 0.f);
    x += br_dpp<0x142>(x, 0.f);
    x += br_dpp<0x143>(x, 0.f);
    return __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(x), 63));
}

// Any number of documents and tiles, one workgroup per sequence: nwaves waves take the pairs round robin and add into
// sums of their own, a lane per document.
__device__ inline void br_doc_final_any(const BrTileScoreParams& p, int b, float* dyn, int nwaves) {
    const BrScoreSeq q(p, b);
    const int docs = q.docs, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int NR = wave < nwaves ? p.Nq * p.R : 0;
    const int chunk = br_doc_final_per_wave(docs, 2);
    float* mine = dyn + (wave < nwaves ? wave : 0) * chunk;
    for (int d0 = 0; d0 < docs; d0 += chunk) {
        const int d1 = d0 + chunk < docs ? d0 + chunk : docs;
        if (wave < nwaves)
            for (int d = lane; d < chunk; d += 64) mine[d] = 0.f;
        for (int j = wave; j < NR; j += nwaves) {
            const float2* base;
            const bool ok = q.row(j, base);
            float mx = -INFINITY, den = 0.f;
            if (ok) {
                for (int f = lane; f < q.hi - q.lo; f += 64) mx = fmaxf(mx, base[f].x);
                mx = br_wave_max(mx);
                mx = mx == -INFINITY ? 0.f : mx;
                for (int f = lane; f < q.hi - q.lo; f += 64) {
                    const float2 ms = base[f];
                    den += ms.y * __builtin_amdgcn_exp2f(ms.x - mx);
                }
                den = br_wave_sum(den);
            }
            const float inv = den == 0.f ? 0.f : 1.f / den;          // (NaN stays NaN)
            for (int d = d0 + lane; d < d1; d += 64) {
                float pr = 1.f / (float)docs;
                if (inv != 0.f) {
                    int t0, nt;
                    q.range(d, t0, nt);
                    pr = 0.f;
                    for (int f = 0; f < nt; ++f) {
                        const float2 ms = base[t0 - q.lo + f];
                        pr += ms.y * __builtin_amdgcn_exp2f(ms.x - mx);
                    }
                    pr *= inv;
                }
                if (p.probs) p.probs[((long long)b * p.Nq * p.R + j) * docs + d] = pr;
                mine[d - d0] += pr;
            }
        }
        __syncthreads();
        for (int d = d0 + threadIdx.x; d < d1; d += blockDim.x) {
            float acc = 0.f;
            for (int w = 0; w < nwaves; ++w) acc += dyn[w * chunk + d - d0];
            p.scores[(long long)b * docs + d] = acc * p.out_scale;
        }
        __syncthreads();
    }
}

}  // namespace

// One sequence (b), pairs chunk * 16 .. of it - with p.chunks == 1 all of them - by one workgroup of 1024 threads; every
// thread of it must call this.  dyn: br_doc_final_lds() bytes.  A wave takes one (head, row) pair: its lanes take the tiles
// - consecutive ones, whole cache lines per load (a lane per document, each reading its own few tiles, is one line per lane
// and load) -, reduce the row's maximum, leave every tile's mass in LDS, then take the documents and add their tiles up.
// The probabilities of sixteen pairs are added in the order of the pairs, such sums in the order of the chunks: the result
// is the same bits however many workgroups share a sequence.  The last one of a sequence to be done adds the chunks up;
// what they exchange goes through device-scope atomics, which need no cache to be written back (a fence here would write
// the attention's output back first).
// Latency-bound - a chain of memory round trips and lane exchanges.  At most 64 documents (PATH 0): a wave requests the partials
// of four pairs together, and 64 pairs take one barrier (5.7 us for 20 documents, 32 heads x 2 rows, by one workgroup; a pair at
// a time with lane exchanges through LDS 8.9).  More documents: a pair at a time, four workgroups to 64 pairs.
template <int PATH>
__device__ __forceinline__ void br_doc_final_tiles_body(const BrTileScoreParams& p, const int b, const int chunk0, float* dyn, const int nwaves) {
    if constexpr (PATH == 2) {
        br_doc_final_any(p, b, dyn, nwaves);
        return;
    } else {
        constexpr int K = PATH == 0 ? 2 : 12;                    // tiles per lane
        constexpr int DPL = PATH == 0 ? 1 : 4;                   // documents per lane
        const BrScoreSeq q(p, b);
        const int docs = q.docs, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
        const int NR = p.Nq * p.R, span = q.hi - q.lo;
        int dt0[DPL], dnt[DPL];
#pragma unroll
        for (int k = 0; k < DPL; ++k) {
            const int d = lane + 64 * k;
            dt0[k] = dnt[k] = 0;
            if (d < docs) {
                q.range(d, dt0[k], dnt[k]);
                dt0[k] = dnt[k] > 0 ? dt0[k] - q.lo : 0;         // (a document without tokens owns no tile)
            }
        }
        constexpr int PPW = PATH == 0 ? 4 : 1;                   // pairs of a wave per round
        constexpr int MD = PATH == 0 ? 64 : 768;                 // floats between two pairs' probabilities
        float* mass = PATH == 0 ? dyn + BR_SCORE_PAIRS * PPW * MD + wave * 128 : dyn + wave * MD;
        const int end = p.chunks > 1 && (chunk0 + 1) * BR_SCORE_PAIRS < NR ? (chunk0 + 1) * BR_SCORE_PAIRS : NR;
        float total = 0.f;                                       // document threadIdx.x's sum
#pragma unroll 1
        for (int j0 = chunk0 * BR_SCORE_PAIRS; j0 < end; j0 += BR_SCORE_PAIRS * PPW) {
            float2 v[PPW][K];
            bool ok[PPW];
#pragma unroll
            for (int n = 0; n < PPW; ++n) {
                const int j = j0 + n * BR_SCORE_PAIRS + wave;
                ok[n] = false;
                if (j >= end) break;
                const float2* base;
                ok[n] = q.row(j, base);
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int f = lane + 64 * k;
                    v[n][k] = base[f < span ? f : 0];            // (always an address of the row)
                }
            }
#pragma unroll
            for (int n = 0; n < PPW; ++n) {
                const int j = j0 + n * BR_SCORE_PAIRS + wave;
                if (j >= end) break;
                float mx = -INFINITY, den = 0.f;
#pragma unroll
                for (int k = 0; k < K; ++k)
                    if (lane + 64 * k < span) mx = fmaxf(mx, v[n][k].x);
                mx = br_wave_max(mx);
                mx = mx == -INFINITY ? 0.f : mx;
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const float e = lane + 64 * k < span ? v[n][k].y * __builtin_amdgcn_exp2f(v[n][k].x - mx) : 0.f;
                    mass[lane + 64 * k] = e;
                    den += e;
                }
                den = br_wave_sum(den);
                __threadfence_block();                           // (one wave wrote and reads: order is all that is needed)
                const bool on = ok[n] && den != 0.f;             // (NaN stays NaN)
                const float inv = on ? 1.f / den : 0.f, uniform = 1.f / (float)docs;
                float pr[DPL];
#pragma unroll
                for (int k = 0; k < DPL; ++k) {
                    float e[8], sd = 0.f;
#pragma unroll
                    for (int f = 0; f < 8; ++f) e[f] = mass[dt0[k] + (f < dnt[k] ? f : 0)];
#pragma unroll
                    for (int f = 0; f < 8; ++f) sd += f < dnt[k] ? e[f] : 0.f;
                    for (int f = 8; f < dnt[k]; ++f) sd += mass[dt0[k] + f];
                    pr[k] = on ? sd * inv : uniform;
                }
                __threadfence_block();
#pragma unroll
                for (int k = 0; k < DPL; ++k) {
                    const int d = lane + 64 * k;
                    if (d >= docs) continue;
                    dyn[(n * BR_SCORE_PAIRS + wave) * MD + d] = pr[k];
                    if (p.probs) p.probs[((long long)b * NR + j) * docs + d] = pr[k];
                }
            }
            __syncthreads();
            if ((int)threadIdx.x < docs) {
#pragma unroll
                for (int n = 0; n < PPW; ++n) {
                    const int left = end - j0 - n * BR_SCORE_PAIRS;
                    if (left <= 0) break;
                    float s = 0.f;
#pragma unroll
                    for (int w = 0; w < BR_SCORE_PAIRS; ++w) s += w < left ? dyn[(n * BR_SCORE_PAIRS + w) * MD + threadIdx.x] : 0.f;
                    total += s;
                }
            }
            __syncthreads();
        }
        if (p.chunks > 1) {
            __shared__ int s_last;
            float* sums = p.sums + (long long)b * p.chunks * docs;
            if ((int)threadIdx.x < docs)
                __hip_atomic_store(sums + (long long)chunk0 * docs + threadIdx.x, total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // this wave's sums have arrived
            __syncthreads();
            if (threadIdx.x == 0) s_last = __hip_atomic_fetch_add(p.count + b, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == p.chunks - 1;
            __syncthreads();
            if (!s_last) return;
            if (threadIdx.x == 0) __hip_atomic_store(p.count + b, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);   // at rest again
            if ((int)threadIdx.x < docs) {
                total = 0.f;
                for (int c0 = 0; c0 < p.chunks; c0 += 8) {
                    float x[8];
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        x[i] = __hip_atomic_load(sums + (long long)(c0 + i < p.chunks ? c0 + i : c0) * docs + threadIdx.x, __ATOMIC_RELAXED,
                                                 __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
                    for (int i = 0; i < 8; ++i)
                        if (c0 + i < p.chunks) total += x[i];
                }
            }
        }
        if ((int)threadIdx.x < docs) p.scores[(long long)b * docs + threadIdx.x] = total * p.out_scale;
    }
}
