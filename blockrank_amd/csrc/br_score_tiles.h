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
    int B, Nq, M, H, R, Rw;
    float out_scale;
    int per_doc;
};

// PATH of the reduction (picked on the host): 0 - at most 64 documents and 128 tiles, 1 - at most 256 and 768, 2 - any.
// Each is compiled on its own so that none carries the registers of the others.
__host__ __device__ inline int br_doc_final_path(int docs, int tiles) {
    if (docs > 256 || tiles > 768) return 2;
    return docs <= 64 && tiles <= 128 ? 0 : 1;
}
#define BR_SCORE_DOC_CHUNK 8192     // documents whose sums are in LDS at a time (more go in several passes)
// Floats of LDS per wave: a sum per document and, where the tiles' masses go through LDS, one per tile.
__host__ __device__ inline int br_doc_final_per_wave(int docs, int path) {
    return (docs < BR_SCORE_DOC_CHUNK ? docs : BR_SCORE_DOC_CHUNK) + (path == 0 ? 128 : (path == 1 ? 768 : 0));
}
// Waves whose sums fit the LDS (16 at most, a workgroup's), and the bytes they take.
__host__ __device__ inline int br_doc_final_waves(int docs, int path) {
    const int n = 62 * 1024 / (4 * br_doc_final_per_wave(docs, path));
    return n < 1 ? 1 : (n > 16 ? 16 : n);
}
__host__ __device__ inline size_t br_doc_final_lds(int docs, int path) {
    return (size_t)br_doc_final_waves(docs, path) * br_doc_final_per_wave(docs, path) * 4;
}

// One sequence (b) by one workgroup; every thread of it must call this.  dyn: br_doc_final_lds() bytes.  The first nwaves
// waves take the (head, row) pairs round robin, the others only join the barrier.  Of a pair, the lanes take the tiles -
// consecutive ones, whole cache lines per load (a lane per document, each reading its own few tiles, is one line per lane
// and load: at 100 documents of six tiles that alone filled the load path of the one compute unit for 20 us) -, reduce the
// row's maximum, leave every tile's mass in LDS, and then take the documents and add their tiles up.  The waves' sums over
// pairs are added in a fixed order at the end.
template <int PATH>
__device__ __forceinline__ void br_doc_final_tiles_body(const BrTileScoreParams& p, const int b, float* dyn, const int nwaves) {
    const int docs = p.M - 2;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    constexpr int K = PATH == 0 ? 2 : (PATH == 1 ? 12 : 8);      // tiles per lane held at a time
    constexpr int PG = PATH == 0 ? 4 : (PATH == 1 ? 2 : 1);      // pairs whose loads are in flight together
    constexpr int DPL = PATH == 0 ? 1 : 4;                       // documents per lane whose tile ranges are held (PATH < 2)
    constexpr int ROOM = K * 64;
    const int* start = p.plan + br_plan_off_start();
    const int* len = p.plan + br_plan_off_len(p.B, p.M);
    const int* tbase = p.plan + br_plan_off_tbase(p.B, p.M);
    const int tps = p.per_doc ? docs : br_plan_tps(p.M, p.H);
    const int NR = wave < nwaves ? p.Nq * p.R : 0;
    const int bm = b * p.M;
    const int st_q = start[bm + p.M - 1], len_q = len[bm + p.M - 1];
    // document d's tiles, first and count; the documents' tiles are [lo, hi) of a row's partials
    auto doc_range = [&](int d, int& t0, int& nt) {
        if (p.per_doc) {
            t0 = d;
            nt = 1;
        } else {
            t0 = tbase[bm + d + 1];
            nt = (len[bm + d + 1] + BR_BN - 1) / BR_BN;
        }
    };
    int lo, hi, t, n;
    doc_range(0, lo, n);
    doc_range(docs - 1, t, n);
    hi = t + n;
    int dt0[DPL], dnt[DPL];
    if constexpr (PATH < 2) {
#pragma unroll
        for (int k = 0; k < DPL; ++k) {
            const int d = lane + 64 * k;
            dt0[k] = dnt[k] = 0;
            if (d < docs) doc_range(d, dt0[k], dnt[k]);
            dt0[k] -= lo;
        }
    }
    const int per_wave = br_doc_final_per_wave(docs, PATH), chunk = docs < BR_SCORE_DOC_CHUNK ? docs : BR_SCORE_DOC_CHUNK;
    float* mine = dyn + (wave < nwaves ? wave : 0) * per_wave;
    float* mass = mine + chunk;
    const float uniform = 1.f / (float)docs;
    auto wmax = [](float x) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x = fmaxf(x, __shfl_xor(x, o));
        return x;
    };
    auto wsum = [](float x) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
        return x;
    };
    for (int d0 = 0; d0 < docs; d0 += chunk) {                   // (one pass but for PATH 2 with very many documents)
    const int d1 = d0 + chunk < docs ? d0 + chunk : docs;
    if (wave < nwaves)
        for (int d = lane; d < chunk; d += 64) mine[d] = 0.f;
    for (int j0 = wave; j0 < NR; j0 += PG * nwaves) {
        float2 v[PG][K];
        const float2* base[PG];
        bool ok[PG];
#pragma unroll
        for (int i = 0; i < PG; ++i) {
            const int j = j0 + i * nwaves < NR ? j0 + i * nwaves : j0;
            const int nh = j / p.R, r = j - nh * p.R;
            int rr = r;
            ok[i] = hi > lo;
            if (!p.per_doc) {
                rr = p.rows[b * p.R + r];
                rr = rr < 0 ? 0 : (rr >= p.Rw ? p.Rw - 1 : rr);
                const int pos = p.H - p.Rw + rr;
                ok[i] = ok[i] && pos >= st_q && pos < st_q + len_q;      // a padded row: its partials were never written
            }
            base[i] = reinterpret_cast<const float2*>(p.part) + (((long long)b * p.Nq + nh) * (p.per_doc ? p.R : p.Rw) + rr) * tps + lo;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                const int f = lane + 64 * k;
                v[i][k] = base[i][f < hi - lo ? f : 0];                   // (always an address of the row)
            }
        }
#pragma unroll
        for (int i = 0; i < PG; ++i) {
            const int j = j0 + i * nwaves;
            if (j >= NR) continue;
            float* pr_out = p.probs ? p.probs + ((long long)b * p.Nq * p.R + j) * docs : nullptr;
            auto give = [&](int d, float pr) {
                if (pr_out) pr_out[d] = pr;
                mine[d - d0] += pr;
            };
            if (!ok[i]) {
                for (int d = d0 + lane; d < d1; d += 64) give(d, uniform);
                continue;
            }
            float mx = -INFINITY;
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (lane + 64 * k < hi - lo) mx = fmaxf(mx, v[i][k].x);
            if constexpr (PATH == 2)
                for (int f = lane + ROOM; f < hi - lo; f += 64) mx = fmaxf(mx, base[i][f].x);
            mx = wmax(mx);
            const float m_sub = mx == -INFINITY ? 0.f : mx;
            float den = 0.f;
            if constexpr (PATH < 2) {
#pragma unroll
                for (int k = 0; k < K; ++k) {
                    const int f = lane + 64 * k;
                    const float e = f < hi - lo ? v[i][k].y * __builtin_amdgcn_exp2f(v[i][k].x - m_sub) : 0.f;
                    mass[f] = e;
                    den += e;
                }
                den = wsum(den);
                __threadfence_block();                   // (one wave wrote and reads: order is all that is needed)
                const float inv = den > 0.f ? 1.f / den : 0.f;
#pragma unroll
                for (int k = 0; k < DPL; ++k) {
                    const int d = lane + 64 * k;
                    if (d >= docs) continue;
                    float sd = 0.f;
                    for (int f = 0; f < dnt[k]; ++f) sd += mass[dt0[k] + f];
                    give(d, den > 0.f ? sd * inv : uniform);
                }
                __threadfence_block();
            } else {
                for (int f = lane; f < hi - lo; f += 64) {
                    const float2 ms = base[i][f];
                    den += ms.y * __builtin_amdgcn_exp2f(ms.x - m_sub);
                }
                den = wsum(den);
                const float inv = den > 0.f ? 1.f / den : 0.f;
                for (int d = d0 + lane; d < d1; d += 64) {
                    int t0, nt;
                    doc_range(d, t0, nt);
                    float sd = 0.f;
                    for (int f = 0; f < nt; ++f) {
                        const float2 ms = base[i][t0 - lo + f];
                        sd += ms.y * __builtin_amdgcn_exp2f(ms.x - m_sub);
                    }
                    give(d, den > 0.f ? sd * inv : uniform);
                }
            }
        }
    }
    __syncthreads();
    for (int d = d0 + threadIdx.x; d < d1; d += blockDim.x) {
        float acc = 0.f;
        for (int w = 0; w < nwaves; ++w) acc += dyn[w * per_wave + d - d0];
        p.scores[(long long)b * docs + d] = acc * p.out_scale;
    }
    if constexpr (PATH == 2) __syncthreads();
    }
}
