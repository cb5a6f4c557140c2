// What follows a prefill kernel in the same call, in one launch: the merge of the split-KV partials of the query blocks,
// zeros in the padded rows no item owns, and - where the caller named the rows - the per-document scores.
#pragma once
#include "br_common.h"
#include "br_score_tiles.h"

namespace {

template <typename T>
__device__ inline void br_store4(T* dst, const float (&x)[4]) {
    typedef T V4 __attribute__((ext_vector_type(4)));
    V4 y;
#pragma unroll
    for (int i = 0; i < 4; ++i) y[i] = (T)x[i];
    *reinterpret_cast<V4*>(dst) = y;
}

// Merge: out = sum_s O_s 2^(m_s - m) / sum_s l_s 2^(m_s - m), a thread per four elements of a row, the loads of eight
// splits in flight together.  ALL: every block's padded rows are zeroed here (the 16-bit prefill kernels do that
// themselves).
// PATH >= 0 (with score_wgs > 0): the first score_wgs workgroups (sp.chunks per sequence) turn the score partials the prefill
// kernel left into per-document scores instead (sp); PATH < 0: the merge alone.
// Latency-bound: a few megabytes at most, and the chain of dependent round trips after a kernel boundary is what it takes
// - the list entry (which carries what the block table would say), the partials, the store.  The padded rows are handed
// out from the last workgroup down, the merge from the first up, so that few do both.
template <typename T, int D, int THREADS, int PATH, bool ALL>
__global__ __launch_bounds__(THREADS) void br_finish_kernel(BrPrefillParams p, int NW, BrTileScoreParams sp, int score_wgs, int sp_waves, int wide) {
    if constexpr (PATH >= 0) {
        extern __shared__ float br_finish_dyn[];
        if ((int)blockIdx.x < score_wgs) {
            br_doc_final_tiles_body<PATH>(sp, blockIdx.x / sp.chunks, blockIdx.x % sp.chunks, br_finish_dyn, sp_waves);
            return;
        }
    } else {
        score_wgs = 0;
    }
    typedef float f4 __attribute__((ext_vector_type(4)));
    const int bid = blockIdx.x - score_wgs, nblk = gridDim.x - score_wgs;
    const BrGeom& ge = p.geom;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, ge.tpb * BR_RB);
    constexpr int CPR = D / 4;                    // float4 chunks per row
    const int tpr = wide ? 64 : CPR;              // threads per row: wide, the lanes of a wave in 64 / CPR groups that share the splits
    const int RPW = THREADS / tpr;                // rows one workgroup merges at a time
    const int step = wide ? 64 / CPR : 1;         // splits between two of a lane's
    const int rows = NW * BR_RB;                  // rows of one (combine entry, head group): NW query-tile waves of 32
    const int subs = (rows + RPW - 1) / RPW;      // such row groups
    const int max_comb = br_plan_max_comb(p.B);
    const int rr = threadIdx.x / tpr, cc = threadIdx.x % CPR, first = wide ? threadIdx.x % 64 / CPR : 0;
    for (int u = bid;; u += nblk) {
        const int subu = u % subs;
        const int w = u / subs;
        const int ci = w / ge.NHG, hg = w - ci * ge.NHG;
        if (ci >= max_comb) break;
        const BrComb c = pv.comb[ci];                                // (read before it is known to be one: one round trip)
        if (ci >= pv.hdr[BR_PH_NCOMB]) break;
        const int r = subu * RPW + rr;                               // row inside the slot
        if (r >= rows) continue;
        const int wave = r / BR_RB, rloc = r - wave * BR_RB;         // the prefill wave that owned it, row of its 32
        const int kvh = hg / ge.HGS, hsub = hg - kvh * ge.HGS;
        const int g = wave / ge.tpb, sub = wave - g * ge.tpb;
        const int row = c.t0 + sub * BR_RB + rloc;
        if (row >= c.len_m || hsub * ge.Gw + g >= ge.G) continue;    // (the second: a wave without a head, ragged group)
        const int head = kvh * ge.G + hsub * ge.Gw + g;
        const long long slot0 = (long long)c.slot0 * ge.NHG + hg;
        const long long sstride = (long long)ge.NHG * rows;          // rows between consecutive splits
        const float2* ml = reinterpret_cast<const float2*>(p.part_ml) + slot0 * rows + r;
        const float* lx = p.part_lx + slot0 * rows + r;
        const bool want_lse = p.lse != nullptr && cc == 0;          // (a group's first lane)
        const float* po = p.part_o + (slot0 * rows + r) * D + cc * 4;
        float mmax = -INFINITY, l = 0.f, lex = 0.f;
        f4 acc = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = first; s0 < c.nsplit; s0 += 8 * step) {
            float2 mls[8];
            float lxs[8];
            f4 ov[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int at = s0 + j * step;
                const bool on = at < c.nsplit;
                mls[j] = on ? ml[at * sstride] : make_float2(-INFINITY, 0.f);
                ov[j] = on ? *reinterpret_cast<const f4*>(po + at * sstride * D) : f4{0.f, 0.f, 0.f, 0.f};
                lxs[j] = (on && want_lse) ? lx[at * sstride] : 0.f;
            }
            float mnew = mmax;
#pragma unroll
            for (int j = 0; j < 8; ++j) mnew = fmaxf(mnew, mls[j].x);
            const float resc = mmax == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mmax - mnew);
            l *= resc;
            lex *= resc;
            acc *= resc;
            mmax = mnew;
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float w8 = mls[j].x == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mls[j].x - mmax);
                l += mls[j].y * w8;
                lex += lxs[j] * w8;
                acc += ov[j] * w8;
            }
        }
        if (wide) {                               // the groups' sums joined
#pragma unroll
            for (int d = CPR; d < 64; d <<= 1) {
                const float mo = __shfl_xor(mmax, d), mnew = fmaxf(mmax, mo);
                const float own = mmax == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mmax - mnew), other = mo == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo - mnew);
                l = l * own + __shfl_xor(l, d) * other;
                lex = lex * own + __shfl_xor(lex, d) * other;
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = acc[e] * own + __shfl_xor(acc[e], d) * other;
                mmax = mnew;
            }
            if (first != 0) continue;
        }
        const float inv = l > 0.f ? 1.f / l : 0.f;
        // (the log-sum-exp from the exact sums, as the rows the prefill kernel finishes itself get it)
        if (want_lse) p.lse[(long long)c.b * p.lse_b + (long long)head * p.lse_h + c.tok_m + row] = mmax + __builtin_amdgcn_logf(lex);
        T* dst = reinterpret_cast<T*>(p.out) + (long long)c.b * p.so_b + (long long)head * p.so_h + (long long)(c.tok_m + row) * p.so_t;
        const float y[4] = {acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
        br_store4<T>(dst + cc * 4, y);
    }
    // Padded token slots: no kernel computes them, so give them a defined value (zero): of documents with no real token at
    // all (the prefill kernel has no item for them) - with ALL of every block (a packed layout has no padded slots).  One
    // (block, eight heads) per wave and step, with ALL eight slots of it: the loop is a chain of dependent loads (block table,
    // then the stores' addresses), so what counts is how many of them are in flight.
    const int hgs = (p.Nq + 7) / 8, parts = ALL ? (p.H + 7) / 8 : 1, n_pad_work = pv.hdr[BR_PH_PACKED] ? 0 : p.B * p.M * hgs * parts;
    constexpr int WAVES = THREADS / 64;
    const int lane = threadIdx.x & 63;
    for (int w = (nblk - 1 - bid) * WAVES + (threadIdx.x >> 6); w < n_pad_work; w += nblk * WAVES) {
        const int bh = w / parts, part = w - bh * parts;
        const int bm = bh / hgs, head0 = (bh - bm * hgs) * 8, heads = p.Nq - head0 < 8 ? p.Nq - head0 : 8;
        const int b = bm / p.M, mm = bm - b * p.M;
        const int st = pv.start[bm], ln = pv.len[bm];
        if (!ALL && (ln != 0 || mm == 0 || mm == p.M - 1)) continue;
        const int r0 = ALL ? part * 8 : 0, r1 = ALL && r0 + 8 < p.H ? r0 + 8 : p.H;
        constexpr int E = 16 / sizeof(T), CP = D / E;
        T* obase = reinterpret_cast<T*>(p.out) + (long long)b * p.so_b + (long long)head0 * p.so_h + (long long)(mm * p.H) * p.so_t;
        for (int idx = lane; idx < heads * CP; idx += 64) {
            T* dst = obase + (long long)(idx / CP) * p.so_h + idx % CP * E;
#pragma unroll 8
            for (int r = r0; r < r1; ++r)
                if (r < st || r >= st + ln) *reinterpret_cast<uint4*>(dst + (long long)r * p.so_t) = uint4{0u, 0u, 0u, 0u};
        }
    }
}

// Whether a wave takes a row of its own (wide) instead of 64 / CPR rows: where the grid's waves hold all rows of a batch with one
// split query tile per sequence.  Then - few sequences - a row has many splits, and fewer of them per lane are fewer round trips
// (one request of 20 documents, 20 splits: 10.8 -> 7.6 us with the scores beside it, 6.4 -> 5.9 alone; four requests the other
// way round: 7.0 -> 9.4 alone).
inline int br_finish_wide(const BrPrefillParams& p, int NW, int combine_grid) {
    return (long long)p.B * p.geom.NHG * NW * BR_RB <= 4LL * combine_grid;
}

// Launch of the finish kernel after a prefill kernel.  combine_grid: workgroups of 256 threads the merge alone would take.
template <typename T, int D, bool ALL>
inline void br_launch_finish(const BrPrefillParams& p, int NW, int combine_grid, hipStream_t stream) {
    const BrTileScoreParams none = {};
    hipLaunchKernelGGL((br_finish_kernel<T, D, 256, -1, ALL>), dim3(combine_grid), dim3(256), 0, stream, p, NW, none, 0, 0, br_finish_wide(p, NW, combine_grid));
}

// ... after a 16-bit one.  sp: the per-document score reduction to run in the same launch (its partials are those the
// prefill kernel just wrote), or nullptr.
template <typename T, int D>
inline void br_launch_finish_scores(const BrPrefillParams& p, int NW, int combine_grid, const BrTileScoreParams* sp, hipStream_t stream) {
    if (!sp) {
        br_launch_finish<T, D, false>(p, NW, combine_grid, stream);
        return;
    }
    const int docs = sp->M - 2, path = br_doc_final_path(docs, br_plan_tps(sp->M, sp->H));
    BrTileScoreParams q = *sp;
    q.chunks = br_doc_final_chunks(q.Nq, q.R, path);
    const int nwaves = br_doc_final_waves(docs, path), wgs = q.B * q.chunks;
    const size_t lds = br_doc_final_lds(docs, path);
    const dim3 grid(wgs + (combine_grid + 3) / 4), block(1024);
    if (path == 0) hipLaunchKernelGGL((br_finish_kernel<T, D, 1024, 0, false>), grid, block, lds, stream, p, NW, q, wgs, nwaves, br_finish_wide(p, NW, combine_grid));
    else if (path == 1) hipLaunchKernelGGL((br_finish_kernel<T, D, 1024, 1, false>), grid, block, lds, stream, p, NW, q, wgs, nwaves, br_finish_wide(p, NW, combine_grid));
    else hipLaunchKernelGGL((br_finish_kernel<T, D, 1024, 2, false>), grid, block, lds, stream, p, NW, q, wgs, nwaves, br_finish_wide(p, NW, combine_grid));
}

}  // namespace
