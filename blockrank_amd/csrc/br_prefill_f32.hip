// Block-sparse prefill attention for fp32 inputs: same plan, same items, same tile walk and row mapping as the 16-bit
// kernel, all products on the fp32 matrix instruction (v_mfma_f32_32x32x2_f32; an fp32 model is held to 1e-5 of an fp32
// reference, which rules out 16-bit products).
//
// A workgroup takes one (item, head group), a wave 32 query rows of one head.  Per 64-key tile, staged in LDS (the next
// one's pieces are loaded into registers meanwhile), and 32-key half:
//   S^T = K Q^T      lane = query row, registers = keys, so the softmax is in the lane but for one exchange
//   O^T += V^T P^T   the accumulator register that holds keys k (lower lanes) and k + 4 (upper lanes) is as it stands the
//                    product's B operand, whose A operand is V's rows k and k + 4 as lanes read them, dims along the lanes
// so P never leaves its registers.  K's 16-byte pieces sit at piece ^ (row & 15): sixteen lanes then read sixteen
// different groups of four banks.
// Bound by the matrix instruction (64 cycles for 2048 products): 560 tokens, 8/2 heads, D=64 15 us (28 us with the
// query block's walk in pieces of four tiles instead of one), 150 us as dot products
// on the vector ALU with two lanes per row; 4 x 20 documents of 160 tokens, 32/8 heads, D=128 639 us, 2628 us so.
//
// Reference semantics: sdpa_blockrank_attention_forward, blockrank_std_attention.py:503-650.
#include "br_mma.h"
#include "br_finish.h"

namespace {

typedef br_f32x16v f32x16;

template <int D, int NW>
__global__ __launch_bounds__(NW * 64) void br_prefill_f32_kernel(BrPrefillParams p, unsigned first) {
    constexpr int NT = NW * 64, PPR = D / 4, ND = D / 32, NPC = BR_BN * PPR / NT + (BR_BN * PPR % NT != 0);
    __shared__ __attribute__((aligned(16))) float Ks[BR_BN * D];
    __shared__ __attribute__((aligned(16))) float Vs[BR_BN * D];
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, lh = lane >> 5;
    const BrGeom& ge = p.geom;
    const int T = ge.tpb * BR_RB;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, T);
    const int unit = (int)(first + blockIdx.x), item = unit / ge.NHG, hg = unit - item * ge.NHG;
    const BrItem it = pv.items[item];                                // (inside the plan for every workgroup of the grid)
    if (item >= pv.hdr[BR_PH_NITEMS]) return;
    const int b = it.b, kvh = hg / ge.HGS, hsub = hg - kvh * ge.HGS;
    const int g = wave / ge.tpb, sub = wave - g * ge.tpb, head = kvh * ge.G + hsub * ge.Gw + g;
    const int len_m = it.len_m, row0 = it.t0 + sub * BR_RB;
    const bool active = row0 < len_m;
    const int self_end = it.t0 + T < len_m ? it.t0 + T : len_m;
    const float* kbase = reinterpret_cast<const float*>(p.k) + (long long)b * p.sk_b + (long long)kvh * p.sk_h;
    const float* vbase = reinterpret_cast<const float*>(p.v) + (long long)b * p.sv_b + (long long)kvh * p.sv_h;

    uint4 qf[D / 8];
    {
        const int last = len_m - 1 - row0, r = ln < last ? ln : last;     // rows past the end repeat the last one, never stored
        const float* qrow = reinterpret_cast<const float*>(p.q) + (long long)b * p.sq_b + (long long)head * p.sq_h +
                            (long long)(it.tok_m + (active ? row0 + r : 0)) * p.sq_t + lh * 4;
#pragma unroll
        for (int c = 0; c < D / 8; ++c) qf[c] = *reinterpret_cast<const uint4*>(qrow + c * 8);
    }
    const int2* tiles_b = pv.tiles + (size_t)b * pv.tps;
    BrWalk walk;
    walk.init(it, self_end, p.H);
    auto next_tile = [&](BrTile& t) -> bool {
        int pi = 0;
        const int wr = walk.next(t, &pi);
        if (wr == 1) {
            if (it.pe > 1) {
                const int2 d = tiles_b[pi];
                t.tok0 = d.x; t.nvalid = d.y; t.kt = 0; t.self = 0;
            } else {
                br_prefix_tile(it, pi, t);
            }
        }
        return wr != 0;
    };
    uint4 kreg[NPC], vreg[NPC];
    // Five to seven waves have more pieces each and no registers left at head dim 128 to keep their addresses from tile to
    // tile (36, 22 and 7 were spilled): there the addresses come from a thread index that the compiler cannot trace back.
    // 4 x 20 documents of 160, 20/4, 24/4 and 28/4 heads: 709, 677 and 635 us -> 605, 615 and 623 us; four or eight waves
    // lose 1 to 4 % by it (32/8 heads: 638 -> 660 us).
    constexpr bool AFRESH = D == 128 && NW > 4 && NW < 8;
    auto load_tile = [&](const BrTile& t) {                              // rows past the tile's real keys are zero
        int tid = threadIdx.x;
        if constexpr (AFRESH) asm volatile("" : "+v"(tid));
#pragma unroll
        for (int i = 0; i < NPC; ++i) {
            const int idx = tid + i * NT, r = idx / PPR, c = idx - r * PPR;
            const bool on = idx < BR_BN * PPR && r < t.nvalid;
            const long long tok = t.tok0 + (on ? r : 0);
            kreg[i] = *reinterpret_cast<const uint4*>(kbase + tok * p.sk_t + c * 4);
            vreg[i] = *reinterpret_cast<const uint4*>(vbase + tok * p.sv_t + c * 4);
            if (!on) kreg[i] = vreg[i] = uint4{0u, 0u, 0u, 0u};
        }
    };
    f32x16 o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = br_zero16();
    float m_run = -INFINITY, l_run = 0.f;
    BrTile cur, nxt;
    bool have = next_tile(cur);
    if (have) load_tile(cur);
    while (have) {
        __syncthreads();                                                 // the previous tile is consumed
        int tid = threadIdx.x;
        if constexpr (AFRESH) asm volatile("" : "+v"(tid));
#pragma unroll
        for (int i = 0; i < NPC; ++i) {
            const int idx = tid + i * NT, r = idx / PPR, c = idx - r * PPR;
            if (idx < BR_BN * PPR) {
                *reinterpret_cast<uint4*>(Ks + r * D + ((c ^ (r & 15)) << 2)) = kreg[i];
                *reinterpret_cast<uint4*>(Vs + r * D + (c << 2)) = vreg[i];
            }
        }
        __syncthreads();
        const bool have_next = next_tile(nxt);
        if (have_next) load_tile(nxt);
        const int key0 = cur.kt * BR_BN;
        int lim = cur.nvalid, nkb = (cur.nvalid + 31) >> 5;
        if (cur.self) {
            const int c = row0 + ln - key0 + 1, vis = row0 + BR_RB - key0, n = vis <= 0 ? 0 : (vis + 31) >> 5;
            lim = c < lim ? c : lim;
            nkb = n < nkb ? n : nkb;
        }
        if (!active) nkb = 0;
        for (int kb = 0; kb < nkb; ++kb) {
            f32x16 s = br_zero16();
            const float* krow = Ks + (kb * 32 + ln) * D;
#pragma unroll
            for (int c = 0; c < D / 8; ++c) s = BrPiece<float>::mma(*reinterpret_cast<const uint4*>(krow + (((2 * c + lh) ^ (ln & 15)) << 2)), qf[c], s);
            float mx = m_run;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[v] = kb * 32 + 8 * (v >> 2) + 4 * lh + (v & 3) < lim ? s[v] * p.scale_log2 : -INFINITY;
                mx = fmaxf(mx, s[v]);
            }
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float sub_m = mx == -INFINITY ? 0.f : mx;
            const float alpha = __builtin_amdgcn_exp2f(m_run - sub_m);
            m_run = mx;
            l_run *= alpha;
#pragma unroll
            for (int d = 0; d < ND; ++d)
#pragma unroll
                for (int v = 0; v < 16; ++v) o[d][v] *= alpha;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                s[v] = __builtin_amdgcn_exp2f(s[v] - sub_m);
                l_run += s[v];
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float* vrow = Vs + (kb * 32 + 8 * (v >> 2) + 4 * lh + (v & 3)) * D + ND * ln;   // dims ND ln .. of the row
                float x[ND];
                typedef float VN __attribute__((ext_vector_type(ND)));
                const VN y = *reinterpret_cast<const VN*>(vrow);
#pragma unroll
                for (int d = 0; d < ND; ++d) x[d] = y[d];
#pragma unroll
                for (int d = 0; d < ND; ++d) o[d] = br_mma2(x[d], s[v], o[d]);
            }
        }
        cur = nxt;
        have = have_next;
    }
    if (!active || row0 + ln >= len_m) return;
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    // o[d][v]: row row0 + ln, dim ND * (8 (v/4) + 4 lh + v%4) + d - per (v/4, lh) 4 ND consecutive dims
    float* dst;
    float inv = 1.f;
    if (it.slot >= 0) {
        const long long prow = ((long long)it.slot * ge.NHG + hg) * (NW * BR_RB) + wave * BR_RB + ln;
        dst = p.part_o + prow * D;
        if (lh == 0) {
            p.part_ml[prow * 2] = m_run;
            p.part_ml[prow * 2 + 1] = l_tot;
        }
    } else {
        inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
        dst = reinterpret_cast<float*>(p.out) + (long long)b * p.so_b + (long long)head * p.so_h + (long long)(it.tok_m + row0 + ln) * p.so_t;
    }
#pragma unroll
    for (int v4 = 0; v4 < 4; ++v4)
#pragma unroll
        for (int i = 0; i < ND; ++i) {
            // element e of the group's 4 ND: dim offset e = ND (v%4) + d
            float y[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = 4 * i + j;
                y[j] = o[e % ND][4 * v4 + e / ND] * inv;
            }
            *reinterpret_cast<float4*>(dst + ND * (8 * v4 + 4 * lh) + 4 * i) = make_float4(y[0], y[1], y[2], y[3]);
        }
}

}  // namespace

int br_launch_prefill_f32(const BrPrefillParams& p, int D, int NW, int combine_grid, hipStream_t stream, hipEvent_t ev_start, hipEvent_t ev_stop) {
    // a workgroup per item the plan may hold and head group: the plan's real items are the first ones, the others leave at once
    // (below 2^24 of them, and at most 2^22 to a launch: a grid is limited to 2^32 threads)
    const unsigned units = (unsigned)(br_plan_max_items(p.B, p.M, p.H, br_tokens_per_tile(p.geom)) * p.geom.NHG), most = 1u << 22;
    if (ev_start) (void)hipEventRecord(ev_start, stream);
#define BR_CASE(DD, WW)                                                                                        \
    if (D == DD && NW == WW) {                                                                                 \
        for (unsigned u = 0; u < units; u += most)                                                             \
            hipLaunchKernelGGL((br_prefill_f32_kernel<DD, WW>), dim3(units - u < most ? units - u : most), dim3(WW * 64), 0, stream, p, u); \
        goto launched;                                                                                         \
    }
    BR_CASE(128, 4) BR_CASE(128, 5) BR_CASE(128, 6) BR_CASE(128, 7) BR_CASE(128, 8)
    BR_CASE(64, 4) BR_CASE(64, 5) BR_CASE(64, 6) BR_CASE(64, 7) BR_CASE(64, 8)
#undef BR_CASE
    return -1;
launched:
    if (ev_stop) (void)hipEventRecord(ev_stop, stream);
    if (D == 128) br_launch_finish<float, 128, true>(p, NW, combine_grid, stream);
    else br_launch_finish<float, 64, true>(p, NW, combine_grid, stream);
    return 0;
}
