// Backward of the block-sparse prefill attention for gfx950 (bf16 inputs, fp32 arithmetic and accumulation).
//
// The reference has no hand-written backward: its trainable hooks (blockrank_std_attention.py:96-262, :472-650,
// used by trainer.py:79-101) are differentiated by torch autograd over dense masked tensors, and its Triton
// hook refuses (blockrank_triton_kernel_attention.py:759-761).  These kernels compute the same gradients
//     P = softmax(S),  dV = P^T dO,  dP = dO V^T,  dS = P * (dP - rowsum(dO * O)),
//     dQ = scale * dS K,  dK = scale * dS^T Q        (dK, dV summed over the query heads of a kv head)
// over exactly the (query row, key) pairs the forward visits.  P is rebuilt from the log-sum-exp the forward
// saved.  Two passes, so that every sum that has one owner is kept in that owner's registers, in one launch (br_bwd_kernel) or
// two (br_bwd_one_launch says where):
//
//   br_bwd_dq_kernel   query-major, over the plan's work items (times head groups): a wave per 32 rows of one query
//                      head.  S^T = K Q^T, dP^T = V dO^T (lane = query row, registers = keys) -> dS^T in bf16 is directly
//                      an operand of dQ^T += K^T dS^T (K through transposing LDS reads).  An item that owns its rows
//                      stores dQ; the items that share the query block's rows (its key walk is split) add into a small
//                      fp32 buffer that a finishing kernel converts.  Also writes -delta = -rowsum(dO * O) for the
//                      second kernel.
//   br_bwd_dkv_kernel  key-major: a wave owns 32 keys and walks every (32-row block, head of the group) that sees them.
//                      S = Q K^T, dP = dO V^T (lane = key, registers = rows) -> P and dS in bf16 are directly operands of
//                      dV^T += dO^T P and dK^T += Q^T dS, with dO and Q through transposing LDS reads.  dK and dV never
//                      leave the registers until the walk ends; keys with one owner are stored in bf16, prefix keys -
//                      every block sees them - are added up in fp32 buffers.
//
// Both are persistent, and a workgroup draws the ticket of its next item while it is on the last of the present one.
// Measured at 4 x 20 documents of 160 tokens, 32/8 heads, D = 128 (medians of 70 launches): in one launch 257 us, in two (dQ / dK,
// dV) 128 / 138, with tickets drawn two items ahead 134 / 155 us, with a workgroup per item and S and dP exchanged between two
// waves 152 / 249 us; at 2 x 16 documents of 256 to 512 in two: 173 / 187 us, 176 / 222 and 227 / 464 us before.
// Past the L2s dQ moves 568 MB in its 128 us (488 of them it cannot do without), dK, dV 536 in 138 (328), the single launch 1093
// in 257.  That binds dQ in part and dK, dV hardly: with every item's rows the same cached ones (results wrong, dQ fetching 109
// instead of 452 MB, dK, dV 70 instead of 431) dQ took 110 instead of 129 us, dK, dV 135 instead of 139 (tenth percentiles).
// What is left of a dK/dV step's 3300 clocks (two waves per SIMD, 2048 of them matrix instructions) is the issue of its row
// DMAs (550) and the wait for the wave with the most work (400 to 1200); of an item's time a fifth is keys, stores and
// looking up the next one, and on a document's own keys half of a wave's steps are rows that do not see them.  Over the whole
// kernel the matrix pipes are busy 23 % of the time and LDS 17 % (dQ: 20 and 17 %, in one launch 23 and 19): per product LDS is active 6.0 of the 8
// clocks that keep a CU's four matrix pipes fed, so it is the next limit, not the present one.  D = 128 dK/dV spills four
// registers before its first item and reads them back once per item, none in the walk.
#include "br_common.h"
#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
// The compiler's scheduler moves nothing across
#define BR_SCHED_FENCE() __builtin_amdgcn_sched_barrier(0)

__device__ inline uint4 ld16(const void* p) { return *reinterpret_cast<const uint4*>(p); }
__device__ inline bf16x8 as_bf16x8(uint4 u) {
    union { uint4 u; bf16x8 v; } c;
    c.u = u;
    return c.v;
}
// Workgroup barrier that waits for this wave's LDS operations only.  __syncthreads() also waits for its outstanding
// global loads, which would make every barrier wait for the rows requested ahead for the next step.
__device__ inline void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// LDS DMA: 64 lanes x 16 (or 4) bytes from a uniform base + per-lane byte offset to lds_addr + lane * 16 (4).  In asm, so
// that the compiler does not make LDS reads of other buffers wait for it; completion is awaited by vm_wait.
__device__ inline void dma16(const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
// Four of them from one base to four consecutive KB of LDS (the constant offset moves both addresses)
__device__ inline void dma16x4(const void* base, const int (&off)[4], unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %5\n\tglobal_load_lds_dwordx4 %0, %4\n\tglobal_load_lds_dwordx4 %1, %4 offset:1024\n\t"
                 "global_load_lds_dwordx4 %2, %4 offset:2048\n\tglobal_load_lds_dwordx4 %3, %4 offset:3072"
                 ::"v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3]), "s"(base), "s"(lds_addr) : "memory", "m0");
}
// The same for the lanes of a mask only (every lane of the wave is active around it): one instruction whatever the mask
__device__ inline void dma16_lanes(unsigned long long mask, const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b64 exec, %3\n\ts_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(lds_addr), "s"(mask) : "memory", "m0");
}
__device__ inline void dma4_lanes(unsigned long long mask, const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b64 exec, %3\n\ts_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(lds_addr), "s"(mask) : "memory", "m0");
}
// ... and where the uniform mask is -1, nothing where it is 0
__device__ inline void dma16_if(int mask, const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\ts_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(lds_addr), "s"(mask) : "memory", "m0");
}
__device__ inline void dma4_if(int mask, const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b32 exec_lo, %3\n\ts_mov_b32 exec_hi, %3\n\ts_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1\n\ts_mov_b64 exec, -1" ::"v"(off), "s"(base), "s"(lds_addr), "s"(mask) : "memory", "m0");
}
// A pointer that is the same in every lane, in scalar registers
template <typename T>
__device__ inline const T* uniform(const T* p) {
    const unsigned long long u = (unsigned long long)p;
    return (const T*)((unsigned long long)(unsigned)__builtin_amdgcn_readfirstlane((int)(u >> 32)) << 32 | (unsigned)__builtin_amdgcn_readfirstlane((int)u));
}
template <int N>
__device__ inline void vm_wait() { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory"); }
// This wave's LDS operations so far are done (and the compiler moves none across)
__device__ inline void lds_fence() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
__device__ inline unsigned lds_addr_of(const void* p) { return (unsigned)(size_t)(__attribute__((address_space(3))) const void*)p; }
__device__ inline unsigned pack2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
}
__device__ inline f32x16 mma(bf16x8 a, bf16x8 b, f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ inline f32x16 zero16() {
    f32x16 z;
#pragma unroll
    for (int i = 0; i < 16; ++i) z[i] = 0.f;
    return z;
}

// Kernel arguments where the compiler loads them at their use: through a pointer it cannot trace back, or it would keep
// them all in scalar registers across a persistent kernel's loop, which do not suffice, and their spills take vector ones.
typedef const __attribute__((address_space(4))) BrBwdParams* BrBwdArgs;
__device__ inline const BrBwdParams& args_now(BrBwdArgs a) {
    asm volatile("" : "+s"(a));
    return *(const BrBwdParams*)a;
}

// One unit of the dK/dV kernel's work: up to four 32-key groups, one per wave, that the rows of one block (m, of one
// sequence and kv head) see.  The block's key groups in order are those of the prefix, which all its rows see (m > 0), then
// its own; a document's own groups are also seen by the rows of the query block.
struct BrDkvItem {
    int valid, b, kvh, m;
    int group;                         // first of the four groups
    int len_m, tok_m, start_m;         // the block: real tokens, the index of the first on the token axis, its slot in the block
    int len_p, tok_p;                  // the prefix as seen from the block (no keys when m is 0)
    int len_q, tok_q;                  // the query block where it sees the block's keys (documents), else no rows
};
// ... and, in the LDS mail only, whether the rows' deltas did not come: then the results are NaN
constexpr int kDkvItemWords = sizeof(BrDkvItem) / 4, kDkvLost = kDkvItemWords;

template <int D>
struct Bwd {
    static constexpr int CPR = D / 8;              // 16-byte pieces per row
    static constexpr int NC = D / 16, ND = D / 32;

    // ---------------------------------------------------------------------------------------------------------
    // dQ (and delta) of one work item: a wave per 32 rows of one head.  64-key tiles of K and V come into one of two LDS
    // buffers by DMA, a tile ahead (one barrier per tile).  Per 32 keys of a tile
    //     S^T = K Q^T, dP^T = V dO^T       (A = keys from LDS, B = the wave's rows, kept in registers)
    //     dQ^T += K^T dS^T                 (dS in bf16 straight from the accumulators; K by transposing reads)
    // 24 MFMAs against 24 KB of LDS reads.
    // ---------------------------------------------------------------------------------------------------------
    static constexpr int rowB = 2 * D;                                    // bytes of a row, in memory and in the buffers
    static constexpr int tileB = BR_BN * rowB, stageB = 2 * tileB;        // a tile of K (or V); K, then V
    static constexpr int dqLdsBytes(int maxw) { return maxw <= 4 ? 2 * stageB : stageB + maxw * BR_RB * rowB; }
    // 16-byte piece c of row r sits at piece c ^ row_swizzle(r): the 32 rows one operand read takes a piece of, and the
    // four rows x 64 bytes a transposing read takes, each spread over all banks
    static __device__ inline unsigned row_swizzle(unsigned r) {
        return CPR == 16 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    }

    // NWT: waves per workgroup, or 0: nw, known at run time only.  COUNT: count the row blocks whose delta is published.  draw and
    // drawn: called once by every wave, before and after the walk.
    template <int NWT, bool COUNT, typename F, typename F2>
    static __device__ __forceinline__ void dq_item(BrBwdArgs args, const BrItem& it, int hg, int nw, char* smem, F&& draw, F2&& drawn) {
        const BrBwdParams& p = args_now(args);
        // (per item values that the compiler cannot trace back: nothing derived from them is kept in registers across items)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int NW = NWT ? NWT : nw;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, lh = lane >> 5;
        const unsigned smem_lds = lds_addr_of(smem);
        const int b = it.b, len_m = it.len_m;
        const int hgs = p.geom.HGS, tpb = p.geom.tpb, T = tpb * BR_RB;
        const int kvh = hgs == 1 ? hg : hg / hgs, hsub = hg - kvh * hgs;
        const int g = tpb == 1 ? wave : wave / tpb, sub = wave - g * tpb;
        const int head = kvh * p.geom.G + hsub * p.geom.Gw + g;
        const int row0 = it.t0 + sub * BR_RB;
        const bool rb_active = row0 < len_m;
        const int self_end = it.t0 + T < len_m ? it.t0 + T : len_m;
        const char* kbase = reinterpret_cast<const char*>(p.k) + 2 * ((unsigned long long)p.k32_b * (unsigned)b + (unsigned long long)p.k32_h * (unsigned)kvh);
        const char* vbase = reinterpret_cast<const char*>(p.v) + 2 * ((unsigned long long)p.v32_b * (unsigned)b + (unsigned long long)p.v32_h * (unsigned)kvh);

        // the item's key walk: the earlier blocks' tiles it covers, then its own block's up to the diagonal
        typedef const __attribute__((address_space(4))) int2* plan_tiles;
        const plan_tiles tiles_b = (plan_tiles)(p.plan + br_plan_off_tiles(p.B, p.M)) + (size_t)b * br_plan_tps(p.M, p.H);
        const bool table = it.pe > 1;
        const int nprev = it.nprev;
        const int f_end = it.ntiles > 0x3fffffff ? 0x7fffffff : it.f_lo + it.ntiles;
        struct Tile {
            int tok0, nvalid, key0, self;
        };
        int f = it.f_lo;
        auto next_tile = [&](Tile& t) -> bool {
            while (f < f_end) {
                const int fi = f++;
                t.self = fi >= nprev;
                t.key0 = 0;
                if (!t.self) {
                    if (table) {
                        t.tok0 = tiles_b[fi].x;
                        t.nvalid = tiles_b[fi].y;
                    } else {
                        t.tok0 = it.tok0 + fi * BR_BN;
                        t.nvalid = it.len0 - fi * BR_BN < BR_BN ? it.len0 - fi * BR_BN : BR_BN;
                    }
                } else {
                    t.key0 = (fi - nprev) * BR_BN;
                    if (t.key0 >= self_end) {
                        f = f_end;
                        return false;
                    }
                    t.tok0 = it.tok_m + t.key0;
                    t.nvalid = self_end - t.key0 < BR_BN ? self_end - t.key0 : BR_BN;
                }
                if (t.nvalid > 0) return true;
            }
            return false;
        };
        constexpr int RPI = 64 / CPR, NI = BR_BN / RPI;              // rows per DMA instruction, instructions per tile and tensor
        auto issue_tile = [&](const Tile& t, int buf) {              // rows past the tile's real keys are zeros
            unsigned lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const unsigned srow = lane_l / CPR, spiece = lane_l % CPR;
            const char* kt = kbase + 2 * (unsigned long long)p.k32_t * (unsigned)t.tok0;
            const char* vt = vbase + 2 * (unsigned long long)p.v32_t * (unsigned)t.tok0;
            auto offset = [&](unsigned stride, int r) { return r * 2 * (int)stride + (int)((spiece ^ row_swizzle(r)) << 4); };
            if (NWT != 0 && t.nvalid == BR_BN) {
#pragma unroll
                for (int j = 0; j < NI / (NWT ? NWT : 1); ++j) {
                    const int q = wave + j * NWT, r = q * RPI + srow;
                    dma16(kt, offset(p.k32_t, r), smem_lds + buf * stageB + q * 1024);
                    dma16(vt, offset(p.v32_t, r), smem_lds + buf * stageB + tileB + q * 1024);
                }
                return;
            }
#pragma unroll 1
            for (int q = wave; q < 2 * NI; q += NW) {
                const int j = q < NI ? q : q - NI, r = j * RPI + srow, at = buf * stageB + q * 1024;
                dma16_lanes(__builtin_amdgcn_ballot_w64(r < t.nvalid), uniform(q < NI ? kt : vt), offset(q < NI ? p.k32_t : p.v32_t, r), smem_lds + at);
                if (r >= t.nvalid) *reinterpret_cast<uint4*>(smem + at + lane_l * 16) = uint4{0u, 0u, 0u, 0u};
            }
        };

        // Q and dO of this wave's rows (lane = row, registers = dims), the rows' log-sum-exp and delta
        bf16x8 qf[NC], dof[NC];
        float lse_l = 0.f, delta_l = 0.f;
        Tile cur = {}, nxt = {};
        bool have = next_tile(cur);
        constexpr int NR = BR_RB / RPI;
        uint4 gq[NR], gd[NR], go[NR];
        const int last = len_m - 1 - row0;
        if (rb_active) {
            const int r = ln < last ? ln : last;       // rows past the block's end repeat its last row; their results are not stored
            const unsigned tok = (unsigned)(it.tok_m + row0);
            const char* qrow = reinterpret_cast<const char*>(p.q) +
                               2 * ((unsigned long long)p.q32_b * (unsigned)b + (unsigned long long)p.q32_h * (unsigned)head + (unsigned long long)p.q32_t * tok);
            const char* grow = reinterpret_cast<const char*>(p.dout) +
                               2 * ((unsigned long long)p.g32_b * (unsigned)b + (unsigned long long)p.g32_h * (unsigned)head + (unsigned long long)p.g32_t * tok);
            const char* orow = reinterpret_cast<const char*>(p.out) +
                               2 * ((unsigned long long)p.o32_b * (unsigned)b + (unsigned long long)p.o32_h * (unsigned)head + (unsigned long long)p.o32_t * tok);
            const long long li = (long long)b * p.lse_b + (long long)head * p.lse_h + tok + r;
            // Loaded whole rows at a time (lane = row j RPI + lane / CPR, piece lane % CPR), turned into operands through the
            // wave's part of the second buffer.  Straight into the operands' layout the 24 instructions take 16 bytes of each
            // of 32 rows twice, and held a wave for 9000 of an item's 41000 clocks.
            lse_l = p.lse[li];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const unsigned rr = j * RPI + lane / CPR, rc = (int)rr < last ? rr : last, o = lane % CPR * 16;
                gd[j] = ld16(grow + (rc * 2 * p.g32_t + o));         // (32-bit offsets from a uniform base)
                go[j] = ld16(orow + (rc * 2 * p.o32_t + o));
                gq[j] = ld16(qrow + (rc * 2 * p.q32_t + o));
            }
        }
        if (have) issue_tile(cur, 0);
        if (rb_active) {
            char* W = smem + stageB + wave * (BR_RB * rowB);
            auto to_operand = [&](const uint4 (&src)[NR], bf16x8 (&dst)[NC]) {     // (a wave's LDS operations complete in order)
#pragma unroll
                for (int j = 0; j < NR; ++j) {
                    const int rr = j * RPI + lane / CPR;
                    *reinterpret_cast<uint4*>(W + rr * rowB + ((lane % CPR ^ row_swizzle(rr)) << 4)) = src[j];
                }
                lds_fence();
#pragma unroll
                for (int c = 0; c < NC; ++c) dst[c] = as_bf16x8(ld16(W + ln * rowB + (((2 * c + lh) ^ row_swizzle(ln)) << 4)));
                lds_fence();
            };
            to_operand(gd, dof);
            // delta: the CPR lanes of a row sum their pieces' products, each ending up with one of the NR rows it has a piece of
            float d[NR];
#pragma unroll
            for (int j = 0; j < NR; ++j) {
                const bf16x8 x = as_bf16x8(go[j]), y = as_bf16x8(gd[j]);
                d[j] = 0.f;
#pragma unroll
                for (int e = 0; e < 8; ++e) d[j] += (float)x[e] * (float)y[e];
            }
#pragma unroll
            for (int n = NR / 2, m = 1; n > 0; n /= 2, m *= 2)
#pragma unroll
                for (int j = 0; j < n; ++j) {
                    const bool up = (lane & m) != 0;
                    const float keep = up ? d[2 * j + 1] : d[2 * j], send = up ? d[2 * j] : d[2 * j + 1];
                    d[j] = keep + __shfl_xor(send, m);
                }
            d[0] += __shfl_xor(d[0], CPR / 2);
            to_operand(gq, qf);
            // (d[2 j], d[2 j + 1] went to lanes by bit 0, and so on: lane % NR is the index of its row)
            float* Wf = reinterpret_cast<float*>(W);
            if (lane % CPR < NR) Wf[lane % NR * RPI + lane / CPR] = d[0];
            lds_fence();
            delta_l = Wf[ln];
            // every item of a row block computes the same delta; the one that starts the key walk publishes it (negated)
            // - where another XCD may be about to read it, past this one's L2
            if (it.f_lo == 0 && lh == 0 && ln <= last)
                __hip_atomic_store(p.delta + ((long long)b * p.lse_b + (long long)head * p.lse_h + it.tok_m + row0 + ln), -delta_l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) qf[c] = dof[c] = as_bf16x8(uint4{0u, 0u, 0u, 0u});
        }
        // everything requested so far is waited for here, so that the loop is entered with no load of the compiler's pending:
        // its waits inside the loop would also cover the tile requested ahead
        vm_wait<0>();
        draw();
        if (COUNT && it.f_lo == 0 && rb_active && lane == 0)         // (its delta is in memory)
            __hip_atomic_fetch_add(p.published + (((size_t)b * p.M + it.m) * p.Nkv + kvh) * BR_COUNTER_LINE, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(qf[c]), "+v"(dof[c]));
        asm volatile("" : "+v"(lse_l), "+v"(delta_l));

        const float scale_log2 = p.scale_log2;
        f32x16 dq[ND];              // lane = row, register v of block db = dim 32 db + 8 (v / 4) + 4 lh + v % 4
#pragma unroll
        for (int db = 0; db < ND; ++db) dq[db] = zero16();

        // 32 keys of a tile; those from lim (per row) on are hidden where masked.  The products in order: S (NC), dP (NC), dQ
        // (2 ND), their LDS operands through a ring of AHEAD registers, each requested AHEAD products before its use; the
        // exponentials pass under the dP products, half of what makes dS under those of dQ.  The order is fenced (see
        // dkv_tile).
        auto compute = [&](int at, bool masked, int lim) {
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int lh = lane_l >> 5, ln = lane_l & 31, s16 = lane_l & 15, crow = 4 * lh + (s16 >> 2);
            const int ra = at + ln * rowB + ((lh ^ row_swizzle(ln)) << 4);
            const int ca = at + crow * rowB + (((2 * ((lane_l >> 4) & 1) + ((s16 & 3) >> 1)) ^ row_swizzle(crow)) << 4) + (s16 & 1) * 8;
            constexpr int AHEAD = 6, N = 2 * NC + 2 * ND;
            auto operand = [&](int i) -> bf16x8 {
                if (i < 2 * NC) return *(lds_bf16x8*)((ra ^ (i % NC << 5)) + (i < NC ? 0 : tileB));
                const int j = i - 2 * NC, o = j / ND * 16 * rowB, c = ca ^ (j % ND << 6);
                s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(c + o));
                s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)((c ^ 32) + o + 8 * rowB));
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
            };
            bf16x8 x[AHEAD];
            f32x16 st = zero16(), dpt = zero16();
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) x[i] = operand(i);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                BR_SCHED_FENCE();
                st = mma(x[i % AHEAD], qf[i], st);
                x[i % AHEAD] = operand(i + AHEAD);
            }
            BR_SCHED_FENCE();
            if (masked) {
                const int rest = lim - 4 * lh;
                float hidden;
                asm volatile("v_mov_b32 %0, 0xff800000" : "=v"(hidden));
#pragma unroll
                for (int v = 0; v < 16; ++v) st[v] = 8 * (v >> 2) + (v & 3) >= rest ? hidden : st[v];
            }
            constexpr int PER = 16 / NC;
#pragma unroll
            for (int i = NC; i < 2 * NC; ++i) {
                BR_SCHED_FENCE();
                dpt = mma(x[i % AHEAD], dof[i - NC], dpt);
                if (i + AHEAD < N) x[i % AHEAD] = operand(i + AHEAD);
#pragma unroll
                for (int v = (i - NC) * PER; v < (i - NC + 1) * PER; ++v) st[v] = __builtin_amdgcn_exp2f(st[v] * scale_log2 - lse_l);
            }
            u32x4 w[2];
            auto ds_pair = [&](int v) { w[v >> 3][(v & 7) >> 1] = pack2(st[v] * (dpt[v] - delta_l), st[v + 1] * (dpt[v + 1] - delta_l)); };
            BR_SCHED_FENCE();
#pragma unroll
            for (int v = 0; v < 8; v += 2) ds_pair(v);
#pragma unroll
            for (int i = 2 * NC; i < N; ++i) {
                BR_SCHED_FENCE();
                const int s = (i - 2 * NC) / ND, db = (i - 2 * NC) % ND;
                dq[db] = mma(x[i % AHEAD], __builtin_bit_cast(bf16x8, w[s]), dq[db]);
                if (i + AHEAD < N) x[i % AHEAD] = operand(i + AHEAD);
                if (s == 0)
#pragma unroll
                    for (int v = 8 + db * (8 / ND); v < 8 + (db + 1) * (8 / ND); v += 2) ds_pair(v);
            }
            BR_SCHED_FENCE();
        };

        int buf = 0;
        while (have) {
            const bool have_next = next_tile(nxt);
            vm_wait<0>();                          // this wave's part of the tile has arrived ...
            lds_barrier();                         // ... and everyone's, and nobody reads the other buffer any more
            if (have_next) issue_tile(nxt, buf ^ 1);
            if (rb_active) {
                // 32-key halves this wave needs: limited by the real keys and, on the block's own keys, by the diagonal,
                // which cuts the half of the wave's own rows only (both start at multiples of 32)
                for (int kb = 0; kb < 2; ++kb) {
                    const int k0 = kb * 32, ahead = cur.self ? row0 - cur.key0 - k0 : 1;
                    if (k0 >= cur.nvalid || ahead < 0) break;
                    const bool diagonal = ahead == 0;
                    compute(smem_lds + buf * stageB + k0 * rowB, diagonal || cur.nvalid - k0 < 32, diagonal ? ln + 1 : cur.nvalid - k0);
                }
            }
            cur = nxt;
            have = have_next;
            buf ^= 1;
        }
        drawn();
        lds_barrier();                             // nobody reads the tiles any more
        if (!rb_active) return;
        // dQ of this wave's rows through LDS the wave has to itself (its operations there complete in order; 16-byte pieces
        // swizzled), so that an instruction writes whole rows
        {
            const BrBwdParams& p = args_now(args);
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int lane = lane_l, ln = lane & 31, lh = lane >> 5;
            char* W = smem + wave * (BR_RB * rowB);
            const float sc = p.scale;
            const int nrows = len_m - row0 < BR_RB ? len_m - row0 : BR_RB;
            if (it.slot < 0) {
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<uint2*>(W + ln * rowB + (((4 * db + q) ^ (ln & (CPR - 1))) << 4) + 8 * lh) =
                            uint2{pack2(dq[db][4 * q] * sc, dq[db][4 * q + 1] * sc), pack2(dq[db][4 * q + 2] * sc, dq[db][4 * q + 3] * sc)};
                lds_fence();
                const int r0 = lane / CPR, c = lane % CPR;
                __bf16* dst = reinterpret_cast<__bf16*>(p.dq) + (long long)b * p.dq_b + (long long)head * p.dq_h + (long long)(it.tok_m + row0 + r0) * p.dq_t + 8 * c;
#pragma unroll
                for (int j = 0; j < BR_RB / RPI; ++j) {
                    const int r = j * RPI + r0;
                    if (r < nrows) *reinterpret_cast<uint4*>(dst + (long long)j * RPI * p.dq_t) = ld16(W + r * rowB + ((c ^ (r & (CPR - 1))) << 4));
                }
            } else {
                // shared rows (the query block): added to [b][head][row of the block][D] fp32, half of the dims at a time
                constexpr int HD = D / 2, PM = HD / 4 - 1;
                float* W4 = reinterpret_cast<float*>(W);
                float* dst = p.dq32 + (((long long)b * p.Nq + head) * p.H + row0) * D;
#pragma unroll
                for (int h = 0; h < 2; ++h) {
#pragma unroll
                    for (int d2 = 0; d2 < ND / 2; ++d2)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const f32x16& a = dq[h * (ND / 2) + d2];
                            *reinterpret_cast<f32x4*>(W4 + ln * HD + (((8 * d2 + 2 * q + lh) ^ (ln & PM)) << 2)) = f32x4{a[4 * q] * sc, a[4 * q + 1] * sc, a[4 * q + 2] * sc, a[4 * q + 3] * sc};
                        }
                    lds_fence();
                    constexpr int RPA = 64 / HD;                     // rows an instruction covers
#pragma unroll 8
                    for (int j = 0; j < BR_RB / RPA; ++j) {
                        const int r = j * RPA + lane / HD, d = lane % HD;
                        if (r < nrows) unsafeAtomicAdd(dst + (long long)r * D + h * HD + d, W4[r * HD + (((d >> 2) ^ (r & PM)) << 2) + (d & 3)]);
                    }
                    lds_fence();
                }
            }
        }
    }

    // ---------------------------------------------------------------------------------------------------------
    // dK, dV of the four key groups of an item, whole head dim, one group (32 keys) per wave.  A step is 32 query rows of
    // one head: the four waves bring their Q and dO rows into a ring of three LDS buffers by DMA, two steps ahead (one
    // barrier per step), and each computes for its keys
    //     S = Q K^T, dP = dO V^T - delta   (A = rows from LDS, B = the wave's keys, kept in registers)
    //     dV += P^T dO, dK += dS^T Q       (P, dS in bf16 straight from the accumulators; dO, Q by transposing reads)
    // 32 MFMAs per wave and step against 40 KB of LDS reads.  Four groups to a set of rows because the DMA is what binds
    // otherwise: a CU takes 64 bytes a clock, and with two groups its eight waves spent 1000 of a step's 3700 clocks on it.
    // ---------------------------------------------------------------------------------------------------------
    static constexpr int rowsQ = BR_RB * rowB, statOff = 2 * rowsQ;       // a buffer: 32 rows of Q, of dO, their lse and -delta
    static constexpr int bufBytes = statOff + 512;
    static constexpr int waveBytes = 2 * rowsQ;                           // a wave's part outside the walk: its K and V, its results
    static constexpr int dkvLdsBytes = 3 * bufBytes > 4 * waveBytes ? 3 * bufBytes : 4 * waveBytes;
    // draw and drawn: called once by every wave, in the last step and after it, if the item has steps.  lost: called where results
    // are stored, whether they are to be NaN.
    template <typename F, typename F2, typename F3>
    static __device__ __forceinline__ void dkv_tile(BrBwdArgs args, const BrDkvItem& it, char* smem, F&& draw, F2&& drawn, F3&& lost) {
        if (it.len_m <= 0) return;               // no keys, no rows
        const BrBwdParams& p = args_now(args);
        // (per item values that the compiler cannot trace back: nothing derived from them is kept in registers across items)
        int tid = threadIdx.x;
        asm volatile("" : "+v"(tid));
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
        const int G = p.geom.G, b = it.b, kvh = it.kvh;
        const unsigned smem_lds = lds_addr_of(smem);

        // the wave's group: a prefix group (pre) or one of the block's own
        const int n_p = (it.len_p + BR_RB - 1) / BR_RB, n_own = (it.len_m + BR_RB - 1) / BR_RB;
        const int g = it.group + wave;
        const bool pre = g < n_p;
        const int key0 = (pre ? g : g - n_p) * BR_RB, key_len = pre ? it.len_p : it.len_m, key_tok = pre ? it.tok_p : it.tok_m;
        const int nkeys = key_len - key0 < BR_RB ? key_len - key0 : BR_RB;    // may be zero or less: nothing to compute

        // The steps: (row block, head) pairs, heads inner; the block's row blocks from the first one that sees the first
        // group, then, if there is an own group among the four, the query block's
        const int rb0 = it.group > n_p ? it.group - n_p : 0;
        const int n_self = n_own - rb0, n_rb = n_self + (it.group + 4 > n_p ? (it.len_q + BR_RB - 1) / BR_RB : 0);
        const int n_steps = n_rb * G;

        constexpr int RPI = 64 / CPR;                                // rows per DMA instruction
        // DMA of rows first .. first + RPI NJ - 1 of a 32-row tile of which nrows exist: one instruction per RPI rows,
        // whatever nrows is; rows that do not exist become zeros
        auto issue_rows = [&](auto nj, const char* base, unsigned stride, int first, int nrows, int at) {
            constexpr int NJ = decltype(nj)::value;
            // (the lane as a value of this step that the compiler cannot trace back: what is derived from it is not kept
            // in registers across the walk)
            unsigned lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const unsigned srow = lane_l / CPR, spiece = lane_l % CPR;
            const int row_bytes = 2 * (int)stride, step_bytes = RPI * row_bytes;
            const char* base1 = base + (long long)first * row_bytes;
            if (nrows >= BR_RB && step_bytes >= 1024 && NJ % 4 == 0) {
                // four instructions per address and LDS base: an instruction's constant offset moves both, so its lanes'
                // offsets are 1024 less each time (not below zero with rows at least D apart)
                int off[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) off[j] = srow * row_bytes + ((spiece ^ row_swizzle(j * RPI + srow)) << 4) + j * (step_bytes - 1024);
#pragma unroll
                for (int j = 0; j < NJ; j += 4) dma16x4(base1 + (long long)j * step_bytes, off, smem_lds + at + j * 1024);
            } else {
                unsigned z;
                asm volatile("v_mov_b32 %0, 0" : "=v"(z));           // (not four registers of zeros for the whole walk)
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int r = first + j * RPI + srow;
                    dma16_lanes(__builtin_amdgcn_ballot_w64(r < nrows), base, r * row_bytes + ((spiece ^ row_swizzle(r)) << 4), smem_lds + at + j * 1024);
                    if (r >= nrows) *reinterpret_cast<uint4*>(smem + at + j * 1024 + lane_l * 16) = uint4{z, z, z, z};
                }
            }
        };
        // The wave's keys as operands (lane = key, registers = dims; past the real keys zeros, whose sums nothing reads).
        // They come through the wave's own part of LDS.
        const unsigned long long tok = (unsigned)(key_tok + (nkeys > 0 ? key0 : 0));
#pragma unroll 1
        for (int t = 0; t < 2; ++t) {
            const unsigned s_b = t ? p.v32_b : p.k32_b, s_h = t ? p.v32_h : p.k32_h, s_t = t ? p.v32_t : p.k32_t;
            issue_rows(std::integral_constant<int, BR_RB / RPI>{}, uniform(reinterpret_cast<const char*>(t ? p.v : p.k) + 2 * ((unsigned long long)s_b * (unsigned)b + (unsigned long long)s_h * (unsigned)kvh + s_t * tok)),
                       s_t, 0, nkeys, wave * waveBytes + t * rowsQ);
        }
        bf16x8 kf[NC], vf[NC];
        vm_wait<0>();
        {
            const int ln = lane & 31, lh = lane >> 5;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int o = wave * waveBytes + ln * rowB + (((2 * c + lh) ^ row_swizzle(ln)) << 4);
                kf[c] = *reinterpret_cast<const bf16x8*>(smem + o);
                vf[c] = *reinterpret_cast<const bf16x8*>(smem + o + rowsQ);
            }
        }
        lds_barrier();                           // every wave has its keys: the row buffers take the place of what they lay in

        // A step's rows: wave w brings half w / 2 of the Q (w even) or dO rows, and the rows' log-sum-exp or negated delta
        // (both halves' waves the same).  Rows past the block's end are zeros: their P is 1, and what it multiplies - dO,
        // dP, delta - is zero.
        constexpr int NJ = BR_RB / RPI / 2, PER_STEP = NJ + 1;       // DMA instructions of a wave
        const int odd = wave & 1, half = wave >> 1;
        const unsigned row_h = odd ? p.g32_h : p.q32_h, row_s = odd ? p.g32_t : p.q32_t;
        const char* row_tb = odd ? reinterpret_cast<const char*>(p.dout) + 2 * (unsigned long long)p.g32_b * (unsigned)b
                                 : reinterpret_cast<const char*>(p.q) + 2 * (unsigned long long)p.q32_b * (unsigned)b;
        const float* stat_b = (odd ? p.delta : p.lse) + (long long)b * p.lse_b;
        const long long lse_h = p.lse_h;
        int d_rb = 0, d_hl = 0, d_buf = 0;                           // the step whose rows are requested next, and its buffer
        struct Request {
            const char* rows;
            const float* stat;
            int nrows, at;
        };
        auto next_request = [&]() -> Request {
            const bool q = d_rb >= n_self;
            const int r0 = (q ? d_rb - n_self : d_rb + rb0) * BR_RB, rest = (q ? it.len_q : it.len_m) - r0;
            const int tok0 = (q ? it.tok_q : it.tok_m) + r0, head = kvh * G + d_hl, at = d_buf * bufBytes;
            if (++d_hl >= G) d_hl = 0, ++d_rb;
            d_buf = d_buf == 2 ? 0 : d_buf + 1;
            return {uniform(row_tb + 2 * ((unsigned long long)row_h * (unsigned)head + (unsigned long long)row_s * (unsigned)tok0)),
                    uniform(stat_b + (long long)head * lse_h + tok0), rest < BR_RB ? rest : BR_RB, __builtin_amdgcn_readfirstlane(at)};
        };
        const int rows_at = odd * rowsQ + half * (rowsQ / 2), stat_at = statOff + odd * 256;
        auto issue_step = [&](const Request& rq) {
            issue_rows(std::integral_constant<int, NJ>{}, rq.rows, row_s, half * (BR_RB / 2), rq.nrows, rq.at + rows_at);
            int ln_l = lane & 31;
            asm volatile("" : "+v"(ln_l));
            dma4_lanes(__builtin_amdgcn_ballot_w64(ln_l < rq.nrows), rq.stat, ln_l * 4, smem_lds + rq.at + stat_at);
            if (rq.nrows < BR_RB && ln_l >= rq.nrows) *reinterpret_cast<float*>(smem + rq.at + stat_at + lane * 4) = 0.f;
        };

        const float scale_log2 = p.scale_log2;
        f32x16 dk[ND], dv[ND];      // lane = key, register v of block db = dim 32 db + 8 (v / 4) + 4 lh + v % 4
#pragma unroll
        for (int db = 0; db < ND; ++db) dk[db] = dv[db] = zero16();
        // Where the step after next's rows are a whole 32, their DMAs (rq; more is -1, or 0: there are none) are issued from
        // inside the computation, spread over its products: a CU takes 32 bytes a clock, and issued together after the
        // barrier they kept every wave waiting for 600 of a step's 3300 clocks.
        auto compute = [&](int buf, bool diagonal, int more, const Request& rq) {
            // LDS addresses of the operand reads: row reads of piece 2c + lh are ra ^ (c << 5); transposing reads of block db,
            // rows 16 s + 4 lh + 0..3 are ca ^ (db << 6), 16 s rows further, and those of the rows eight further the same
            // ^ 32 and 8 rows further.  From a lane index that the compiler cannot trace back: none of the sixteen
            // addresses is then kept in registers across the walk.
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int base = smem_lds + buf * bufBytes, lh = lane_l >> 5, ln = lane_l & 31, s16 = lane_l & 15, crow = 4 * lh + (s16 >> 2);
            const int ra = base + ln * rowB + ((lh ^ row_swizzle(ln)) << 4);
            const int ca = base + crow * rowB + (((2 * ((lane_l >> 4) & 1) + ((s16 & 3) >> 1)) ^ row_swizzle(crow)) << 4) + (s16 & 1) * 8;
            int rd = ra + rowsQ;
            int cd = ca;
            asm volatile("" : "+v"(rd), "+v"(cd));
            const int la = base + statOff + 16 * lh;
            // The step's products in order: S (NC), dV (2 ND), dP (NC), dK (2 ND) - an order in which P in fp32, P in bf16 and
            // dP never need registers at once.  Their LDS operands go through a ring of AHEAD registers, each requested
            // AHEAD products before its use; half of the exponentials pass under dV products, half of what makes dS of P
            // and dP under those of dK.  The order is fenced: left to itself the compiler's scheduler gathers reads and
            // products until each waits for its own operand, or spills.
            constexpr int AHEAD = 3, N = 2 * NC + 4 * ND, NP = NC + 2 * ND;
            auto operand = [&](int i) -> bf16x8 {
                const int j = i % NP;
                if (j < NC) return *(lds_bf16x8*)((i < NP ? ra : rd) ^ (j << 5));
                const int s = (j - NC) / ND, db = (j - NC) % ND, o = s * 16 * rowB + (i < NP ? rowsQ : 0);
                s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(((i < NP ? ca : cd) ^ (db << 6)) + o));
                s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(((i < NP ? ca : cd) ^ (db << 6) ^ 32) + o + 8 * rowB));
                return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
            };
            auto dma_slot = [&](int i) {
                constexpr int EVERY = N / PER_STEP;
                if (i % EVERY != 2 || i / EVERY >= PER_STEP) return;
                const int j = i / EVERY;
                unsigned lane_d = lane;
                asm volatile("" : "+v"(lane_d));
                if (j < NJ) {
                    const unsigned srow = lane_d / CPR;
                    dma16_if(more, rq.rows + (unsigned long long)((half * (BR_RB / 2) + j * RPI) * 2) * row_s,
                             (int)(srow * 2 * row_s + ((lane_d % CPR ^ row_swizzle(j * RPI + srow)) << 4)), smem_lds + rq.at + rows_at + j * 1024);
                } else {
                    dma4_if(more, rq.stat, (int)(lane_d & 31) * 4, smem_lds + rq.at + stat_at);
                }
            };
            bf16x8 x[AHEAD];
            f32x16 sc = zero16(), dp;
            float lse[8];                            // of half of the accumulator's rows at a time
            auto load_lse = [&](int s) {
#pragma unroll
                for (int v4 = 0; v4 < 2; ++v4) {
                    const f32x4 t = *(lds_f32x4*)(la + 64 * s + 32 * v4);
                    lse[4 * v4] = t[0]; lse[4 * v4 + 1] = t[1]; lse[4 * v4 + 2] = t[2]; lse[4 * v4 + 3] = t[3];
                }
            };
            auto load_stat = [&](f32x16& c, int at) {
#pragma unroll
                for (int v4 = 0; v4 < 4; ++v4) {
                    const f32x4 t = *(lds_f32x4*)(at + 32 * v4);
                    c[4 * v4] = t[0]; c[4 * v4 + 1] = t[1]; c[4 * v4 + 2] = t[2]; c[4 * v4 + 3] = t[3];
                }
            };
            load_lse(0);
#pragma unroll
            for (int i = 0; i < AHEAD; ++i) x[i] = operand(i);
#pragma unroll
            for (int i = 0; i < NC; ++i) {
                BR_SCHED_FENCE();
                sc = mma(x[i % AHEAD], kf[i], sc);
                x[i % AHEAD] = operand(i + AHEAD);
                dma_slot(i);
            }
            BR_SCHED_FENCE();
            if (diagonal) {              // the wave's own 32 rows: key ln is hidden from the rows before it
                const int first = ln - 4 * lh;
                float hidden;
                asm volatile("v_mov_b32 %0, 0xff800000" : "=v"(hidden));
#pragma unroll
                for (int v = 0; v < 16; ++v) sc[v] = 8 * (v >> 2) + (v & 3) < first ? hidden : sc[v];
            }
            u32x4 w[2];                              // P, then dS, in bf16
            auto exp2_pair = [&](int v) {
                sc[v] = __builtin_amdgcn_exp2f(sc[v] * scale_log2 - lse[v & 7]);
                sc[v + 1] = __builtin_amdgcn_exp2f(sc[v + 1] * scale_log2 - lse[(v & 7) + 1]);
                w[v >> 3][(v & 7) >> 1] = pack2(sc[v], sc[v + 1]);
            };
            auto ds_pair = [&](int v) { w[v >> 3][(v & 7) >> 1] = pack2(sc[v] * dp[v], sc[v + 1] * dp[v + 1]); };
#pragma unroll
            for (int v = 0; v < 8; v += 2) exp2_pair(v);
            load_lse(1);
#pragma unroll
            for (int i = NC; i < NP; ++i) {
                BR_SCHED_FENCE();
                const int s = (i - NC) / ND, db = (i - NC) % ND;
                dv[db] = mma(x[i % AHEAD], __builtin_bit_cast(bf16x8, w[s]), dv[db]);
                x[i % AHEAD] = operand(i + AHEAD);
                dma_slot(i);
                if (s == 0)
#pragma unroll
                    for (int v = 8 + db * (8 / ND); v < 8 + (db + 1) * (8 / ND); v += 2) exp2_pair(v);
            }
            BR_SCHED_FENCE();
            load_stat(dp, la + 256);
#pragma unroll
            for (int i = NP; i < NP + NC; ++i) {
                BR_SCHED_FENCE();
                dp = mma(x[i % AHEAD], vf[i - NP], dp);
                x[i % AHEAD] = operand(i + AHEAD);
                dma_slot(i);
            }
            BR_SCHED_FENCE();
#pragma unroll
            for (int v = 0; v < 8; v += 2) ds_pair(v);
#pragma unroll
            for (int i = NP + NC; i < N; ++i) {
                BR_SCHED_FENCE();
                const int s = (i - NP - NC) / ND, db = (i - NP - NC) % ND;
                dk[db] = mma(x[i % AHEAD], __builtin_bit_cast(bf16x8, w[s]), dk[db]);
                if (i + AHEAD < N) x[i % AHEAD] = operand(i + AHEAD);
                dma_slot(i);
                if (s == 0)
#pragma unroll
                    for (int v = 8 + db * (8 / ND); v < 8 + (db + 1) * (8 / ND); v += 2) ds_pair(v);
            }
            BR_SCHED_FENCE();
        };

#pragma unroll 1
        for (int i = 0; i < 2 && i < n_steps; ++i) issue_step(next_request());
        int buf = 0, rb = 0, hl = 0;
        for (int i = 0; i < n_steps; ++i) {
            if (i + 1 < n_steps) vm_wait<PER_STEP>();    // this wave's part of the step's rows has arrived (the next step's may not have) ...
            else vm_wait<0>();
            lds_barrier();                       // ... and everyone's, and nobody reads the buffer of the step before any more
            if (i + 1 == n_steps) draw();        // (nothing else is in flight then that its value would be waited for with)
            // own groups: the row blocks before the group's own do not see it, that one is cut by the diagonal; prefix groups
            // are seen by all rows of the block (and not by these query rows: the query block's own items have them)
            const int ahead = rb < n_self ? (rb + rb0) * BR_RB - key0 : 1;
            const bool work = nkeys > 0 && (pre ? rb < n_self : ahead >= 0), more = i + 2 < n_steps;
            const Request rq = next_request();                   // (past the last step: not used)
            const bool later = more && work && rq.nrows == BR_RB;
            if (more && !later) issue_step(rq);
            if (work) compute(buf, !pre && ahead == 0, __builtin_amdgcn_readfirstlane(later ? -1 : 0), rq);
            if (++hl >= G) hl = 0, ++rb;
            buf = buf == 2 ? 0 : buf + 1;
        }

        if (n_steps > 0) drawn();
        lds_barrier();                           // nobody reads the rows any more
        // One tensor's sums of the wave's keys, through LDS the wave has to itself (its operations there complete in order;
        // 16-byte pieces swizzled), so that an instruction writes whole rows
        const bool to_sums = pre || it.m == 0 && p.M > 1;        // prefix keys, which more blocks see
        auto put = [&](f32x16 (&acc)[ND], bool is_k, char* T) {
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int lane = lane_l, ln = lane & 31, lh = lane >> 5;
            const BrBwdParams& p = args_now(args);
            const float f = lost() ? __builtin_nanf("") : is_k ? p.scale : 1.f;
            if (to_sums) {
                // prefix keys: added to the fp32 sums
                constexpr int PM = D / 4 - 1 < 31 ? D / 4 - 1 : 31;
                float* T4 = reinterpret_cast<float*>(T);
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<f32x4*>(T4 + ln * D + (((8 * db + 2 * q + lh) ^ (ln & PM)) << 2)) =
                            f32x4{acc[db][4 * q] * f, acc[db][4 * q + 1] * f, acc[db][4 * q + 2] * f, acc[db][4 * q + 3] * f};
                lds_fence();
                float* dst = (is_k ? p.dk32 : p.dv32) + (((long long)b * p.Nkv + kvh) * p.H + key0) * D;
#pragma unroll
                for (int k0 = 0; k0 < BR_RB; k0 += 8) {          // eight keys' reads ahead of their additions
                    float t[8][D / 64];
#pragma unroll
                    for (int k = 0; k < 8; ++k)
#pragma unroll
                        for (int h = 0; h < D / 64; ++h) {
                            const int d = lane + 64 * h;
                            t[k][h] = T4[(k0 + k) * D + (((d >> 2) ^ ((k0 + k) & PM)) << 2) + (d & 3)];
                        }
#pragma unroll
                    for (int k = 0; k < 8; ++k)
#pragma unroll
                        for (int h = 0; h < D / 64; ++h)
                            if (k0 + k < nkeys) unsafeAtomicAdd(dst + (long long)(k0 + k) * D + lane + 64 * h, t[k][h]);
                }
            } else {
                // one owner: stored in bf16
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        *reinterpret_cast<uint2*>(T + ln * rowB + (((4 * db + q) ^ (ln & (CPR - 1))) << 4) + 8 * lh) =
                            uint2{pack2(acc[db][4 * q] * f, acc[db][4 * q + 1] * f), pack2(acc[db][4 * q + 2] * f, acc[db][4 * q + 3] * f)};
                lds_fence();
                const long long dt = is_k ? p.dk_t : p.dv_t;
                const int r0 = lane / CPR, c = lane % CPR;
                __bf16* dst = (is_k ? reinterpret_cast<__bf16*>(p.dk) + (long long)b * p.dk_b + (long long)kvh * p.dk_h
                                    : reinterpret_cast<__bf16*>(p.dv) + (long long)b * p.dv_b + (long long)kvh * p.dv_h) + (long long)(key_tok + key0 + r0) * dt + 8 * c;
#pragma unroll
                for (int j = 0; j < BR_RB / RPI; ++j) {
                    const int r = j * RPI + r0;
                    if (r < nkeys) *reinterpret_cast<uint4*>(dst + (long long)j * RPI * dt) = ld16(T + r * rowB + ((c ^ (r & (CPR - 1))) << 4));
                }
            }
            lds_fence();
        };
        if (nkeys > 0) {
#pragma unroll 1
            for (int t = 0; t < 2; ++t) {                        // (a loop for the size of the code)
                put(dk, t == 0, smem + wave * waveBytes);
#pragma unroll
                for (int db = 0; db < ND; ++db) dk[db] = dv[db];
            }
        }
    }
};

// Persistent over the plan's items (times head groups), like the prefill kernel: a workgroup draws tickets from its XCD's
// queue, then from the global one, with ALL then from the others'.  ALL: dK and dV follow in the same launch.  Then a workgroup leaves only when no queue has a
// ticket left, and none is handed out by workgroup index: whoever waits for a delta afterwards waits for workgroups that run.
template <int D, int MAXW, bool ALL>
__device__ __forceinline__ void dq_loop(BrBwdArgs args, char* smem) {
    __shared__ int s_mail[2][BR_ITEM_INTS + 2];
    __shared__ int s_ticket;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = blockIdx.x & 7, nx = ALL ? 0 : ((int)gridDim.x - x + 7) >> 3;
    int queue = x;                                   // BR_GLOBAL_QUEUE: the own queue is dry (wave 0)
    auto draw = [&]() { const BrBwdParams& p = args_now(args); return atomicAdd(p.tickets + (8 + queue) * p.ticket_step, 1); };
    auto ticket_of = [&](int drawn) { return drawn + (queue == BR_GLOBAL_QUEUE ? 0 : nx); };      // (where the value is used: adding waits for it)
    auto look_up = [&](int t, int* mail) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const BrBwdParams& p = args_now(args);
        typedef const __attribute__((address_space(4))) int* plan_words;
        const plan_words hdr = (plan_words)p.plan;
        const int nhg = p.geom.NHG;
        if (queue == x && t >= hdr[BR_PH_QCOUNT + x] * nhg) {
            queue = BR_GLOBAL_QUEUE;
            t = 0x7fffffff;
            if (hdr[BR_PH_QCOUNT + queue] > 0) {
                if (lane == 0) t = draw();
                t = __builtin_amdgcn_readfirstlane(t);
            }
        }
        while (t >= hdr[BR_PH_QCOUNT + queue] * nhg) {
            unsigned left = 0;
            if (ALL) {                                   // another XCD's queue, the next one that has tickets
                const int i = lane < 8 ? lane + x & 7 : 0;
                const int at = __hip_atomic_load(p.tickets + (8 + i) * p.ticket_step, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                left = (unsigned)__builtin_amdgcn_ballot_w64(lane < 8 && at < p.plan[BR_PH_QCOUNT + i] * nhg);
            }
            if (left == 0) {
                if (lane == 0) mail[BR_ITEM_INTS + 1] = 0;
                return;
            }
            queue = (__builtin_ctz(left) + x) & 7;
            if (lane == 0) t = draw();
            t = __builtin_amdgcn_readfirstlane(t);
        }
        const int li = t / nhg;
        const plan_words item = hdr + br_plan_off_items(p.B, p.M, p.H, p.geom.tpb * BR_RB) + (size_t)(hdr[BR_PH_QOFF + queue] + li) * BR_ITEM_INTS;
        int v = 1;
#pragma unroll
        for (int i = 0; i < BR_ITEM_WORDS_USED; ++i) v = lane == i ? item[i] : v;
        v = lane == BR_ITEM_INTS ? t - li * nhg : v;
        if (lane < BR_ITEM_INTS + 2) mail[lane] = v;
    };
    // (the first round has no item: it looks up the first one, whose ticket is the workgroup's index, or with ALL drawn)
    if (threadIdx.x == 0) s_ticket = ALL ? draw() : blockIdx.x >> 3;
    if (threadIdx.x < BR_ITEM_INTS + 2) s_mail[0][threadIdx.x] = threadIdx.x == BR_ITEM_INTS + 1 ? 2 : 0;
    __syncthreads();
    for (int cur = 0;; cur ^= 1) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int word = s_mail[cur][lane < BR_ITEM_INTS + 2 ? lane : 0];
#define BR_W(i) __builtin_amdgcn_readlane(word, i)
        const int state = BR_W(BR_ITEM_INTS + 1);       // 0: no more, 2: no item yet
        if (state == 0) break;
        BrItem it;
        it.b = BR_W(0); it.m = BR_W(1); it.t0 = BR_W(2); it.f_lo = BR_W(3); it.nprev = BR_W(4); it.ntiles = BR_W(5); it.slot = BR_W(6);
        it.pe = BR_W(7); it.len_m = BR_W(8); it.start_m = BR_W(9); it.len0 = BR_W(10); it.start0 = BR_W(11); it.tok_m = BR_W(12);
        it.tok0 = BR_W(13);
        it.pad[0] = it.pad[1] = 0;
        const int hg = BR_W(BR_ITEM_INTS);
#undef BR_W
        // the ticket of the next item is drawn when this one's rows are there, and looked up when its walk is over
        int drawn = 0;
        if (state == 1)
            Bwd<D>::template dq_item<MAXW == 4 ? 4 : 0, ALL>(args, it, hg, (int)blockDim.x >> 6, smem, [&]() { if (threadIdx.x == 0) drawn = draw(); },
                                                        [&]() { if (threadIdx.x == 0) s_ticket = ticket_of(drawn); });
        if (wave == 0) look_up(__builtin_amdgcn_readfirstlane(s_ticket), s_mail[cur ^ 1]);
        lds_barrier();
    }
}

// All items of one (block m, sequence, kv head) read the same Q and dO rows: they form a set.  Sets are dealt to eight queues, one per XCD
// (each has its own L2, and workgroups are placed on them round robin by index), so that a set's rows are fetched into
// one L2; a queue's sets have the kv heads in turn, or its XCD would use the L2 channels of one head's addresses only.
// The grid is persistent and draws tickets from its queue: with a workgroup per item the dispatcher, which deals
// workgroups to an XCD's four shader engines strictly in turn and waits for the engine whose turn it is, kept only half of
// the wave slots busy (items last 5 to 80 us; 101 us where the items' own times add up to 35).
// ALL: behind dQ in the same launch.  An item is then started when the deltas of its rows are there - published counts a (block,
// kv head)'s (32 rows, query head) pairs -, and every ticket is drawn: a workgroup that is still at dQ holds none.
template <int D, bool ALL>
__device__ __forceinline__ void dkv_loop(BrBwdArgs args, char* smem) {
    __shared__ int s_set[7][64], s_mail[2][16];
    __shared__ int s_ticket;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x = blockIdx.x & 7, nx = ALL ? 0 : ((int)gridDim.x - x + 7) >> 3;
    auto published = [&](const BrBwdParams& p, int b, int m, int kvh) {
        return __hip_atomic_load(p.published + (((size_t)b * p.M + m) * p.Nkv + kvh) * BR_COUNTER_LINE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto draw = [&]() { const BrBwdParams& p = args_now(args); return atomicAdd(p.tickets + x * p.ticket_step, 1); };
    // Wave 0 looks tickets up in windows of the queue's sets (tickets come in rising order, so it only moves forward); lane i
    // of s_set: set w_set + i.  Inside a window the items come in the order of the row blocks they walk, longest first.
    // Windows are small, so that the items of a set still run at about the same time, but the last one is as large as it
    // can be: what runs last is short.
    int w_set = 0, w_first = 0, w_total = 0, w_size = 0, w_rows = 0;
    auto look_up = [&](int t, int* mail) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const BrBwdParams& p = args_now(args);
        const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.geom.tpb * BR_RB);
        const int M = p.M;
        while (t >= w_first + w_total) {
            w_set += w_size;
            w_first += w_total;
            const int left = (M * p.B * p.Nkv - x + 7) / 8 - w_set;
            if (left <= 0) {
                if (lane == 0) mail[0] = 0;
                return;
            }
            w_size = left <= 64 ? left : 16;
            const int g = (w_set + lane) * 8 + x, blk = g / p.Nkv, b = blk % p.B, mg = blk / p.B;
            int n = 0, n_own = 0, n_p = 0;
            if (lane < w_size) {
                n_own = (pv.len[b * M + mg] + BR_RB - 1) / BR_RB;
                if (n_own > 0 && mg > 0) n_p = (pv.len[b * M] + BR_RB - 1) / BR_RB;
                n = n_own + n_p > 4 ? (n_own + n_p + 3) / 4 : 1;     // (a block without tokens still has padded slots to clear)
                s_set[0][lane] = (g + blk) % p.Nkv;
                s_set[1][lane] = b;
                s_set[2][lane] = mg;
                if (ALL)
                    s_set[6][lane] = p.max_looks > 0 && published(p, b, mg, (g + blk) % p.Nkv) >= n_own * p.geom.G &&
                                     (mg == 0 || published(p, b, M - 1, (g + blk) % p.Nkv) >= (pv.len[b * M + M - 1] + BR_RB - 1) / BR_RB * p.geom.G);
            }
            s_set[3][lane] = n_own;
            s_set[4][lane] = n_p;
            s_set[5][lane] = n;
            w_rows = n_own;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                n += __shfl_xor(n, d);
                const int o = __shfl_xor(w_rows, d);
                w_rows = o > w_rows ? o : w_rows;
            }
            w_total = __builtin_amdgcn_readfirstlane(n);
            w_rows = __builtin_amdgcn_readfirstlane(w_rows);
            if (ALL) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        // the set's item that walks rows row blocks of the block, or -1: item c starts with own group 4 c - n_p, whose first
        // row block that is
        const int n_own = s_set[3][lane], n_p = s_set[4][lane], n = s_set[5][lane];
        int local = t - w_first, rows = w_rows, chunk;
        unsigned long long have;
        for (;; --rows) {
            // items 0 .. n_p / 4 walk all of the block's rows
            const int full = n_p / 4 + 1 < n ? n_p / 4 + 1 : n, first = n_own - rows + n_p;
            int mine = 0;
            chunk = 0;
            if (rows == n_own) mine = full;
            else if (rows < n_own && first % 4 == 0 && first / 4 < n) mine = 1, chunk = first / 4;
            for (;;) {
                have = __builtin_amdgcn_ballot_w64(mine > 0);
                const int c = __popcll(have);
                if (local < c || c == 0) break;
                local -= c;
                --mine;
                ++chunk;
            }
            if (have != 0) break;
        }
        const bool here = (have >> lane & 1) != 0 && __builtin_amdgcn_mbcnt_hi((unsigned)(have >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)have, 0u)) == (unsigned)local;
        const int pos = __builtin_ctzll(__builtin_amdgcn_ballot_w64(here));
        chunk = __builtin_amdgcn_readlane(chunk, pos);
        const int kvh = __builtin_amdgcn_readfirstlane(s_set[0][pos]), b = __builtin_amdgcn_readfirstlane(s_set[1][pos]), mg = __builtin_amdgcn_readfirstlane(s_set[2][pos]);
        // (scalar loads: vector ones would be waited for behind the DMAs in flight)
        typedef const __attribute__((address_space(4))) int* plan_words;
        const plan_words lens = (plan_words)pv.len + b * M, toks = (plan_words)pv.tok + b * M, starts = (plan_words)pv.start + b * M;
        const bool doc = mg > 0 && mg < M - 1;
        int lost = 0;
        if (ALL && !__builtin_amdgcn_readfirstlane(s_set[6][pos])) {
            // Every ticket of dQ is with a workgroup that is running its item or the one before.  (The bound only keeps a
            // workspace that two passes share by mistake from holding the GPU.  What an item that gives up would store was
            // not computed from its rows' deltas: it stores NaN, which whoever reads the gradients sees.)
            const int own = (lens[mg] + BR_RB - 1) / BR_RB * p.geom.G, behind = mg > 0 ? (lens[M - 1] + BR_RB - 1) / BR_RB * p.geom.G : 0;
            lost = 1;
            for (int i = 0; i < p.max_looks; ++i) {
                if (__builtin_amdgcn_readfirstlane(published(p, b, mg, kvh) >= own && published(p, b, M - 1, kvh) >= behind)) {
                    lost = 0;
                    break;
                }
                __builtin_amdgcn_s_sleep(8);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        const int w[kDkvItemWords + 1] = {1, b, kvh, mg, chunk * 4, lens[mg], toks[mg], starts[mg], mg > 0 ? lens[0] : 0, toks[0], doc ? lens[M - 1] : 0, toks[M - 1], lost};
        int v = 0;
#pragma unroll
        for (int i = 0; i <= kDkvLost; ++i) v = lane == i ? w[i] : v;
        if (lane <= kDkvLost) mail[lane] = v;
    };
    // (the first round has no item: it looks up the first one, by the workgroup's index or with ALL by a ticket that it draws)
    if (threadIdx.x < 16) s_mail[0][threadIdx.x] = threadIdx.x == 0 ? 2 : 0;
    __syncthreads();
    for (int cur = 0;; cur ^= 1) {
        int lane = threadIdx.x & 63;
        asm volatile("" : "+v"(lane));
        const int word = s_mail[cur][lane < kDkvItemWords ? lane : 0];
        BrDkvItem it;
#define BR_W(i) __builtin_amdgcn_readlane(word, i)
        it.valid = BR_W(0); it.b = BR_W(1); it.kvh = BR_W(2); it.m = BR_W(3); it.group = BR_W(4); it.len_m = BR_W(5); it.tok_m = BR_W(6); it.start_m = BR_W(7);
        it.len_p = BR_W(8); it.tok_p = BR_W(9); it.len_q = BR_W(10); it.tok_q = BR_W(11);
#undef BR_W
        if (!it.valid) break;
        // padded slots of the block (dk and dv of this kv head): zeros, written with the block's first item
        if (it.valid == 1 && it.group == 0 && !args_now(args).plan[BR_PH_PACKED]) {
            const BrBwdParams& p = args_now(args);
            const int st = it.start_m, len_m = it.len_m, npad = p.H - len_m;
            constexpr int CP8 = D / 8;
            const uint4 z = {0u, 0u, 0u, 0u};
            __bf16* kb_ = reinterpret_cast<__bf16*>(p.dk) + (long long)it.b * p.dk_b + (long long)it.kvh * p.dk_h;
            __bf16* vb_ = reinterpret_cast<__bf16*>(p.dv) + (long long)it.b * p.dv_b + (long long)it.kvh * p.dv_h;
            int tid = threadIdx.x;
            asm volatile("" : "+v"(tid));
            for (int i = tid; i < npad * CP8; i += 256) {
                const int r = i / CP8, c8 = i - r * CP8;
                const long long pos = (long long)it.m * p.H + (r < st ? r : r + len_m);
                *reinterpret_cast<uint4*>(kb_ + pos * p.dk_t + c8 * 8) = z;
                *reinterpret_cast<uint4*>(vb_ + pos * p.dv_t + c8 * 8) = z;
            }
        }
        // The ticket of the next item is drawn in the last step of this one: drawn an item or two ahead, a workgroup kept it
        // through an item of 50 us and more while others had run out of work.
        int drawn = 0;
        if (threadIdx.x == 0) s_ticket = it.valid == 2 && !ALL ? blockIdx.x >> 3 : -1;
        if (it.valid == 1)
            Bwd<D>::dkv_tile(args, it, smem, [&]() { if (threadIdx.x == 0) drawn = draw(); }, [&]() { if (threadIdx.x == 0) s_ticket = drawn + nx; },
                             [&]() { return ALL && s_mail[cur][kDkvLost] != 0; });
        if (wave == 0) {
            int t = __builtin_amdgcn_readfirstlane(s_ticket);
            if (t < 0) t = __builtin_amdgcn_readfirstlane(threadIdx.x == 0 ? draw() : 0) + nx;        // (an item without steps)
            look_up(t, s_mail[cur ^ 1]);
        }
        lds_barrier();
    }
}

template <int D, int MAXW>
__global__ __launch_bounds__(MAXW * 64, 2) void br_bwd_dq_kernel(BrBwdParams) {
    // (one object, at LDS address 0: the DMA's targets, the tile buffers, are at most 64 KiB)
    __shared__ __attribute__((aligned(1024))) char smem[Bwd<D>::dqLdsBytes(MAXW)];
    dq_loop<D, MAXW, false>((BrBwdArgs)__builtin_amdgcn_kernarg_segment_ptr(), smem);
}

template <int D>
__global__ __launch_bounds__(256, 2) void br_bwd_dkv_kernel(BrBwdParams) {
    // (one object, at LDS address 0: the DMA's targets, the row buffers, are below 64 KiB)
    __shared__ __attribute__((aligned(1024))) char smem[Bwd<D>::dkvLdsBytes];
    dkv_loop<D, false>((BrBwdArgs)__builtin_amdgcn_kernarg_segment_ptr(), smem);
}

// Both in one launch, where a (block, kv head)'s keys wait for its own rows' deltas only, which a dQ item publishes before its
// walk: dQ's last items no longer leave the chip half empty, nor does the start of a second launch.  Each counter, of tickets and
// of deltas, has a cache line of its own: an XCD that counts takes the line from the others.  The whole step, forward included,
// 32/8 heads, D = 128, two launches with the tickets in one line / with a line each / this one: 4 x 20 documents of 160 tokens
// 348.5 / 348.0 / 341.2 us, 2 x 16 of 256 to 512 485 / 485 / 467, runs differing by 0.2 %; one launch with all tickets in one line
// took 382 us for the first where this one took 355, with the deltas' counters packed 356 where it took 348.
template <int D>
__global__ __launch_bounds__(256, 2) void br_bwd_kernel(BrBwdParams) {
    const BrBwdArgs args = (BrBwdArgs)__builtin_amdgcn_kernarg_segment_ptr();
    constexpr int DQ = Bwd<D>::dqLdsBytes(4), DKV = Bwd<D>::dkvLdsBytes;
    __shared__ __attribute__((aligned(1024))) char smem[DQ > DKV ? DQ : DKV];
    dq_loop<D, 4, true>(args, smem);
    dkv_loop<D, true>(args, smem);
}

// Clears n16 16-byte pieces and the n_counters ticket counters (and counters of published deltas)
__global__ __launch_bounds__(256) void br_fill_zero_kernel(uint4* p, size_t n16, int* counters, size_t n_counters) {
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n_counters; i += (size_t)gridDim.x * blockDim.x) counters[i] = 0;
    const uint4 z = {0u, 0u, 0u, 0u};
    for (size_t i = blockIdx.x * (size_t)blockDim.x + threadIdx.x; i < n16; i += (size_t)gridDim.x * blockDim.x) p[i] = z;
}

// dQ of the rows whose key walk was split (the plan's combine list names their query tiles): fp32 sums -> bf16;
// and zeros for the padded slots of dq.
template <int D>
__global__ __launch_bounds__(256) void br_bwd_dq_finish_kernel(BrBwdParams p) {
    const BrGeom& ge = p.geom;
    const int T = ge.tpb * BR_RB;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, T);
    constexpr int C4 = D / 4;
    const int m = p.M - 1;
    const long long n = (long long)pv.hdr[BR_PH_NCOMB] * p.Nq * T * C4;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const int c = (int)(i % C4);
        long long r = i / C4;
        const int row_in = (int)(r % T);
        r /= T;
        const int head = (int)(r % p.Nq), ci = (int)(r / p.Nq);
        const BrComb cb = pv.comb[ci];
        const int row = cb.t0 + row_in;
        if (row >= pv.len[cb.b * p.M + m]) continue;
        const f32x4 x = *reinterpret_cast<const f32x4*>(p.dq32 + (((long long)cb.b * p.Nq + head) * p.H + row) * D + c * 4);
        __bf16* dst = reinterpret_cast<__bf16*>(p.dq) + (long long)cb.b * p.dq_b + (long long)head * p.dq_h +
                      (long long)(pv.tok[cb.b * p.M + m] + row) * p.dq_t + c * 4;
        *reinterpret_cast<bf16x4*>(dst) = __builtin_convertvector(x, bf16x4);
    }
    // dK, dV of the prefix keys (summed over the workgroups of every viewing block)
    if (p.M > 1) {
        const long long nk = (long long)p.B * p.Nkv * p.H * C4;
        for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < nk; i += (long long)gridDim.x * blockDim.x) {
            const int c = (int)(i % C4);
            long long r = i / C4;
            const int key = (int)(r % p.H);
            r /= p.H;
            const int kvh = (int)(r % p.Nkv), b = (int)(r / p.Nkv);
            if (key >= pv.len[b * p.M]) continue;
            const long long src = (((long long)b * p.Nkv + kvh) * p.H + key) * D + c * 4;
            const long long tokk = pv.tok[b * p.M] + key;
            *reinterpret_cast<bf16x4*>(reinterpret_cast<__bf16*>(p.dk) + (long long)b * p.dk_b + (long long)kvh * p.dk_h + tokk * p.dk_t + c * 4) =
                __builtin_convertvector(*reinterpret_cast<const f32x4*>(p.dk32 + src), bf16x4);
            *reinterpret_cast<bf16x4*>(reinterpret_cast<__bf16*>(p.dv) + (long long)b * p.dv_b + (long long)kvh * p.dv_h + tokk * p.dv_t + c * 4) =
                __builtin_convertvector(*reinterpret_cast<const f32x4*>(p.dv32 + src), bf16x4);
        }
    }
    if (pv.hdr[BR_PH_PACKED]) return;
    constexpr int CP8 = D / 8;
    const uint4 z = {0u, 0u, 0u, 0u};
    for (int w = blockIdx.x; w < p.B * p.M * p.Nq; w += gridDim.x) {
        const int bm = w / p.Nq, head = w - bm * p.Nq;
        const int b = bm / p.M, mm = bm - b * p.M;
        const int st = pv.start[bm], ln = pv.len[bm], npad = p.H - ln;
        __bf16* base = reinterpret_cast<__bf16*>(p.dq) + (long long)b * p.dq_b + (long long)head * p.dq_h;
        for (int idx = threadIdx.x; idx < npad * CP8; idx += blockDim.x) {
            const int r = idx / CP8, c8 = idx - r * CP8;
            const long long pos = (long long)mm * p.H + (r < st ? r : r + ln);
            *reinterpret_cast<uint4*>(base + pos * p.dq_t + c8 * 8) = z;
        }
    }
}

// Workgroups of four waves per compute unit: two, or at head dim 64, where registers and LDS allow it, three - if there are
// items enough for them (counted as if every block were full).  32/8 heads, us with two and three (dQ / dK, dV): 4 x 20
// documents of 160 tokens (3520 items) 82 / 92 and 72 / 82, 2 x 16 of 256 to 512 (4608) 117 / 132 and 104 / 120, 8 x 20 of 384
// to 512 (22528) 554 / 629 and 489 / 561, 2 x 12 of 33 to 250 (1792) 43 / 48 and 37 / 48; 8/2 heads, 4 x 20 of 96 to 224 (1232)
// 32.0 / 41.2 and 33.0 / 40.9.  Of batches much emptier than that, packed (the passes' kernels together): 4 x 20 of 16 to 64
// with one of 512 (1600 items of 11776) 140 and 131, 1 x 50, lognormal about 90 (1664 of 5824) 125 and 123; no layout
// tried that the rule takes lost anything.
int wgs_per_cu(int B, int M, int H, int D, const BrGeom& g, int n_cu) {
    const long long items = (long long)B * M * ((H + g.tpb * BR_RB - 1) / (g.tpb * BR_RB)) * g.NHG;
    return D == 64 && items >= 6LL * n_cu ? 3 : 2;
}

// p.published: one launch, which the caller chooses by br_bwd_one_launch
template <int D>
int launch_all(const BrBwdParams& p, int NW, int n_cu, hipStream_t stream) {
    const size_t n16 = (size_t)p.B * (p.Nq + 2 * p.Nkv) * p.H * D / 4;      // dq32, dk32, dv32 are contiguous
    hipLaunchKernelGGL(br_fill_zero_kernel, dim3(n_cu * 4), dim3(256), 0, stream, reinterpret_cast<uint4*>(p.dq32), n16, p.tickets,
                       p.published ? (BR_BWD_TICKETS + (size_t)p.B * p.M * p.Nkv) * BR_COUNTER_LINE : (size_t)(BR_BWD_TICKETS - 1) * p.ticket_step + 1);
    const int per_cu = wgs_per_cu(p.B, p.M, p.H, D, p.geom, n_cu);
    const int n_wg = n_cu * per_cu < 8 ? 8 : n_cu * per_cu;                 // (every queue needs a workgroup)
    if (p.published) {
        hipLaunchKernelGGL((br_bwd_kernel<D>), dim3(n_wg), dim3(256), 0, stream, p);
        hipLaunchKernelGGL((br_bwd_dq_finish_kernel<D>), dim3(n_cu * 4), dim3(256), 0, stream, p);
        return 0;
    }
    if (NW == 4) hipLaunchKernelGGL((br_bwd_dq_kernel<D, 4>), dim3(n_wg), dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((br_bwd_dq_kernel<D, 8>), dim3(n_cu < 8 ? 8 : n_cu), dim3(NW * 64), 0, stream, p);
    hipLaunchKernelGGL((br_bwd_dkv_kernel<D>), dim3(n_wg), dim3(256), 0, stream, p);
    hipLaunchKernelGGL((br_bwd_dq_finish_kernel<D>), dim3(n_cu * 4), dim3(256), 0, stream, p);
    return 0;
}

}  // namespace

// Whether dQ and dK, dV share a launch where the workspace has room for the counts it needs.  Three workgroups to a CU make two
// launches: their tails are short, and what waits in one launch costs more (the pass's kernels, one launch and two): 2 x 16
// documents of 33 to 250 tokens 109.6 and 97.8 us, 2 x 22 118.8 and 114.4, 2 x 20 of 160 97.7 and 95.2, 4 x 20 158.4 and 159.2,
// 8 x 20 of 384 to 512 1158 and 1164.  Two share one: 8/2 heads, 4 x 20 of 96 to 224, 87.8 and 92.4.  Other than four waves to
// a workgroup (three, five, six, seven or eight heads to one): dK, dV has four.
bool br_bwd_one_launch(int B, int M, int H, int D, const BrGeom& g, int NW, int n_cu) {
    return NW == 4 && wgs_per_cu(B, M, H, D, g, n_cu) == 2;
}

// Returns 0 on success, -1 if D has no instance.
int br_launch_bwd(const BrBwdParams& p, int D, int NW, int n_cu, hipStream_t stream) {
    if (D == 128) return launch_all<128>(p, NW, n_cu, stream);
    if (D == 64) return launch_all<64>(p, NW, n_cu, stream);
    return -1;
}
