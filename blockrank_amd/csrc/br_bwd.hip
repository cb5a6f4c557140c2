// Backward of the block-sparse prefill attention for gfx950 (bf16 inputs, fp32 arithmetic and accumulation).
//
// The reference has no hand-written backward: its trainable hooks (blockrank_std_attention.py:96-262, :472-650,
// used by trainer.py:79-101) are differentiated by torch autograd over dense masked tensors, and its Triton
// hook refuses (blockrank_triton_kernel_attention.py:759-761).  These kernels compute the same gradients
//     P = softmax(S),  dV = P^T dO,  dP = dO V^T,  dS = P * (dP - rowsum(dO * O)),
//     dQ = scale * dS K,  dK = scale * dS^T Q        (dK, dV summed over the query heads of a kv head)
// over exactly the (query row, key) pairs the forward visits.  P is rebuilt from the log-sum-exp the forward
// saved.  Two kernels, so that every sum that has one owner is kept in that owner's registers:
//
//   br_bwd_dq_kernel   query-major: walks the forward's own work items, one
//                      workgroup per (item, head group), a wave per 32 rows of one query head.  Per 64-key tile
//                      (K, V staged in LDS):  S^T = K Q^T, dP^T = V dO^T  (lane = query row, registers = keys)
//                      -> dS^T in bf16 is directly the A operand of dQ += dS K (K through transposing LDS reads).
//                      An item that owns its rows stores dQ; the items that share the query block's rows (its key
//                      walk is split) add into a small fp32 buffer that a finishing kernel converts.  Also writes
//                      delta = rowsum(dO * O) for the second kernel.
//   br_bwd_dkv_kernel  key-major: one workgroup per (64-key tile, kv head); a wave owns 32 of the keys and walks,
//                      for half of the group's query heads, every 32-row block that sees them (the rest of the
//                      key's own block from the diagonal on; for prefix keys all later blocks; for document keys
//                      the query block).  S = Q K^T, dP = dO V^T (lane = key, registers = rows) -> P and dS in
//                      bf16 are directly the A operands of dV += P^T dO and dK += dS^T Q, with dO and Q as
//                      "lane = dim, registers = rows" operands obtained by transposing LDS reads of the wave's
//                      own copy of the rows.  dK and dV never leave the registers until the walk ends: no atomics.
#include "br_common.h"

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
// Scheduling directives: a group of n instructions of one kind, placed in the order the directives are written
#define BR_SCHED_MFMA(n) __builtin_amdgcn_sched_group_barrier(0x008, n, 0)
#define BR_SCHED_DSREAD(n) __builtin_amdgcn_sched_group_barrier(0x100, n, 0)
#define BR_SCHED_EXP(n) __builtin_amdgcn_sched_group_barrier(0x402, n, 0)      // vector and transcendental instructions
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
// that the compiler does not make LDS reads of the other buffer wait for it; completion is awaited by vm_wait_all.
__device__ inline void dma16(const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
__device__ inline void dma4(const void* base, int off, unsigned lds_addr) {
    asm volatile("s_mov_b32 m0, %2\n\tglobal_load_lds_dword %0, %1" ::"v"(off), "s"(base), "s"(lds_addr) : "memory", "m0");
}
__device__ inline void vm_wait_all() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
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
// accumulator registers 8s .. 8s+7 as one bf16 operand
__device__ inline bf16x8 pack8(const f32x16& x, int s) {
    f32x8 t;
#pragma unroll
    for (int e = 0; e < 8; ++e) t[e] = x[8 * s + e];
    return __builtin_convertvector(t, bf16x8);
}

template <int D>
struct Bwd {
    static constexpr int RS = 2 * D + 32;          // LDS row stride in bytes: the 32 bytes of padding put the four rows of a transposing read in different banks
    static constexpr int CPR = D / 8;              // 16-byte pieces per row
    static constexpr int NC = D / 16, ND = D / 32;
    static constexpr int tileBytes = BR_BN * RS;
    static constexpr int rowsBytes = BR_RB * RS;

    // Row (r0 + lane % 32), dims 16c + 8 * (lane / 32) .. +7 of a row-major LDS tile: the operand layout of a
    // product that contracts over the head dim.
    static __device__ inline bf16x8 read_row(const char* tile, int r0, int c, int ln, int lh) {
        return as_bf16x8(ld16(tile + (r0 + ln) * RS + c * 32 + lh * 16));
    }
    // Column (32 db + lane % 32), rows r0 + 4 lh + {0..3, 8..11} of a row-major LDS tile: the operand layout of a
    // product that contracts over rows, in the order in which a 32x32 accumulator's registers 8s .. 8s+7 hold
    // them (r0 = 16 s).  Two transposing reads: in each group of 16 lanes, lane s points at row (s >> 2),
    // dims 4 (s & 3) .. +3 of the group's 16 dims and receives the four rows of dim s.
    static __device__ inline bf16x8 read_col(const char* tile, int r0, int db, int lane) {
        const int s = lane & 15, hi = (lane >> 4) & 1, lh = lane >> 5;
        const char* p = tile + (r0 + 4 * lh + (s >> 2)) * RS + (32 * db + 16 * hi + 4 * (s & 3)) * 2;
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(__attribute__((address_space(3))) const char*)p);
        s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(__attribute__((address_space(3))) const char*)(p + 8 * RS));
        union { s16x8 s8; bf16x8 b8; } a;
        a.s8 = __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7);
        return a.b8;
    }

    // The same from a swizzled, unpadded buffer: at is the LDS address of the first four rows' read (see dkv_tile)
    static __device__ inline bf16x8 tr_pair(int at) {
        s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)at);
        s16x4 up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)((at ^ 32) + 8 * 2 * D));
        return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, up, 0, 1, 2, 3, 4, 5, 6, 7));
    }

    // ---------------------------------------------------------------------------------------------------------
    // dQ (and delta) of one work item
    // ---------------------------------------------------------------------------------------------------------
    static constexpr int dqLdsBytes = 2 * tileBytes;

    static __device__ __forceinline__ void dq_item(const BrBwdParams& p, const BrPlanView& pv, const BrItem& it, int hg, char* smem, int NW) {
        const int tid = threadIdx.x, NT = NW * 64;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, lh = lane >> 5;
        const BrGeom& ge = p.geom;
        const int T = ge.tpb * BR_RB;
        const int b = it.b;
        const int kvh = hg / ge.HGS, hsub = hg - kvh * ge.HGS;
        const int g = wave / ge.tpb, sub = wave - g * ge.tpb;
        const int head = kvh * ge.G + hsub * ge.Gw + g;
        const int len_m = it.len_m;
        const int row0 = it.t0 + sub * BR_RB;
        const bool rb_active = row0 < len_m;
        const int self_end = it.t0 + T < len_m ? it.t0 + T : len_m;
        const int qtok0 = it.tok_m;
        char* Ks = smem;
        char* Vs = smem + tileBytes;
        const char* kbase = reinterpret_cast<const char*>(p.k) + 2 * ((unsigned long long)p.k32_b * (unsigned)b + (unsigned long long)p.k32_h * (unsigned)kvh);
        const char* vbase = reinterpret_cast<const char*>(p.v) + 2 * ((unsigned long long)p.v32_b * (unsigned)b + (unsigned long long)p.v32_h * (unsigned)kvh);

        // Q and dO of this wave's rows (lane = row, registers = dims), the rows' log-sum-exp and delta
        bf16x8 qf[NC], dof[NC];
        float lse_l = 0.f, delta_l = 0.f;
        if (rb_active) {
            const int last = len_m - 1 - row0;
            const int r = ln < last ? ln : last;       // rows past the block's end repeat its last row; they are masked below
            const unsigned tok = (unsigned)(qtok0 + row0 + r);
            const char* qrow = reinterpret_cast<const char*>(p.q) +
                               2 * ((unsigned long long)p.q32_b * (unsigned)b + (unsigned long long)p.q32_h * (unsigned)head + (unsigned long long)p.q32_t * tok);
            const char* grow = reinterpret_cast<const char*>(p.dout) +
                               2 * ((unsigned long long)p.g32_b * (unsigned)b + (unsigned long long)p.g32_h * (unsigned)head + (unsigned long long)p.g32_t * tok);
            const char* orow = reinterpret_cast<const char*>(p.out) +
                               2 * ((unsigned long long)p.o32_b * (unsigned)b + (unsigned long long)p.o32_h * (unsigned)head + (unsigned long long)p.o32_t * tok);
            float dsum = 0.f;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                qf[c] = as_bf16x8(ld16(qrow + c * 32 + lh * 16));
                dof[c] = as_bf16x8(ld16(grow + c * 32 + lh * 16));
                const bf16x8 o8 = as_bf16x8(ld16(orow + c * 32 + lh * 16));
#pragma unroll
                for (int e = 0; e < 8; ++e) dsum += (float)o8[e] * (float)dof[c][e];
            }
            delta_l = dsum + __shfl_xor(dsum, 32);
            const long long li = (long long)b * p.lse_b + (long long)head * p.lse_h + tok;
            lse_l = p.lse[li];
            // every item of a row block computes the same delta; the one that starts the key walk publishes it
            if (it.f_lo == 0 && lh == 0 && ln <= last) p.delta[li] = -delta_l;
        } else {
#pragma unroll
            for (int c = 0; c < NC; ++c) qf[c] = dof[c] = as_bf16x8(uint4{0u, 0u, 0u, 0u});
        }

        f32x16 dq[ND];
#pragma unroll
        for (int db = 0; db < ND; ++db) dq[db] = zero16();

        // the item's key walk: the earlier blocks' tiles it covers, then its own block's up to the diagonal
        const int2* tiles_b = pv.tiles + (size_t)b * pv.tps;
        const bool table = it.pe > 1;
        const int nprev = it.nprev;
        const int f_end = it.ntiles > 0x3fffffff ? 0x7fffffff : it.f_lo + it.ntiles;
        // The walk is software-pipelined: a thread's pieces of the next tile are loaded into registers while the
        // current tile (in LDS) is computed.
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
                        const int2 d = tiles_b[fi];
                        t.tok0 = d.x;
                        t.nvalid = d.y;
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
        constexpr int NPC = BR_BN * CPR / 256;     // 16-byte pieces of K (and of V) per thread and tile (at least 256 threads)
        uint4 kreg[NPC], vreg[NPC];
        auto load_tile = [&](const Tile& t) {      // rows past the tile's real keys are zero
#pragma unroll
            for (int i = 0; i < NPC; ++i) {
                const int idx = tid + i * NT;
                const int r = idx / CPR, c = idx - r * CPR;
                kreg[i] = vreg[i] = uint4{0u, 0u, 0u, 0u};
                if (idx < BR_BN * CPR && r < t.nvalid) {
                    kreg[i] = ld16(kbase + 2 * ((long long)(t.tok0 + r) * p.k32_t + c * 8));
                    vreg[i] = ld16(vbase + 2 * ((long long)(t.tok0 + r) * p.v32_t + c * 8));
                }
            }
        };
        Tile cur, nxt;
        bool have = next_tile(cur);
        if (have) load_tile(cur);
        // Everything requested so far (Q, dO, O, the first tile) is needed before the first product anyway: wait here,
        // so that the loop is entered with no load pending.  Otherwise the compiler's wait-count bookkeeping keeps
        // partial waits in front of every use of Q and dO inside the loop, and those waits count the tile requested
        // ahead - the look-ahead would wait for itself.
        __builtin_amdgcn_s_waitcnt(0x0F70);          // vmcnt(0); expcnt and lgkmcnt not waited for
        while (have) {
            const bool self = cur.self;
            const int nvalid = cur.nvalid, key0 = cur.key0;
            lds_barrier();                         // every wave has finished with the previous tile
#pragma unroll
            for (int i = 0; i < NPC; ++i) {
                const int idx = tid + i * NT;
                const int r = idx / CPR, c = idx - r * CPR;
                if (idx < BR_BN * CPR) {
                    *reinterpret_cast<uint4*>(Ks + r * RS + c * 16) = kreg[i];
                    *reinterpret_cast<uint4*>(Vs + r * RS + c * 16) = vreg[i];
                }
            }
            const bool have_next = next_tile(nxt);
            if (have_next) load_tile(nxt);
            lds_barrier();

            // 32-key halves this wave needs: limited by the real keys and, on the block's own keys, by the diagonal
            int nkb = (nvalid + 31) >> 5;
            if (self) {
                const int vis = row0 + BR_RB - key0;
                const int c = vis <= 0 ? 0 : (vis + 31) >> 5;
                nkb = c < nkb ? c : nkb;
            }
            if (!rb_active) nkb = 0;
            for (int kb = 0; kb < nkb; ++kb) {
                f32x16 st = zero16(), dpt = zero16();
#pragma unroll
                for (int c = 0; c < NC; ++c) {
                    st = mma(read_row(Ks, kb * 32, c, ln, lh), qf[c], st);
                    dpt = mma(read_row(Vs, kb * 32, c, ln, lh), dof[c], dpt);
                }
                const int lim_c = self ? row0 + ln - key0 + 1 : BR_BN;                 // keys [0, lim) of the tile are visible
                int lim = nvalid < lim_c ? nvalid : lim_c;
                if (row0 + ln >= len_m) lim = 0;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int key = kb * 32 + 8 * (v >> 2) + 4 * lh + (v & 3);
                    // hidden pairs get exponent -inf, i.e. probability 0, without a branch (every operand is finite)
                    const float pr = __builtin_amdgcn_exp2f(key < lim ? st[v] * p.scale_log2 - lse_l : -INFINITY);
                    st[v] = pr * (dpt[v] - delta_l) * p.scale;
                }
#pragma unroll
                for (int s = 0; s < 2; ++s) {
                    const bf16x8 a = pack8(st, s);
                    // K as "lane = dim" operand of this 16-key step: the transposing reads are issued together, ahead of the products
                    bf16x8 kc[ND];
#pragma unroll
                    for (int db = 0; db < ND; ++db) kc[db] = read_col(Ks, kb * 32 + 16 * s, db, lane);
#pragma unroll
                    for (int db = 0; db < ND; ++db) dq[db] = mma(a, kc[db], dq[db]);
                }
            }
            cur = nxt;
            have = have_next;
        }
        // dQ of this wave's rows: lane = dim 32 db + ln, register v = row 8 (v/4) + 4 lh + v%4
        if (!rb_active) return;
        if (it.slot < 0) {
            __bf16* dst = reinterpret_cast<__bf16*>(p.dq) + (long long)b * p.dq_b + (long long)head * p.dq_h +
                          (long long)(qtok0 + row0 + 4 * lh) * p.dq_t + ln;
#pragma unroll
            for (int db = 0; db < ND; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int r = 8 * (v >> 2) + (v & 3);
                    if (row0 + 4 * lh + r < len_m) dst[(long long)r * p.dq_t + db * 32] = (__bf16)dq[db][v];
                }
        } else {
            // shared rows (the query block): [b][head][row of the block][D] fp32
            float* dqp = p.dq32 + (((long long)b * p.Nq + head) * p.H + row0 + 4 * lh) * D + ln;
#pragma unroll
            for (int db = 0; db < ND; ++db)
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const int r = 8 * (v >> 2) + (v & 3);
                    if (row0 + 4 * lh + r < len_m) unsafeAtomicAdd(dqp + r * D + db * 32, dq[db][v]);
                }
        }
    }

    // ---------------------------------------------------------------------------------------------------------
    // dK, dV of one 64-key tile of one kv head: 128 threads, wave w owns keys 32 w .. 32 w + 31 of the tile, whole
    // head dim.  A step is 32 query rows of one head: their Q and dO rows come into one of two LDS buffers by DMA, a
    // whole step ahead (one barrier per step), and each wave computes for its keys
    //     S = Q K^T, dP = dO V^T - delta   (A = rows from LDS, B = the wave's keys, kept in registers)
    //     dV += P^T dO, dK += dS^T Q       (P, dS in bf16 straight from the accumulators; dO, Q by transposing reads)
    // 32 MFMAs per wave and step against 40 KB of LDS reads.
    // ---------------------------------------------------------------------------------------------------------
    static constexpr int rowB = 2 * D;                                    // bytes of a row, in memory and in the buffers
    static constexpr int bufBytes = 2 * BR_RB * rowB + 512;               // 32 rows of Q, of dO; lse and -delta of the rows
    static constexpr int dkvLdsBytes = 2 * bufBytes;
    // 16-byte piece c of row r sits at piece c ^ row_swizzle(r): the 32 rows one operand read takes a piece of, and the
    // four rows x 64 bytes a transposing read takes, each spread over all banks
    static __device__ inline int row_swizzle(int r) {
        return CPR == 16 ? ((r & 3) << 2) | ((r >> 2) & 3) : (((r >> 1) & 1) << 2) | ((r >> 2) & 3);
    }

    // mq < 0: the tile's one owner - the rows are the rest of the keys' own block from the diagonal on and, for document
    // keys, the query block.  Otherwise the keys are prefix keys and the rows those of block mq: the sums of the
    // workgroups of all viewing blocks meet in fp32 buffers (atomic adds).
    static __device__ __forceinline__ void dkv_tile(const BrBwdParams& p, const BrPlanView& pv, int b, int m, int kt, int kvh, int mq, char* smem) {
        const int tid = threadIdx.x;
        const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, ln = lane & 31, lh = lane >> 5;
        const int G = p.geom.G, M = p.M;
        const int len_m = pv.len[b * M + m], tok_m = pv.tok[b * M + m];
        const int key0 = kt * BR_BN + wave * 32;                              // the wave's first key
        const int nkeys = len_m - key0 < 32 ? len_m - key0 : 32;              // may be zero or less: nothing to compute
        const unsigned smem_lds = lds_addr_of(smem);

        // the wave's keys as operands (lane = key, registers = dims); past the real keys zeros, whose sums nothing reads
        bf16x8 kf[NC], vf[NC];
        {
            const bool on = ln < nkeys;
            const unsigned tok = (unsigned)(tok_m + (on ? key0 + ln : 0));
            const char* krow = reinterpret_cast<const char*>(p.k) + 2 * ((unsigned long long)p.k32_b * (unsigned)b + (unsigned long long)p.k32_h * (unsigned)kvh + (unsigned long long)p.k32_t * tok);
            const char* vrow = reinterpret_cast<const char*>(p.v) + 2 * ((unsigned long long)p.v32_b * (unsigned)b + (unsigned long long)p.v32_h * (unsigned)kvh + (unsigned long long)p.v32_t * tok);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                kf[c] = as_bf16x8(on ? ld16(krow + c * 32 + lh * 16) : uint4{0u, 0u, 0u, 0u});
                vf[c] = as_bf16x8(on ? ld16(vrow + c * 32 + lh * 16) : uint4{0u, 0u, 0u, 0u});
            }
        }

        // The steps: (32-row block that sees these keys, head of the group), the same for both waves
        struct Step {
            int r0, nrows, tok, head, self;
        };
        const bool pre = mq >= 0;
        const int blk0 = pre ? mq : m;
        const int blk1 = !pre && m > 0 && m < M - 1 ? M - 1 : -1;
        int seg = 0;                                                 // 2 = exhausted
        int cur_blk = blk0, cur_len = pv.len[b * M + blk0], cur_tok = pv.tok[b * M + blk0];
        int rb = blk0 == m ? kt * (BR_BN / BR_RB) : 0, hl = 0;
        auto next_step = [&](Step& st) -> bool {
            while (seg < 2) {
                if (rb * BR_RB >= cur_len) {
                    seg = (seg == 0 && blk1 >= 0) ? 1 : 2;
                    if (seg == 1) {
                        cur_blk = blk1;
                        cur_len = pv.len[b * M + blk1];
                        cur_tok = pv.tok[b * M + blk1];
                        rb = 0;
                    }
                    continue;
                }
                const int r0 = rb * BR_RB;
                st.r0 = r0;
                st.nrows = cur_len - r0 < BR_RB ? cur_len - r0 : BR_RB;
                st.tok = cur_tok + r0;
                st.head = kvh * G + hl;
                st.self = cur_blk == m;
                if (++hl >= G) {
                    hl = 0;
                    ++rb;
                }
                return true;
            }
            return false;
        };

        // DMA of a step's rows: wave 0 the Q rows and their log-sum-exp, wave 1 the dO rows and their (negated) delta.
        // Rows past the block's end are zeros: their P is 1, and what it multiplies - dO, dP, delta - is zero.
        constexpr int RPI = 64 / CPR, NI = BR_RB / RPI;              // rows per DMA instruction, instructions
        const char* row_t = reinterpret_cast<const char*>(wave == 0 ? p.q : p.dout);
        const unsigned row_b = wave == 0 ? p.q32_b : p.g32_b, row_h = wave == 0 ? p.q32_h : p.g32_h, row_s = wave == 0 ? p.q32_t : p.g32_t;
        const float* stat = wave == 0 ? p.lse : p.delta;
        const char* row_tb = row_t + 2 * (unsigned long long)row_b * (unsigned)b;
        const float* stat_b = stat + (long long)b * p.lse_b;
        auto issue = [&](const Step& st, int buf) {
            // (the lane as a value of this step that the compiler cannot trace back: what is derived from it is not kept
            // in registers across the walk)
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int srow = lane_l / CPR, spiece = lane_l % CPR, ln_l = lane_l & 31;
            const char* base = row_tb + 2 * ((unsigned long long)row_h * (unsigned)st.head + (unsigned long long)row_s * (unsigned)st.tok);
            const unsigned dst = smem_lds + buf * bufBytes + wave * (BR_RB * rowB);
            const int step_bytes = RPI * 2 * (int)row_s;
            if (st.nrows == BR_RB) {
#pragma unroll
                for (int j = 0; j < NI; ++j)
                    dma16(base + (long long)j * step_bytes, srow * 2 * (int)row_s + ((spiece ^ row_swizzle(j * RPI + srow)) << 4), dst + j * 1024);
            } else {
#pragma unroll
                for (int j = 0; j < NI; ++j) {
                    const int r = j * RPI + srow;
                    if (r < st.nrows) dma16(base, r * 2 * (int)row_s + ((spiece ^ row_swizzle(r)) << 4), dst + j * 1024);
                    else *reinterpret_cast<uint4*>(smem + buf * bufBytes + wave * (BR_RB * rowB) + j * 1024 + lane_l * 16) = uint4{0u, 0u, 0u, 0u};
                }
            }
            const unsigned sdst = 2 * BR_RB * rowB + wave * 256;
            if (ln_l < st.nrows) dma4(stat_b + (long long)st.head * p.lse_h + st.tok, ln_l * 4, smem_lds + buf * bufBytes + sdst);
            else *reinterpret_cast<float*>(smem + buf * bufBytes + sdst + lane_l * 4) = 0.f;
        };

        f32x16 dk[ND], dv[ND];      // lane = key, register v of block db = dim 32 db + 8 (v / 4) + 4 lh + v % 4
#pragma unroll
        for (int db = 0; db < ND; ++db) dk[db] = dv[db] = zero16();
        auto compute = [&](int buf, bool diagonal) {
            // LDS addresses of the operand reads: row reads of piece 2c + lh are ra ^ (c << 5); transposing reads of block db,
            // rows 16 s + 4 lh + 0..3 are ca ^ (db << 6), 16 s rows further, and those of the rows eight further the same
            // ^ 32 and 8 rows further.  From a lane index that the compiler cannot trace back: none of the sixteen
            // addresses is then kept in registers across the walk.
            int lane_l = lane;
            asm volatile("" : "+v"(lane_l));
            const int base = smem_lds + buf * bufBytes, lh = lane_l >> 5, ln = lane_l & 31, s16 = lane_l & 15, crow = 4 * lh + (s16 >> 2);
            const int ra = base + ln * rowB + ((lh ^ row_swizzle(ln)) << 4);
            const int ca = base + crow * rowB + (((2 * ((lane_l >> 4) & 1) + ((s16 & 3) >> 1)) ^ row_swizzle(crow)) << 4) + (s16 & 1) * 8;
            const int la = base + 2 * BR_RB * rowB + 16 * lh;
            constexpr int AHEAD = 3;     // operand reads in flight ahead of the product that uses them
            bf16x8 x[AHEAD];
            f32x16 sc = zero16();
#pragma unroll
            for (int c = 0; c < AHEAD; ++c) x[c] = *(lds_bf16x8*)(ra ^ (c << 5));
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                sc = mma(x[c % AHEAD], kf[c], sc);
                if (c + AHEAD < NC) x[c % AHEAD] = *(lds_bf16x8*)(ra ^ ((c + AHEAD) << 5));
            }
            BR_SCHED_DSREAD(AHEAD);
#pragma unroll
            for (int i = 0; i + AHEAD < NC; ++i) {
                BR_SCHED_MFMA(1);
                BR_SCHED_DSREAD(1);
            }
            BR_SCHED_MFMA(AHEAD);
            BR_SCHED_FENCE();
            if (diagonal) {              // the wave's own 32 rows: key ln is hidden from the rows before it
                const int first = ln - 4 * lh;
#pragma unroll
                for (int v = 0; v < 16; ++v) sc[v] = 8 * (v >> 2) + (v & 3) < first ? -INFINITY : sc[v];
            }
            f32x16 dp;
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
                const f32x4 t = *(lds_f32x4*)(la + 256 + 32 * v4);
                dp[4 * v4] = t[0]; dp[4 * v4 + 1] = t[1]; dp[4 * v4 + 2] = t[2]; dp[4 * v4 + 3] = t[3];
            }
#pragma unroll
            for (int c = 0; c < 2; ++c) x[c] = *(lds_bf16x8*)((ra ^ (c << 5)) + BR_RB * rowB);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                dp = mma(x[c & 1], vf[c], dp);
                if (c + 2 < NC) x[c & 1] = *(lds_bf16x8*)((ra ^ ((c + 2) << 5)) + BR_RB * rowB);
            }
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
                const f32x4 l4 = *(lds_f32x4*)(la + 32 * v4);
#pragma unroll
                for (int e = 0; e < 4; ++e) sc[4 * v4 + e] = __builtin_amdgcn_exp2f(sc[4 * v4 + e] * p.scale_log2 - l4[e]);
            }
            // the exponentials pass under the dP products
            BR_SCHED_DSREAD(6);
#pragma unroll
            for (int i = 0; i + 2 < NC; i += 2) {
                BR_SCHED_MFMA(1);
                BR_SCHED_DSREAD(2);
                BR_SCHED_EXP(8);
                BR_SCHED_MFMA(1);
                BR_SCHED_DSREAD(1);
                BR_SCHED_EXP(4);
            }
            BR_SCHED_MFMA(2);
            BR_SCHED_FENCE();
#pragma unroll
            for (int v = 0; v < 16; ++v) dp[v] *= sc[v];
            const bf16x8 pa[2] = {pack8(sc, 0), pack8(sc, 1)}, da[2] = {pack8(dp, 0), pack8(dp, 1)};
            BR_SCHED_FENCE();
            {
                // read i: rows 16 (i / 2 ND) .., block (i / 2) % ND, dO (even) or Q (odd); two reads ahead of the products
                auto rd = [&](int i) { return tr_pair((ca ^ ((i >> 1) % ND << 6)) + (i / (2 * ND)) * 16 * rowB + (i & 1 ? 0 : BR_RB * rowB)); };
                constexpr int N = 4 * ND;
                bf16x8 x[2] = {rd(0), rd(1)};
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const int s = i / (2 * ND), db = (i >> 1) % ND;
                    const bf16x8 w = i & 1 ? da[s] : pa[s];
                    f32x16& acc = i & 1 ? dk[db] : dv[db];
                    acc = mma(x[i & 1], w, acc);
                    if (i + 2 < N) x[i & 1] = rd(i + 2);
                }
                BR_SCHED_DSREAD(4);
#pragma unroll
                for (int i = 0; i + 2 < N; ++i) {
                    BR_SCHED_MFMA(1);
                    BR_SCHED_DSREAD(2);
                }
                BR_SCHED_MFMA(2);
                BR_SCHED_FENCE();
            }
        };

        Step cur, nxt;
        bool have = next_step(cur);
        if (have) issue(cur, 0);
        // the keys are waited for here: the compiler's own wait inside the loop would also cover the rows requested ahead
#pragma unroll
        for (int c = 0; c < NC; ++c) asm volatile("" : "+v"(kf[c]), "+v"(vf[c]));
        int buf = 0;
        while (have) {
            const bool have_next = next_step(nxt);
            vm_wait_all();                       // this wave's part of the step's rows has arrived ...
            lds_barrier();                       // ... and everyone's, and nobody reads the other buffer any more
            if (have_next) issue(nxt, buf ^ 1);
            // the wave has a pair to compute in this step unless its first key follows the step's rows (on its own block the
            // rows go in steps of 32 from the tile's first key on: only the step of the wave's own rows is cut by the diagonal)
            if (nkeys > 0 && !(cur.self && cur.r0 < key0)) compute(buf, cur.self && cur.r0 == key0);
            cur = nxt;
            have = have_next;
            buf ^= 1;
        }

        if (pre) {
            // prefix keys: rows of D floats through LDS, so that an instruction adds to one key's consecutive dims
            lds_barrier();                       // nobody reads the rows any more
            if (nkeys <= 0) return;
            float* T = reinterpret_cast<float*>(smem + wave * bufBytes);          // [32 keys][D], 16-byte pieces swizzled
            constexpr int PM = D / 4 - 1 < 31 ? D / 4 - 1 : 31;
            auto add = [&](f32x16 (&acc)[ND], float* dst, float f) {
#pragma unroll
                for (int db = 0; db < ND; ++db)
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const f32x4 t = {acc[db][4 * q] * f, acc[db][4 * q + 1] * f, acc[db][4 * q + 2] * f, acc[db][4 * q + 3] * f};
                        *reinterpret_cast<f32x4*>(T + ln * D + (((8 * db + 2 * q + lh) ^ (ln & PM)) << 2)) = t;
                    }
                __threadfence_block();           // (one wave writes and reads: its LDS operations complete in order)
                dst += (((long long)b * p.Nkv + kvh) * p.H + key0) * D;
                for (int k = 0; k < nkeys; ++k)
#pragma unroll
                    for (int d = lane; d < D; d += 64) unsafeAtomicAdd(dst + (long long)k * D + d, T[k * D + (((d >> 2) ^ (k & PM)) << 2) + (d & 3)]);
                __threadfence_block();
            };
            add(dk, p.dk32, p.scale);
            add(dv, p.dv32, 1.f);
            return;
        }
        if (nkeys <= 0) return;
        // one owner: bf16.  A lane holds dims 8 q + 4 lh + 0..3 of its key; the halves of a wave exchange pieces so that
        // every lane stores eight consecutive dims
        auto store = [&](f32x16 (&acc)[ND], void* dst_, long long db_, long long dh_, long long dt_, float f) {
            __bf16* dst = reinterpret_cast<__bf16*>(dst_) + (long long)b * db_ + (long long)kvh * dh_ + (long long)(tok_m + key0 + ln) * dt_ + 8 * lh;
#pragma unroll
            for (int db = 0; db < ND; ++db)
#pragma unroll
                for (int q = 0; q < 4; q += 2) {
                    unsigned a[2], c[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) {
                        a[i] = pack2(acc[db][4 * q + 2 * i] * f, acc[db][4 * q + 2 * i + 1] * f);
                        c[i] = pack2(acc[db][4 * q + 4 + 2 * i] * f, acc[db][4 * q + 5 + 2 * i] * f);
                    }
                    const auto x0 = __builtin_amdgcn_permlane32_swap(a[0], c[0], false, false);
                    const auto x1 = __builtin_amdgcn_permlane32_swap(a[1], c[1], false, false);
                    if (ln < nkeys) *reinterpret_cast<uint4*>(dst + 32 * db + 8 * q) = uint4{x0[0], x1[0], x0[1], x1[1]};
                }
        };
        store(dk, p.dk, p.dk_b, p.dk_h, p.dk_t, p.scale);
        store(dv, p.dv, p.dv_b, p.dv_h, p.dv_t, 1.f);
    }
};

template <int D, int MAXW>
__global__ __launch_bounds__(MAXW * 64, MAXW <= 4 ? (D == 64 ? 3 : 2) : 1) void br_bwd_dq_kernel(BrBwdParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const BrGeom& ge = p.geom;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, ge.tpb * BR_RB);
    const int item = blockIdx.x / ge.NHG, hg = blockIdx.x - item * ge.NHG;
    if (item >= pv.hdr[BR_PH_NITEMS]) return;
    const BrItem it = pv.items[item];
    Bwd<D>::dq_item(p, pv, it, hg, smem, blockDim.x >> 6);
}

// Work is enumerated as (group, slot): a group is one (block m, sequence, kv head) and holds every workgroup that
// reads that block's Q and dO rows - for each 64-key tile of the block and each 32-key half its main workgroup,
// plus (m >= 1) the workgroups that take the block's rows to the prefix keys.  The hardware deals workgroups
// round robin to the 8 XCDs by index, and each XCD has its own L2: group g is therefore laid out on indices
// congruent to g mod 8, so that all its workgroups run on one XCD and the rows are fetched from HBM into one L2
// only (measured at the Mistral-7B shape with 20 documents: 0.39 GB of HBM reads per launch against 1.25 GB with
// a plain enumeration, where every row block was fetched by up to eight workgroups on different XCDs; 0.27 GB
// is the algorithmic minimum).
template <int D>
__global__ __launch_bounds__(128, 2) void br_bwd_dkv_kernel(BrBwdParams p) {
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.geom.tpb * BR_RB);
    const int KT = (p.H + BR_BN - 1) / BR_BN;
    const int S = 2 * KT;                                    // slots per group
    const int x = blockIdx.x & 7, j = blockIdx.x >> 3;
    const int g = (j / S) * 8 + x, slot = j % S;
    if (g >= p.M * p.B * p.Nkv) return;
    const int kvh = g % p.Nkv, b = (g / p.Nkv) % p.B, mg = g / (p.Nkv * p.B);
    const bool extra = slot >= KT;
    const int kt = extra ? slot - KT : slot;
    if (extra && mg == 0) return;
    const int m = extra ? 0 : mg;
    const int len_m = pv.len[b * p.M + m];
    // padded slots of this block (dk and dv of this kv head): zeros, written by the block's first workgroup
    if (kt == 0 && !extra && !pv.hdr[BR_PH_PACKED]) {
        const int st = pv.start[b * p.M + m], npad = p.H - len_m;
        constexpr int CP8 = D / 8;
        const uint4 z = {0u, 0u, 0u, 0u};
        __bf16* kb_ = reinterpret_cast<__bf16*>(p.dk) + (long long)b * p.dk_b + (long long)kvh * p.dk_h;
        __bf16* vb_ = reinterpret_cast<__bf16*>(p.dv) + (long long)b * p.dv_b + (long long)kvh * p.dv_h;
        for (int i = threadIdx.x; i < npad * CP8; i += blockDim.x) {
            const int r = i / CP8, c8 = i - r * CP8;
            const long long pos = (long long)m * p.H + (r < st ? r : r + len_m);
            *reinterpret_cast<uint4*>(kb_ + pos * p.dk_t + c8 * 8) = z;
            *reinterpret_cast<uint4*>(vb_ + pos * p.dv_t + c8 * 8) = z;
        }
    }
    if (kt * BR_BN >= len_m) return;                     // no real key in this tile
    Bwd<D>::dkv_tile(p, pv, b, m, kt, kvh, m == 0 && p.M > 1 ? mg : -1, smem);
}

__global__ __launch_bounds__(256) void br_fill_zero_kernel(uint4* p, size_t n16) {
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

template <int D, int MAXW>
int launch_dq(const BrBwdParams& p, int NW, hipStream_t stream) {
    constexpr int lds = Bwd<D>::dqLdsBytes;
    static_assert(lds <= 65536, "dynamic LDS above 64 KiB would need hipFuncSetAttribute");
    hipLaunchKernelGGL((br_bwd_dq_kernel<D, MAXW>), dim3(p.max_items * p.geom.NHG), dim3(NW * 64), lds, stream, p);
    return 0;
}

template <int D>
int launch_all(const BrBwdParams& p, int NW, int n_cu, hipStream_t stream) {
    const size_t n16 = (size_t)p.B * (p.Nq + 2 * p.Nkv) * p.H * D / 4;      // dq32, dk32, dv32 are contiguous
    hipLaunchKernelGGL(br_fill_zero_kernel, dim3(n_cu * 4), dim3(256), 0, stream, reinterpret_cast<uint4*>(p.dq32), n16);
    const int rc = NW <= 4 ? launch_dq<D, 4>(p, NW, stream) : launch_dq<D, 8>(p, NW, stream);
    if (rc) return rc;
    constexpr int lds = Bwd<D>::dkvLdsBytes;
    static_assert(lds <= 65536, "dynamic LDS above 64 KiB would need hipFuncSetAttribute");
    const int KT = (p.H + BR_BN - 1) / BR_BN;
    hipLaunchKernelGGL((br_bwd_dkv_kernel<D>), dim3((p.M * p.B * p.Nkv + 7) / 8 * 8 * 2 * KT), dim3(128), lds, stream, p);
    hipLaunchKernelGGL((br_bwd_dq_finish_kernel<D>), dim3(n_cu * 4), dim3(256), 0, stream, p);
    return 0;
}

}  // namespace

// Returns 0 on success, -1 if D has no instance.
int br_launch_bwd(const BrBwdParams& p, int D, int NW, int n_cu, hipStream_t stream) {
    if (D == 128) return launch_all<128>(p, NW, n_cu, stream);
    if (D == 64) return launch_all<64>(p, NW, n_cu, stream);
    return -1;
}
