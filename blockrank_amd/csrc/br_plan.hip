// Request plan: turns the (B, M, H) block mask into the block table (start, len per block) and the
// work-item list the persistent prefill kernel consumes.  Built on the device with no host
// synchronisation, once per forward pass (the block structure is the same for every layer).
//
// The additive 5-D mask of the reference (blockrank_std_attention.py:293-309) carries exactly this
// information: which keys of each block are real.  Everything else (causality inside a block, which
// earlier blocks a block may see) follows from the block index, so the kernels never read a mask.
#include "br_common.h"

namespace {

constexpr int kPlanThreads = 512;

// One wave per block: count real tokens, find the first and the last.  len is written negated
// (-1 - count) when the real tokens are not one contiguous span; the plan kernel repairs the sign
// and raises the header flag.
__global__ __launch_bounds__(256) void br_block_table_kernel(const uint8_t* __restrict__ valid, int BM, int H,
                                                             int* __restrict__ start, int* __restrict__ len) {
    const int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int lane = threadIdx.x & 63;
    if (wave >= BM) return;
    const uint8_t* row = valid + (size_t)wave * H;
    int cnt = 0, first = H, last = -1;
    for (int j = lane; j < H; j += 64) {
        if (row[j]) {
            ++cnt;
            first = j < first ? j : first;
            last = j > last ? j : last;
        }
    }
    for (int o = 32; o > 0; o >>= 1) {
        cnt += __shfl_xor(cnt, o);
        int f = __shfl_xor(first, o);
        int l = __shfl_xor(last, o);
        first = f < first ? f : first;
        last = l > last ? l : last;
    }
    if (lane == 0) {
        bool contiguous = cnt == 0 || (last - first + 1 == cnt);
        start[wave] = cnt == 0 ? 0 : first;
        len[wave] = contiguous ? cnt : -1 - cnt;
    }
}

__device__ inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// Exclusive scans of N values per thread over the workgroup, one pair of barriers for all of them (wave-level scans with
// lane shuffles, then the wave totals): x[i] becomes the exclusive prefix of x[i], tot[i] the total.
template <int N>
__device__ void block_exclusive_scan_n(int (&x)[N], int (&tot)[N], int* shn /* N * kPlanThreads / 64 ints */) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    int incl[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
        incl[i] = x[i];
        for (int o = 1; o < 64; o <<= 1) {
            int y = __shfl_up(incl[i], o);
            if (lane >= o) incl[i] += y;
        }
        if (lane == 63) shn[i * (kPlanThreads / 64) + wave] = incl[i];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        int base = 0, t = 0;
        for (int w = 0; w < kPlanThreads / 64; ++w) {
            const int v = shn[i * (kPlanThreads / 64) + w];
            if (w < wave) base += v;
            t += v;
        }
        tot[i] = t;
        x[i] = base + incl[i] - x[i];
    }
    __syncthreads();
}

// par: workgroups of the prefill grid per head group, i.e. how many of a plan's items run side by side.
// pool: split-KV partial slots the caller's workspace has room for (br_split_pool).
__global__ __launch_bounds__(kPlanThreads) void br_plan_kernel(int* __restrict__ plan, int B, int M, int H, int T, int packed, int par, int pool) {
    constexpr int kW = kPlanThreads / 64;
    __shared__ int s_scan[(BR_NQUEUES + 2) * kW];
    __shared__ int s_bad;
    const int tid = threadIdx.x;
    int* hdr = plan;
    int* start = plan + br_plan_off_start();
    int* len = plan + br_plan_off_len(B, M);
    int* tok = plan + br_plan_off_tok(B, M);
    int* prev_tiles = plan + br_plan_off_prev(B, M);
    int* tbase = plan + br_plan_off_tbase(B, M);
    int2* tiles = reinterpret_cast<int2*>(plan + br_plan_off_tiles(B, M));
    const int tps = br_plan_tps(M, H);
    const int max_items = br_plan_max_items(B, M, H, T);
    BrItem* items = reinterpret_cast<BrItem*>(plan + br_plan_off_items(B, M, H, T));
    BrComb* comb = reinterpret_cast<BrComb*>(plan + br_plan_off_comb(B, M, H, T));
    const int BM = B * M;
    // Every block's length and (further down) queue, staged in LDS once: most of what follows is loops of a single thread
    // over a sequence's blocks, and from global memory every step of those is a round trip of its own.  (Larger batches
    // read the table itself.)
    constexpr int kStage = 8192;
    __shared__ int s_len[kStage];
    __shared__ signed char s_bq[kStage];
    const bool staged = BM <= kStage;

    static_assert(BR_PLAN_HDR <= kPlanThreads, "a thread per word of the header");
    if (tid < BR_PLAN_HDR) hdr[tid] = 0;
    for (int b = tid; b < B; b += kPlanThreads) plan[br_plan_off_meet(B, M, H, T) + b] = 0;
    if (tid == 0) s_bad = 0;
    __syncthreads();
    for (int p = tid; p < BM; p += kPlanThreads) {
        int l = len[p];
        if (l < 0) {
            l = -1 - l;
            len[p] = l;
            s_bad = 1;
        }
        if (staged) s_len[p] = l;
    }
    __syncthreads();
    auto blk_len = [&](int p) -> int { return staged ? s_len[p] : len[p]; };
    auto blk_tiles = [&](int p) -> int { return ceil_div(blk_len(p), BR_BN); };

    // Where each block's first real token sits on the token axis, its first tile descriptor and the descriptors
    // themselves (blocks 0..M-2 of a sequence one after the other): running sums over all blocks, the tiles' relative to
    // the sequence's first block, whose sum is in LDS or, if it lies in an earlier stretch, carried along.
    __shared__ int s_x[kPlanThreads];
    {
        int base_tok = 0, base_tile = 0, carry = 0;
#pragma unroll 1
    for (int p0 = 0; p0 < BM; p0 += kPlanThreads) {
            const int p = p0 + tid, b = p / M, m = p - b * M;
            const bool on = p < BM;
            const int L = on ? blk_len(p) : 0;
            int x[2] = {L, on && m < M - 1 ? ceil_div(L, BR_BN) : 0}, tot[2];
            block_exclusive_scan_n<2>(x, tot, s_scan);
            s_x[tid] = base_tile + x[1];
            __syncthreads();
            if (on) {
                const int tk = packed ? base_tok + x[0] : m * H + start[p];
                const int t = base_tile + x[1] - (b * M >= p0 ? s_x[b * M - p0] : carry);
                tok[p] = tk;
                tbase[p] = t;
                if (m == M - 1) prev_tiles[b] = t;
                else
#pragma unroll 1
                    for (int kt = 0; kt * BR_BN < L; ++kt)
                        tiles[(size_t)b * tps + t + kt] = make_int2(tk + kt * BR_BN, L - kt * BR_BN < BR_BN ? L - kt * BR_BN : BR_BN);
            }
            const int last = (p0 + kPlanThreads - 1) / M * M;
            carry = last >= p0 ? s_x[last - p0] : carry;
            base_tok += tot[0];
            base_tile += tot[1];
        }
    }
    __syncthreads();

    // Work distribution.
    // All items but the query blocks' keep their natural order (sequence, block, query tile) and that list is cut
    // into eight contiguous runs of equal estimated work, one per XCD queue: an XCD then works on a few adjacent
    // blocks at a time (their K/V stay in its L2), and the runs end together, so that no workgroup has to go looking
    // for work in other queues at the end of the kernel (polling the ticket counters there slows the memory accesses
    // of every workgroup still working).  Estimated work of an item: its key tiles plus a constant for set-up and
    // epilogue.  A query block reads the K/V of every earlier block of its sequence: its key walk is cut where those
    // blocks pass from one XCD's run to the next and each stretch is handed to that XCD (at the front of its queue:
    // long items first), so that the walk finds the tiles in the L2 that the blocks' own items fill anyway instead of
    // pulling all K/V of the sequence into a second L2.
    constexpr int kItemOverhead = 2;
    auto item_weight = [&](int nprev_t, int tt, int L) {
        int e = (tt + 1) * T < L ? (tt + 1) * T : L;
        return nprev_t + ceil_div(e, BR_BN) + kItemOverhead;
    };
    int* bq = plan + br_plan_off_bq(B, M);
    __shared__ int s_qfirst[8];
    __shared__ int s_base[BR_NQUEUES], s_nsplit[BR_NQUEUES];
    if (tid < 8) s_qfirst[tid] = 0x7fffffff;
    __syncthreads();

    // Ordinary (not query-block) items of the pair p = (b, m): how many, their weight, the prefix tiles they walk.
    auto ordinary = [&](int p, int& nq, int& npt, int& L) -> int {
        nq = 0; npt = 0; L = 0;
        if (p >= BM) return 0;
        const int b = p / M, m = p - b * M;
        if (m == M - 1) return 0;
        L = blk_len(p);
        nq = ceil_div(L, T);
        npt = br_prev_blocks(m, M) > 0 ? blk_tiles(b * M) : 0;
        int w = 0;
#pragma unroll 1
        for (int tt = 0; tt < nq; ++tt) w += item_weight(npt, tt, L);
        return w;
    };

    // Totals: all items' weight (with the query blocks'), the ordinary items' weight and number.  The thread's own
    // prefixes are kept where there is one stretch (at most kPlanThreads blocks, any batch but the largest).
    const bool one_stretch = BM <= kPlanThreads;
    long long w_all = 0, w_ord = 0;
    int n_ord = 0, my_x = 0, my_w = 0;
#pragma unroll 1
    for (int p0 = 0; p0 < BM; p0 += kPlanThreads) {
        const int p = p0 + tid;
        int nq, npt, L;
        int w = ordinary(p, nq, npt, L), wq = 0;
        if (p < BM && p % M == M - 1) {
            const int b = p / M, Lq = blk_len(p), pt = M > 1 ? prev_tiles[b] : 0;
#pragma unroll 1
            for (int tt = 0; tt * T < Lq; ++tt) wq += item_weight(pt, tt, Lq);
        }
        int x[3] = {w + wq, w, nq}, tot[3];
        block_exclusive_scan_n<3>(x, tot, s_scan);
        w_all += tot[0];
        w_ord += tot[1];
        n_ord += tot[2];
        my_w = x[1];
        my_x = x[2];
    }
    // the run of equal weight (of eight) that an item with the weight w before it falls into: w * 8 / total, without dividing
    auto run_of = [&](long long w) -> int {
        int q = 0;
#pragma unroll
        for (int g = 1; g < 8; ++g) q += w_ord > 0 && w >= (w_ord * g + 7) >> 3;
        return q;
    };
    // the thread's prefixes (items, weight) in stretch p0, whose base the caller carries
    auto prefixes = [&](int p, int& nq, int& npt, int& L, int& base_x, long long& base_w, int& off_x, long long& off_w) {
        const int w = ordinary(p, nq, npt, L);
        if (one_stretch) {
            off_x = my_x;
            off_w = my_w;
            return;
        }
        int x[2] = {nq, w}, tot[2];
        block_exclusive_scan_n<2>(x, tot, s_scan);
        off_x = base_x + x[0];
        off_w = base_w + x[1];
        base_x += tot[0];
        base_w += tot[1];
    };

    // Queue of every ordinary item (by the weight before it), first item of every queue, queue of every block (that of
    // its first item).
    {
        int base_x = 0;
        long long base_w = 0;
#pragma unroll 1
    for (int p0 = 0; p0 < BM; p0 += kPlanThreads) {
            const int p = p0 + tid;
            int nq, npt, L, off_x;
            long long off_w;
            prefixes(p, nq, npt, L, base_x, base_w, off_x, off_w);
            int q0 = -1;
#pragma unroll 1
            for (int k = 0; k < nq; ++k) {
                const int q = run_of(off_w);
                if (k == 0) q0 = q;
                atomicMin(&s_qfirst[q], off_x + k);
                off_w += item_weight(npt, nq - 1 - k, L);
            }
            if (p < BM) {
                bq[p] = q0;
                if (staged) s_bq[p] = (signed char)q0;
            }
        }
    }
    __syncthreads();
    if (tid == 0) {
        // a queue that received no item starts where the next one starts
        int nxt = n_ord;
        for (int g = 7; g >= 0; --g) {
            if (s_qfirst[g] == 0x7fffffff) s_qfirst[g] = nxt;
            nxt = s_qfirst[g];
        }
    }
    __syncthreads();

    // The stretches of a sequence's earlier blocks that one XCD's queue owns: first tile, tiles, queue.  The queues
    // follow the blocks' order, so there are at most eight; a stretch shorter than min_seg tiles stays with the next
    // one.  They are in LDS, a list for each of the kWalkers threads that walk sequences (a dynamically indexed local
    // array would be scratch memory, a round trip of microseconds per access; registers picked by unrolled compares made
    // this kernel 54 KB of code, most of its time spent fetching instructions it runs once).
    constexpr int kWalkers = 128;
    __shared__ int s_seg_lo[kWalkers][8], s_seg_n[kWalkers][8];
    __shared__ signed char s_seg_q[kWalkers][8];
    const int me = tid & (kWalkers - 1);
    auto build_segs = [&](int b, int min_seg) -> int {
        int n_seg = 0, seg_lo = 0, seg_n = 0, seg_q = -1;
        auto push = [&]() {
            s_seg_lo[me][n_seg] = seg_lo;
            s_seg_n[me][n_seg] = seg_n;
            s_seg_q[me][n_seg] = (signed char)seg_q;
            ++n_seg;
        };
        // (four blocks' table entries read together, and from LDS or from memory, not from where a select points: one thread's
        // reads one after the other were most of this loop)
        auto scan = [&](const auto* lens, const auto* queues) {
            constexpr int U = 4;
#pragma unroll 1
            for (int m0 = 0; m0 < M - 1; m0 += U) {
                int tokens[U], q[U];
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    const int m = m0 + k < M - 1 ? m0 + k : M - 1;   // (past the last: the query block, which is not asked)
                    tokens[k] = lens[m];
                    q[k] = queues[m];
                }
#pragma unroll
                for (int k = 0; k < U; ++k) {
                    if (tokens[k] == 0 || m0 + k >= M - 1) continue;
                    if (seg_q >= 0 && q[k] != seg_q && seg_n >= min_seg && n_seg < 7) {
                        push();
                        seg_lo += seg_n;
                        seg_n = 0;
                        seg_q = q[k];
                    }
                    if (seg_q < 0) seg_q = q[k];
                    seg_n += ceil_div(tokens[k], BR_BN);
                }
            }
        };
        if (staged) scan(s_len + b * M, s_bq + b * M);
        else scan(len + b * M, bq + b * M);
        if (seg_q >= 0) push();
        return n_seg;
    };
    // The key walk of query tile tt of sequence b's query block, stretch by stretch in walk order: fn(first tile, tiles, pieces,
    // queue).  Every stretch is cut into pieces of at most `chunk` tiles; the query block's own tiles go with the
    // last stretch (a sequence without earlier keys has them alone, in the global queue).  Returns the number of pieces.
    auto walk_stretches = [&](int b, int tt, int chunk, int n_seg, auto&& fn) -> int {
        const int L = blk_len(b * M + M - 1);
        const int e = (tt + 1) * T < L ? (tt + 1) * T : L;
        const int nself = ceil_div(e, BR_BN);
        int count = 0;
#pragma unroll 1
        for (int i = 0; i < (n_seg > 0 ? n_seg : 1); ++i) {
            const int lo = n_seg > 0 ? s_seg_lo[me][i] : 0, q = n_seg > 0 ? s_seg_q[me][i] : BR_GLOBAL_QUEUE;
            const int n = (n_seg > 0 ? s_seg_n[me][i] : 0) + (i >= n_seg - 1 ? nself : 0);
            int parts = ceil_div(n, chunk);
            parts = parts < 1 ? 1 : parts;
            fn(lo, n, parts, q);
            count += parts;
        }
        return count;
    };
    // ... how many pieces there are
    auto count_pieces = [&](int b, int tt, int chunk, int n_seg) -> int { return walk_stretches(b, tt, chunk, n_seg, [](int, int, int, int) {}); };
    // a[q] += n for a register-resident array of the nine queues; returns the value before
    auto bump = [](int (&a)[BR_NQUEUES], int q, int n) -> int {
        int r = 0;
#pragma unroll
        for (int i = 0; i < BR_NQUEUES; ++i)
            if (i == q) {
                r = a[i];
                a[i] = r + n;
            }
        return r;
    };

    // Length of a piece.  The walks are cut so that the batch has enough items to fill the grid, and no further: every
    // piece costs a set-up, an epilogue and a set of partials to write and merge, while a long piece still ends with the
    // others because the pieces are handed out first.  So: the estimated work per workgroup (all items' key tiles plus
    // their constant, over the workgroups that run side by side) less one ordinary item - the workgroup that takes a
    // piece still has to fit one of those before the kernel ends, which is what decides at a batch of one - and at
    // least BR_MIN_CHUNK, or, where the other items leave compute units without a workgroup, as little as gives each of those
    // a piece (a walk of four tiles is then what the kernel waits for: 8 documents of 64 tokens, 8/2 heads, D = 64, in fp32
    // 28 -> 15 us with pieces of one tile, 14 ragged documents in fp16 17.6 -> 14.0; as short as that with twice the items
    // - two workgroups per unit - walks of 50 tiles lost a fifth to the merge and to each other); and long enough that the batch's pieces fit the pool of partial slots: lengthen until they
    // do, and where longer pieces no longer help (what remains are the cuts between XCDs) join short stretches to
    // their neighbours; with both beyond every walk's length nothing is split at all, so this ends.
    int chunk = (int)(w_all / (par > 0 ? par : 1)) - (n_ord > 0 ? (int)(w_ord / n_ord) : 0);
    int min_chunk = BR_MIN_CHUNK;
    if (n_ord < par / 2) {
        const int idle = par / 2 - n_ord, c = (int)((w_all - w_ord + idle - 1) / idle);
        min_chunk = c < 1 ? 1 : (c < BR_MIN_CHUNK ? c : BR_MIN_CHUNK);
    }
    chunk = chunk < min_chunk ? min_chunk : chunk;
    int min_seg = min_chunk, need_before = 0x7fffffff;
    // Thread tid of the first kWalkers walks the sequences tid, tid + kWalkers, ...  With one sequence per thread (every
    // batch but the largest) its stretch list is built once; otherwise it is rebuilt at every visit.
    int segs = 0;
    const bool one_each = B <= kWalkers;
    if (one_each && tid < B) segs = build_segs(tid, min_seg);
    auto for_my_sequences = [&](auto&& fn) {
#pragma unroll 1
        for (int b = tid < kWalkers ? tid : B; b < B; b += kWalkers) {
            if (!one_each) segs = build_segs(b, min_seg);
            fn(b, blk_len(b * M + M - 1));
        }
    };
    for (;;) {
        int mine = 0;
        for_my_sequences([&](int b, int Lq) {
#pragma unroll 1
            for (int tt = 0; tt * T < Lq; ++tt) {
                const int ns = count_pieces(b, tt, chunk, segs);
                mine += ns > 1 ? ns : 0;
            }
        });
        int need, one[1] = {mine}, tot1[1];
        block_exclusive_scan_n<1>(one, tot1, s_scan);
        need = tot1[0];
        if (need <= pool) break;
        if (need >= need_before) {
            min_seg *= 2;
            if (one_each && tid < B) segs = build_segs(tid, min_seg);
        }
        need_before = need;
        if (chunk < (1 << 24)) chunk += (chunk + 1) / 2;
    }

    // Layout of the items array: [global queue][queue 0: its pieces, its ordinary items][queue 1: ...] ...
    // Every thread counts the pieces of its sequences' query blocks per queue; scans give it its offsets.
    int my_cnt[BR_NQUEUES], my_off[BR_NQUEUES], my_comb = 0, my_slots = 0;
#pragma unroll
    for (int q = 0; q < BR_NQUEUES; ++q) my_cnt[q] = 0;
    for_my_sequences([&](int b, int Lq) {
#pragma unroll 1
        for (int tt = 0; tt * T < Lq; ++tt) {
            const int ns = walk_stretches(b, tt, chunk, segs, [&](int, int, int parts, int q) { bump(my_cnt, q, parts); });
            my_comb += ns > 1;
            my_slots += ns > 1 ? ns : 0;
        }
    });
    // (all eleven counts through one scan)
    int sc[BR_NQUEUES + 2], sc_tot[BR_NQUEUES + 2];
#pragma unroll
    for (int q = 0; q < BR_NQUEUES; ++q) sc[q] = my_cnt[q];
    sc[BR_NQUEUES] = my_comb;
    sc[BR_NQUEUES + 1] = my_slots;
    block_exclusive_scan_n<BR_NQUEUES + 2>(sc, sc_tot, s_scan);
#pragma unroll
    for (int q = 0; q < BR_NQUEUES; ++q) {
        my_off[q] = sc[q];
        if (tid == 0) s_nsplit[q] = sc_tot[q];
    }
    const int off_comb = sc[BR_NQUEUES], off_slot = sc[BR_NQUEUES + 1];
    const int n_comb_total = sc_tot[BR_NQUEUES], n_slot_total = sc_tot[BR_NQUEUES + 1];
    __syncthreads();
    if (tid == 0) {
        int nxt = s_nsplit[BR_GLOBAL_QUEUE];
        for (int g = 0; g < 8; ++g) {
            s_base[g] = nxt;
            const int ord = (g < 7 ? s_qfirst[g + 1] : n_ord) - s_qfirst[g];
            hdr[BR_PH_QOFF + g] = nxt;
            hdr[BR_PH_QCOUNT + g] = s_nsplit[g] + ord;
            nxt += s_nsplit[g] + ord;
        }
        s_base[BR_GLOBAL_QUEUE] = 0;
        hdr[BR_PH_QOFF + BR_GLOBAL_QUEUE] = 0;
        hdr[BR_PH_QCOUNT + BR_GLOBAL_QUEUE] = s_nsplit[BR_GLOBAL_QUEUE];
        hdr[BR_PH_NITEMS] = nxt;
        hdr[BR_PH_NCOMB] = n_comb_total;
        hdr[BR_PH_PACKED] = packed;
        hdr[BR_PH_NONCONTIG] = s_bad;
        hdr[BR_PH_MAX_ITEMS] = max_items;
        hdr[BR_PH_MAX_COMB] = br_plan_max_comb(B);
        hdr[BR_PH_T] = T;
        hdr[BR_PH_POOL] = pool;
        hdr[BR_PH_NSLOTS] = n_slot_total;
        hdr[BR_PH_MEET] = (int)br_plan_off_meet(B, M, H, T);
        hdr[BR_PH_B] = B;
    }
    __syncthreads();

    // Ordinary items: queue g's start at s_base[g] + its pieces, in their natural order.
    {
        int base_x = 0;
        long long base_w = 0;
#pragma unroll 1
    for (int p0 = 0; p0 < BM; p0 += kPlanThreads) {
            const int p = p0 + tid;
            int nq, npt, L, off_x;
            long long off_w;
            prefixes(p, nq, npt, L, base_x, base_w, off_x, off_w);
            if (nq > 0) {
                const int b = p / M, m = p - b * M;
                BrItem it;
                it.b = b; it.m = m; it.pe = br_prev_blocks(m, M);
                it.len_m = L; it.start_m = start[p]; it.len0 = len[b * M]; it.start0 = start[b * M];
                it.tok_m = tok[p]; it.tok0 = tok[b * M];
                it.pad[0] = it.pad[1] = 0;
                it.nprev = npt;
                it.f_lo = 0; it.ntiles = 0x7fffffff; it.slot = -1;
                // a block's query tiles are handed out from the last (the longest walk) to the first: what a queue
                // ends on are short items
#pragma unroll 1
            for (int k = 0; k < nq; ++k) {
                    const int tt = nq - 1 - k;
                    const int q = run_of(off_w);
                    it.t0 = tt * T;
                    items[s_base[q] + s_nsplit[q] + (off_x + k - s_qfirst[q])] = it;
                    off_w += item_weight(npt, tt, L);
                }
            }
        }
    }
    // The query blocks' pieces (the thread of every sequence, in the order and at the offsets of the counting pass above).
    int pos[BR_NQUEUES];
#pragma unroll
    for (int q = 0; q < BR_NQUEUES; ++q) pos[q] = s_base[q] + my_off[q];
    int slot = off_slot, ci = off_comb;
    for_my_sequences([&](int b, int L) {
        const int pq = b * M + M - 1;
        BrItem it;
        it.b = b; it.m = M - 1; it.pe = br_prev_blocks(M - 1, M);
        it.len_m = L; it.start_m = start[pq]; it.len0 = len[b * M]; it.start0 = start[b * M];
        it.tok_m = tok[pq]; it.tok0 = tok[b * M];
        it.pad[0] = it.pad[1] = 0;
        it.nprev = M > 1 ? prev_tiles[b] : 0;
#pragma unroll 1
        for (int tt = 0; tt * T < L; ++tt) {
            const int ns = count_pieces(b, tt, chunk, segs);
            if (ns > 1) {
                BrComb cb;
                cb.b = b; cb.t0 = tt * T; cb.slot0 = slot; cb.nsplit = ns;
                cb.len_m = L; cb.tok_m = it.tok_m; cb.pad[0] = cb.pad[1] = 0;
                comb[ci++] = cb;
            }
            it.t0 = tt * T;
            walk_stretches(b, tt, chunk, segs, [&](int lo, int n, int parts, int q) {
                // (piece s: tiles s n / parts to (s + 1) n / parts, by the remainder carried along - a division is forty instructions of
                // one thread)
                const int each = n / parts, rest = n - each * parts;
                BrItem* to = items + bump(pos, q, parts);
                int carry = 0;
                it.f_lo = lo;
#pragma unroll 1
                for (int s = 0; s < parts; ++s) {
                    carry += rest;
                    const int more = carry >= parts ? 1 : 0;
                    carry -= more ? parts : 0;
                    it.ntiles = ns > 1 ? each + more : 0x7fffffff;
                    it.slot = ns > 1 ? slot++ : -1;
                    *to++ = it;
                    it.f_lo += each + more;
                }
            });
        }
    });
}

// Block table straight from per-block lengths (left- or right-aligned spans): the packed-layout
// entry, where the caller already knows the lengths and there is no (B, M, H) mask to scan.
__global__ void br_block_table_from_len_kernel(const int* __restrict__ lens, int BM, int H, int left_padded,
                                               int* __restrict__ start, int* __restrict__ len) {
    int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= BM) return;
    int l = lens[p];
    l = l < 0 ? 0 : (l > H ? H : l);
    len[p] = l;
    start[p] = left_padded ? H - l : 0;
}

// Ticket counters, the count of workgroups that have left and the score counters back to zero (what the last workgroups
// of a launch that ran to its end do themselves).
__global__ void br_plan_rearm_kernel(int* __restrict__ plan) {
    const int i = threadIdx.x;
    if (i < BR_NQUEUES) plan[br_qticket(i)] = 0;
    if (i == BR_NQUEUES) plan[BR_PH_DONE] = 0;
    for (int b = i; b < plan[BR_PH_B]; b += blockDim.x) plan[plan[BR_PH_MEET] + b] = 0;
}

}  // namespace

void br_launch_plan_rearm(int* plan, hipStream_t stream) {
    hipLaunchKernelGGL(br_plan_rearm_kernel, dim3(1), dim3(64), 0, stream, plan);
}

void br_launch_plan(const uint8_t* valid, const int* lens, int left_padded, int packed, int B, int M, int H, int T, int par, int pool,
                    int* plan, hipStream_t stream) {
    int* start = plan + br_plan_off_start();
    int* len = plan + br_plan_off_len(B, M);
    const int BM = B * M;
    if (valid) {
        int waves_per_wg = 4;
        hipLaunchKernelGGL(br_block_table_kernel, dim3((BM + waves_per_wg - 1) / waves_per_wg), dim3(256), 0, stream, valid,
                           BM, H, start, len);
    } else {
        hipLaunchKernelGGL(br_block_table_from_len_kernel, dim3((BM + 255) / 256), dim3(256), 0, stream, lens, BM, H,
                           left_padded, start, len);
    }
    hipLaunchKernelGGL(br_plan_kernel, dim3(1), dim3(kPlanThreads), 0, stream, plan, B, M, H, T, packed, par, pool);
}
