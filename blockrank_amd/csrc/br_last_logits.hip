// The reference's s_last tensor - scale * q.k of the query block's last rows against every key slot, for callers that
// still want it (blockrank_std_attention.py:639-645) - and its gradient, through which the auxiliary attention loss
// trains (trainer.py:91-101).  Both are contractions, so both run on the matrix cores: the logits on the 16-bit
// (fp32 inputs: fp32) matrix instruction over the head dim, the gradients on the fp32 one (v_mfma_f32_32x32x2_f32)
// over rows and keys, since the incoming gradient is fp32 and is not to be rounded.
#include "br_mma.h"

namespace {

typedef br_f32x16v f32x16;
__device__ inline f32x16 zero16() { return br_zero16(); }
__device__ inline f32x16 mma2(float a, float b, f32x16 c) { return br_mma2(a, b, c); }

constexpr int kGroupHeads = 2;      // a 32-row operand holds 16 row slots (rows 0..R-1 used) of two heads

struct BrLogitsParams {
    const void* q;
    const void* k;
    const int* plan;
    const int* rows;        // (B, R) positions inside the query block
    float* logits;          // (B, Nq, R, M*H)
    long long sq_b, sq_h, sq_t, sk_b, sk_h, sk_t;
    int B, Nq, Nkv, M, H, R, T;
    float scale, neg;
};

// A wave holds 32 key slots (lane = key) and goes through the kv head's query heads two at a time: A = the two heads'
// 16 row slots, B = the keys, so that a register of the result is one (head, row) and its 32 lanes are consecutive
// slots - 128-byte stores.  Write-bound: at B=2, 14 blocks of 256 slots, 32/8 heads, 16 rows (14.7 MB written) 11.5 us,
// 46 us as one thread per key on the vector ALU.
template <typename T, int D>
__global__ __launch_bounds__(256) void br_last_logits_kernel(BrLogitsParams p) {
    constexpr int NP = D / BrPiece<T>::STEP;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.T);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const int b = blockIdx.z, kvh = blockIdx.y, G = p.Nq / p.Nkv;
    const int S = p.M * p.H;
    const int slot0 = blockIdx.x * 128 + wave * 32;
    if (slot0 >= S) return;
    const int key = slot0 + ln, kk = key < S ? key : S - 1;
    const int blk = kk / p.H, j = kk - blk * p.H;
    const int st = pv.start[b * p.M + blk], len = pv.len[b * p.M + blk];
    const bool kvalid = key < S && j >= st && j < st + len;
    // (a slot that holds no real token has no key row to read - in a packed layout not even storage; its product is 0
    // and its logit the masked value)
    uint4 kf[NP];
    {
        const T* krow = reinterpret_cast<const T*>(p.k) + (long long)b * p.sk_b + (long long)kvh * p.sk_h +
                        (long long)(kvalid ? pv.tok[b * p.M + blk] + j - st : 0) * p.sk_t + lh * BrPiece<T>::N;
#pragma unroll
        for (int c = 0; c < NP; ++c) kf[c] = kvalid ? *reinterpret_cast<const uint4*>(krow + c * BrPiece<T>::STEP) : uint4{0u, 0u, 0u, 0u};
    }
    const int mq = b * p.M + p.M - 1;
    const int st_q = pv.start[mq], len_q = pv.len[mq], tok_q = pv.tok[mq];
    const int r = ln & 15;
    const int pos_r = r < p.R ? p.rows[b * p.R + r] : -1;
    const int pos = pos_r >= st_q && pos_r < st_q + len_q ? pos_r : -1;      // -1: no such row, or padding
    for (int h0 = 0; h0 < G; h0 += kGroupHeads) {
        const int h = h0 + (ln >> 4);
        const bool on = pos >= 0 && h < G;
        const T* qrow = reinterpret_cast<const T*>(p.q) + (long long)b * p.sq_b + (long long)(kvh * G + (on ? h : 0)) * p.sq_h +
                        (long long)(tok_q + (on ? pos - st_q : 0)) * p.sq_t + lh * BrPiece<T>::N;
        uint4 qf[NP];
#pragma unroll
        for (int c = 0; c < NP; ++c) qf[c] = on ? *reinterpret_cast<const uint4*>(qrow + c * BrPiece<T>::STEP) : uint4{0u, 0u, 0u, 0u};
        f32x16 s = zero16();
#pragma unroll
        for (int c = 0; c < NP; ++c) s = BrPiece<T>::mma(qf[c], kf[c], s);
        float* out = p.logits + ((long long)b * p.Nq + kvh * G + h0) * p.R * S + key;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            // register v of lane half lh is row slot 8 (v/4) + 4 lh + v%4 of the pair of heads
            const int i0 = 8 * (v >> 2) + (v & 3);
            const int p_lo = __builtin_amdgcn_readlane(pos, i0), p_hi = __builtin_amdgcn_readlane(pos, i0 + 4);
            const int ps = lh ? p_hi : p_lo, i = i0 + 4 * lh, hh = i >> 4, rr = i & 15;
            const bool allow = kvalid && ps >= 0 && (blk < p.M - 1 || j <= ps);
            if (rr < p.R && h0 + hh < G && key < S) out[(long long)(hh * p.R + rr) * S] = s[v] * p.scale + (allow ? 0.f : p.neg);
        }
    }
}

// ---- gradient ----
// s[b,n,r,key] = scale * q[b,n,row_r] . k[b,n/G,key] + constant for real rows and real keys (the additive mask is a
// constant, so disallowed real keys carry gradient like the reference's additive-mask logits do); slots without a token
// and rows that are padding do not depend on q or k at all.
struct BrLogitsBwdParams {
    const float* ds;        // (B, Nq, R, M*H) gradient of the logits
    const void* q;
    const void* k;
    const int* plan;
    const int* rows;        // (B, R) positions inside the query block
    void* dq;               // only the chosen rows are written
    void* dk;               // every key token is written
    float* part;            // [chunks][B][Nq][R][D] sums of dq per chunk of key slots (chunks > 1)
    long long sq_b, sq_h, sq_t, sk_b, sk_h, sk_t;
    long long dq_b, dq_h, dq_t, dk_b, dk_h, dk_t;
    int B, Nq, Nkv, M, H, R, T;
    int chunks, chunk_slots;
    int add;                // 1: add to what dq and dk hold (the attention's own gradients) instead of storing
    int vec;                // dk's rows and strides allow stores of a lane's D/32 dims at once
    float scale;
};

// One dim group: N = D/32 consecutive elements per lane, so that 32 lanes cover a row.
template <typename T, int N>
using Dims = T __attribute__((ext_vector_type(N)));
template <typename T, int N>
__device__ inline void load_dims(const T* src, float (&x)[N]) {
    const Dims<T, N> v = *reinterpret_cast<const Dims<T, N>*>(src);
#pragma unroll
    for (int i = 0; i < N; ++i) x[i] = (float)v[i];
}

// dk[key] = scale * sum over the kv head's query heads n and rows r of ds[n, r, key] * q[n, row_r].  A wave owns 32 key
// slots: A = ds^T (row = key: the loads run along the slots), B = the query rows out of LDS (column ln holds dims
// N ln .. N ln + N - 1, one accumulator per element, so that a key's row is stored by 32 lanes in one piece).
// Reads ds once, dk once or twice: bandwidth-bound where most of ds is zero - the ranking loss sends something back through two
// of sixteen rows, and two pairs of which a wave holds zeros alone cost no products (unless a query row is not finite: zero times
// that is NaN) -, bound by the fp32 matrix rate where nothing is.  The pointers are advanced, not kept (two waves per SIMD: with
// one address per load and row it was one, 30 us of a launch of its own where this is 15: B=2, 14 blocks of 250 slots, 32/8
// heads, 16 rows).
template <typename T, int D>
__device__ inline void last_logits_dk(const BrLogitsBwdParams& p, int tile, int kvh, float* qs, int* tokl) {
    constexpr int N = D / 32, QROWS = 64;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.T);
    const int b = blockIdx.z, G = p.Nq / p.Nkv;
    const int S = p.M * p.H;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const bool packed = pv.hdr[BR_PH_PACKED] != 0;
    if (threadIdx.x < 128) {
        // where the slot's gradient goes: its token, a padded slot (gets the zeros its sums are), or nowhere
        const int key = tile * 128 + threadIdx.x;
        int t = -1;
        if (key < S) {
            const int blk = key / p.H, j = key - blk * p.H;
            const int st = pv.start[b * p.M + blk], len = pv.len[b * p.M + blk];
            if (j >= st && j < st + len) t = pv.tok[b * p.M + blk] + j - st;
            else if (!packed && !p.add) t = -2 - key;
        }
        tokl[threadIdx.x] = t;
    }
    const int mq = b * p.M + p.M - 1;
    const int st_q = pv.start[mq], len_q = pv.len[mq], tok_q = pv.tok[mq];
    const int key = tile * 128 + wave * 32 + ln;
    f32x16 acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = zero16();
    const int hc = QROWS / p.R;                                  // heads per pass
    for (int h0 = 0; h0 < G; h0 += hc) {
        const int n = (h0 + hc <= G ? hc : G - h0) * p.R;        // (head, row) pairs of this pass, consecutive in ds
        __syncthreads();                                         // (tokl on the first pass; qs read on the others)
        const bool on = tokl[wave * 32 + ln] >= 0;
        const float* dsp = p.ds + ((long long)b * p.Nq + kvh * G + h0) * p.R * S + (on ? key : 0) + (lh < n ? (long long)lh * S : 0);
        // all of the pass's ds values are requested before the query rows are staged (pairs past the last one read it again:
        // no branch around a load)
        float a[QROWS / 2];
#pragma unroll
        for (int u = 0; u < QROWS / 2; ++u) {
            a[u] = on && 2 * u + lh < n ? *dsp : 0.f;
            dsp += 2 * u + 2 + lh < n ? 2 * (long long)S : 0;
        }
        constexpr int E = BrPiece<T>::N, PPR = D / E;              // 16-byte pieces per row
        int odd = 0;
#pragma unroll 2
        for (int i0 = 0; i0 < QROWS * PPR; i0 += 256) {
            const int i = i0 + threadIdx.x, jq = i / PPR, c = i - jq * PPR;
            const int h = jq < n ? jq / p.R : 0, pos = p.rows[b * p.R + (jq < n ? jq - h * p.R : 0)];
            const bool row_on = jq < n && pos >= st_q && pos < st_q + len_q;
            float x[E];
            load_dims<T, E>(reinterpret_cast<const T*>(p.q) + (long long)b * p.sq_b + (long long)(kvh * G + h0 + h) * p.sq_h +
                                (long long)(row_on ? tok_q + pos - st_q : (len_q > 0 ? tok_q : 0)) * p.sq_t + c * E, x);
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const float y = row_on ? x[e] * p.scale : 0.f;
                odd |= !(fabsf(y) < INFINITY);
                qs[jq * D + c * E + e] = y;
            }
        }
        odd = __syncthreads_or(odd);
#pragma unroll
        for (int u = 0; u < QROWS / 2; ++u) {
            if (2 * u >= n) break;
            const float au = a[u];
            if (!odd && __ballot(au != 0.f) == 0) continue;      // (zeros times finite numbers)
            float x[N];
            load_dims<float, N>(qs + (2 * u + lh) * D + N * ln, x);
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i] = mma2(au, x[i], acc[i]);
        }
    }
    // where the rows go; what eight of them are added to is requested before the first of the eight is stored
    T* const base = reinterpret_cast<T*>(p.dk) + (long long)b * p.dk_b + (long long)kvh * p.dk_h + N * ln;
    const bool vec_add = p.vec && p.add;
#pragma unroll
    for (int v0 = 0; v0 < 16; v0 += 8) {
        int t[8];
        Dims<T, N> old[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int v = v0 + e;
            t[e] = tokl[wave * 32 + 8 * (v >> 2) + 4 * lh + (v & 3)];
            if (vec_add) old[e] = *reinterpret_cast<const Dims<T, N>*>(base + (long long)(t[e] < 0 ? 0 : t[e]) * p.dk_t);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if (t[e] == -1) continue;
            T* dst = base + (long long)(t[e] >= 0 ? t[e] : -2 - t[e]) * p.dk_t;
            if (p.vec) {
                Dims<T, N> y;
#pragma unroll
                for (int i = 0; i < N; ++i) y[i] = (T)(vec_add ? (float)old[e][i] + acc[i][v0 + e] : acc[i][v0 + e]);
                *reinterpret_cast<Dims<T, N>*>(dst) = y;
            } else {
#pragma unroll
                for (int i = 0; i < N; ++i) dst[i] = (T)(p.add ? (float)dst[i] + acc[i][v0 + e] : acc[i][v0 + e]);
            }
        }
    }
}

// The dq row of (sequence, head, row) from its sum; rows named twice are summed into their first occurrence (value(r)
// is the sum of row r).
template <typename T, typename F>
__device__ inline void put_dq(const BrLogitsBwdParams& p, const BrPlanView& pv, int b, int n, int r, int d, F&& value) {
    const int mq = b * p.M + p.M - 1;
    const int st = pv.start[mq], pos = p.rows[b * p.R + r];
    if (pos < st || pos >= st + pv.len[mq]) return;              // a padded row: its logits do not depend on q
    for (int r2 = 0; r2 < r; ++r2)
        if (p.rows[b * p.R + r2] == pos) return;
    float v = value(r);
    for (int r2 = r + 1; r2 < p.R; ++r2)
        if (p.rows[b * p.R + r2] == pos) v += value(r2);
    T* dst = reinterpret_cast<T*>(p.dq) + (long long)b * p.dq_b + (long long)n * p.dq_h + (long long)(pv.tok[mq] + pos - st) * p.dq_t + d;
    v *= p.scale;
    *dst = (T)(p.add ? (float)*dst + v : v);
}

// Sums over a chunk of the key slots of ds[n, r, key] * k[key] for two heads of a kv head.  A = ds (row = row slot of
// the pair of heads; a lane's 16-byte piece holds four consecutive slots), B = the key rows (column ln: N consecutive
// dims).  The four waves of a workgroup take turns of 64 slots and meet in LDS at the end.  One workgroup per (sequence,
// head) walking all slots took 1313 us at B=2, 14 blocks of 256 slots, 32/8 heads (64 workgroups, a chain of dependent
// two-byte loads); the slots are therefore cut into chunks until the grid covers the chip: 19 us alone, and 6 for their sum.
// 32 padded slots cost nothing.
template <typename T, int D>
__device__ inline void last_logits_dq(const BrLogitsBwdParams& p, int chunk, int kvh, int h0, float* red, int* tokl) {
    constexpr int N = D / 32;
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.T);
    const int G = p.Nq / p.Nkv, b = blockIdx.z;
    const int S = p.M * p.H;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, ln = lane & 31, lh = lane >> 5;
    const int r = ln & 15, h = h0 + (ln >> 4);
    const bool row_on = r < p.R && h < G;
    const float* dsp = p.ds + (((long long)b * p.Nq + kvh * G + (row_on ? h : 0)) * p.R + (row_on ? r : 0)) * S;
    const T* kb = reinterpret_cast<const T*>(p.k) + (long long)b * p.sk_b + (long long)kvh * p.sk_h + N * ln;
    const bool quads = (S & 3) == 0 && (reinterpret_cast<uintptr_t>(p.ds) & 15) == 0;                             // a row's 16-byte pieces are aligned
    f32x16 acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i) acc[i] = zero16();
    const int c0 = chunk * p.chunk_slots, c1 = c0 + p.chunk_slots < S ? c0 + p.chunk_slots : S;
    for (int s0 = c0; s0 < c1; s0 += 256) {
        __syncthreads();
        {
            const int key = s0 + threadIdx.x;
            int t = -1;
            if (key < c1) {
                const int blk = key / p.H, j = key - blk * p.H;
                const int st = pv.start[b * p.M + blk], len = pv.len[b * p.M + blk];
                if (j >= st && j < st + len) t = pv.tok[b * p.M + blk] + j - st;
            }
            tokl[threadIdx.x] = t;
        }
        __syncthreads();
        // four steps of eight slots at a time: their loads are all in flight before the first product
        constexpr int U = 4;
#pragma unroll 1
        for (int k0 = wave * 64; k0 < wave * 64 + 64; k0 += 8 * U) {
            if (__ballot(tokl[k0 + ln] >= 0) == 0) continue;     // padding
            float a[U][4];
            Dims<T, N> kr[U][4];
            bool real[U][4];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int kl = k0 + 8 * u + 4 * lh;
#pragma unroll
                for (int e = 0; e < 4; ++e) a[u][e] = 0.f;
                if (row_on && quads && s0 + kl < c1) load_dims<float, 4>(dsp + s0 + kl, a[u]);
                if (row_on && !quads) {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (s0 + kl + e < c1) a[u][e] = dsp[s0 + kl + e];
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int t = tokl[kl + e];
                    real[u][e] = t >= 0;
                    kr[u][e] = *reinterpret_cast<const Dims<T, N>*>(kb + (long long)(t >= 0 ? t : 0) * p.sk_t);   // (token 0 is always there to read)
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float av = real[u][e] ? a[u][e] : 0.f;
#pragma unroll
                    for (int i = 0; i < N; ++i) acc[i] = mma2(av, real[u][e] ? (float)kr[u][e][i] : 0.f, acc[i]);
                }
        }
    }
    // waves 2, 3 -> 0, 1; wave 1 -> 0; wave 0 leaves the total
    auto cell = [&](int buf, int v) -> float* { return red + (buf * 32 + 8 * (v >> 2) + 4 * lh + (v & 3)) * D + N * ln; };
    auto leave = [&](int buf) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int i = 0; i < N; ++i) cell(buf, v)[i] = acc[i][v];
    };
    auto take = [&](int buf) {
#pragma unroll
        for (int v = 0; v < 16; ++v)
#pragma unroll
            for (int i = 0; i < N; ++i) acc[i][v] += cell(buf, v)[i];
    };
    __syncthreads();
    if (wave >= 2) leave(wave - 2);
    __syncthreads();
    if (wave < 2) take(wave);
    __syncthreads();
    if (wave == 1) leave(0);
    __syncthreads();
    if (wave == 0) take(0);
    __syncthreads();
    if (wave == 0) leave(0);
    __syncthreads();
    for (int i = threadIdx.x; i < 32 * D; i += 256) {
        const int row = i / D, d = i - row * D, rr = row & 15, hh = h0 + (row >> 4);
        if (rr >= p.R || hh >= G) continue;
        const int n = kvh * G + hh;
        if (p.chunks > 1) p.part[((((long long)chunk * p.B + b) * p.Nq + n) * p.R + rr) * D + d] = red[i];
        else put_dq<T>(p, pv, b, n, rr, d, [&](int r2) { return red[((row & 16) + r2) * D + d]; });
    }
}

// Both at once - neither fills the chip, and what they read twice is still in cache: the first workgroups take dq's chunks, the
// others dk's tiles of keys.  B=2, 14 blocks of up to 250 slots, 32/8 heads, 16 rows: 27 us where two of the rows carry
// a gradient, 38 where all do (31 + 20 in two launches); 8 x 12 documents of 384 to 512 tokens 239 (205 + 98).
template <typename T, int D>
__global__ __launch_bounds__(256, 2) void br_last_logits_bwd_kernel(BrLogitsBwdParams p) {
    __shared__ __attribute__((aligned(16))) float rows[64 * D];
    __shared__ int tokl[256];
    const int G = p.Nq / p.Nkv, groups = (G + kGroupHeads - 1) / kGroupHeads, tiles = (p.M * p.H + 127) / 128;
    const int y = blockIdx.x / p.chunks, i = (int)blockIdx.x - p.chunks * groups * p.Nkv;
    if (i < 0) last_logits_dq<T, D>(p, blockIdx.x - y * p.chunks, y / groups, y % groups * kGroupHeads, rows, tokl);
    else last_logits_dk<T, D>(p, i % tiles, i / tiles, rows, tokl);
}

template <typename T, int D>
__global__ __launch_bounds__(256) void br_last_logits_bwd_dq_sum_kernel(BrLogitsBwdParams p) {
    const BrPlanView pv = br_plan_view(p.plan, p.B, p.M, p.H, p.T);
    const long long per = (long long)p.B * p.Nq * p.R * D, i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= per) return;
    const int d = (int)(i % D), r = (int)(i / D % p.R), bn = (int)(i / D / p.R);
    put_dq<T>(p, pv, bn / p.Nq, bn % p.Nq, r, d, [&](int r2) {
        const float* src = p.part + ((long long)bn * p.R + r2) * D + d;
        float v = 0.f;
        for (int c = 0; c < p.chunks; c += 8) {                  // eight loads in flight
            float t[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) t[e] = c + e < p.chunks ? src[(c + e) * per] : 0.f;
#pragma unroll
            for (int e = 0; e < 8; ++e) v += t[e];
        }
        return v;
    });
}

template <typename T, int D>
void launch_bwd(const BrLogitsBwdParams& p, hipStream_t stream) {
    const int S = p.M * p.H, G = p.Nq / p.Nkv, groups = (G + kGroupHeads - 1) / kGroupHeads;
    hipLaunchKernelGGL((br_last_logits_bwd_kernel<T, D>), dim3(((S + 127) / 128 + p.chunks * groups) * p.Nkv, 1, p.B), dim3(256), 0, stream, p);
    if (p.chunks > 1) {
        const long long per = (long long)p.B * p.Nq * p.R * D;
        hipLaunchKernelGGL((br_last_logits_bwd_dq_sum_kernel<T, D>), dim3((unsigned)((per + 255) / 256)), dim3(256), 0, stream, p);
    }
}

}  // namespace

// Chunks the key slots are cut into for dq: enough workgroups for two on every CU, at least 256 slots each.
int br_last_logits_bwd_chunks(int B, int Nq, int Nkv, int M, int H, int n_cu) {
    const int G = Nq / Nkv, per = Nkv * ((G + kGroupHeads - 1) / kGroupHeads) * B, most = (int)(((long long)M * H + 255) / 256);
    const int want = (2 * n_cu + per - 1) / per;
    return want < 1 ? 1 : (want < most ? want : most);
}

void br_launch_last_logits(const void* q, const void* k, const int* plan, const int* rows, float* logits, const long long* sq,
                           const long long* sk, int B, int Nq, int Nkv, int M, int H, int D, int R, int T, float scale,
                           float neg, int dtype, hipStream_t stream) {
    BrLogitsParams p;
    p.q = q; p.k = k; p.plan = plan; p.rows = rows; p.logits = logits;
    p.sq_b = sq[0]; p.sq_h = sq[1]; p.sq_t = sq[2];
    p.sk_b = sk[0]; p.sk_h = sk[1]; p.sk_t = sk[2];
    p.B = B; p.Nq = Nq; p.Nkv = Nkv; p.M = M; p.H = H; p.R = R; p.T = T; p.scale = scale; p.neg = neg;
    const dim3 grid((M * H + 127) / 128, Nkv, B);
    if (dtype == 0 && D == 64) hipLaunchKernelGGL((br_last_logits_kernel<float, 64>), grid, dim3(256), 0, stream, p);
    else if (dtype == 0) hipLaunchKernelGGL((br_last_logits_kernel<float, 128>), grid, dim3(256), 0, stream, p);
    else if (dtype == 1 && D == 64) hipLaunchKernelGGL((br_last_logits_kernel<__bf16, 64>), grid, dim3(256), 0, stream, p);
    else if (dtype == 1) hipLaunchKernelGGL((br_last_logits_kernel<__bf16, 128>), grid, dim3(256), 0, stream, p);
    else if (D == 64) hipLaunchKernelGGL((br_last_logits_kernel<_Float16, 64>), grid, dim3(256), 0, stream, p);
    else hipLaunchKernelGGL((br_last_logits_kernel<_Float16, 128>), grid, dim3(256), 0, stream, p);
}

// part: room for br_last_logits_bwd_chunks() * B * Nq * R * D floats, or null (the slots are then not cut).
void br_launch_last_logits_bwd(const float* ds, const void* q, const void* k, const int* plan, const int* rows, void* dq, void* dk, float* part,
                               const long long* sq, const long long* sk, const long long* sdq, const long long* sdk, int B, int Nq,
                               int Nkv, int M, int H, int D, int R, int T, float scale, int add, int n_cu, int dtype, hipStream_t stream) {
    BrLogitsBwdParams p;
    p.ds = ds; p.q = q; p.k = k; p.plan = plan; p.rows = rows; p.dq = dq; p.dk = dk; p.part = part;
    p.sq_b = sq[0]; p.sq_h = sq[1]; p.sq_t = sq[2];
    p.sk_b = sk[0]; p.sk_h = sk[1]; p.sk_t = sk[2];
    p.dq_b = sdq[0]; p.dq_h = sdq[1]; p.dq_t = sdq[2];
    p.dk_b = sdk[0]; p.dk_h = sdk[1]; p.dk_t = sdk[2];
    p.B = B; p.Nq = Nq; p.Nkv = Nkv; p.M = M; p.H = H; p.R = R; p.T = T; p.scale = scale; p.add = add;
    const int S = M * H;
    p.chunks = part ? br_last_logits_bwd_chunks(B, Nq, Nkv, M, H, n_cu) : 1;
    p.chunk_slots = ((S + 255) / 256 + p.chunks - 1) / p.chunks * 256;
    const int n = D / 32, es = dtype == 0 ? 4 : 2;
    p.vec = reinterpret_cast<uintptr_t>(dk) % (n * es) == 0 && sdk[0] % n == 0 && sdk[1] % n == 0 && sdk[2] % n == 0;
    if (dtype == 0 && D == 64) launch_bwd<float, 64>(p, stream);
    else if (dtype == 0) launch_bwd<float, 128>(p, stream);
    else if (dtype == 1 && D == 64) launch_bwd<__bf16, 64>(p, stream);
    else if (dtype == 1) launch_bwd<__bf16, 128>(p, stream);
    else if (D == 64) launch_bwd<_Float16, 64>(p, stream);
    else launch_bwd<_Float16, 128>(p, stream);
}
