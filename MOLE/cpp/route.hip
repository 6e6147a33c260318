// Routing: top-k with lowest-index ties, gate values, per-expert counts, k-major locations,
// capacity and the dispatch permutation.  Deterministic: no atomics, every sum has a fixed order.
//
// Replaces tutel's extract_critical (called at MOLE/moe/layer.py:445-446) and the softmax half of
// MOLETopk.forward (MOLE/utils/Ugate.py:13).
//
// Up to four launches, all on the caller's stream:
//   route_tokens    64 tokens per block of 16 waves, or 16 or 4 of four waves.  A group of 16 lanes (64 beyond 256 experts, and beyond
//                   64 where the tokens are few) owns one token and holds
//                   its scores in registers - softmaxed on the spot when it is given logits; k rounds of a lane-pattern
//                   arg-max with the (score desc, index asc) order.
//   then, up to 8192 pairs,
//   route_rank      one block: locations, counts, capacity, kept rows, row offsets, l_aux from the chosen experts alone;
//   otherwise route_tokens goes on: wave j ranks choice j, a token's rank being the
//                   number of the block's earlier tokens with the same expert, from one ballot per bit of the index; and
//   route_scan      one wave per (choice, expert): exclusive prefix over the blocks' histograms.
//   route_finish    one block: per-expert totals, capacity, kept rows, row offsets, l_aux; for small problems also the scan
//                   and the last stage.
//   route_finalize  loc = base(choice, expert) + block prefix + in-block rank; row = offset + loc.
// A single block of tokens does all of it itself.
#include "common.h"

#include <algorithm>
#include <limits.h>
#include <math.h>

#include <mutex>
#include <stdlib.h>

namespace mole {

constexpr int RT_THREADS = 256;
constexpr int RT_TOKENS = 64;   // tokens per block of route_tokens; a choice is ranked by one wave over all 64
constexpr float FP32_EPS = 1.1920928955078125e-07f;

// A load that is always issued (the caller clamps the address to something valid) and gives +0 where the value
// must not count.  Written as "ok ? p[i] : 0" the load sits under a branch, and the compiler then waits for every
// load in flight at each such branch: a batch of loads meant to overlap runs one after the other.
__device__ __forceinline__ float load_or_zero(const float *p, bool ok) {
    return __uint_as_float(__float_as_uint(*p) & (ok ? 0xffffffffu : 0u));
}
__device__ __forceinline__ int load_or_zero(const int *p, bool ok) { return *p & (ok ? -1 : 0); }

// torch.topk's order of scores as an unsigned key: NaN ranks above everything and NaNs are equal among
// themselves, then +inf .. -inf with -0 == +0.  Every key of a real score is above 0, which stands for "not
// available" (outside the gate, or already chosen).  Equal keys are ranked by expert index, lowest first.
__device__ __forceinline__ uint32_t topk_key(float v) {
    uint32_t u = __float_as_uint(v);
    if (v != v) return 0xffffffffu;
    if (u == 0x80000000u) u = 0u;
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float topk_unkey(uint32_t key) {
    return __uint_as_float((key & 0x80000000u) ? (key ^ 0x80000000u) : ~key);
}

// max / min over aligned groups of 2^logG lanes, result in every lane of the group.  Within a row of 16 lanes the
// exchange is a DPP lane pattern (no LDS, no index registers): neighbours, pairs, then the mirrored half row and
// the mirrored row, each of which pairs a lane with one from the other already-reduced half.  32-lane groups add
// one crossbar swizzle, the whole wave reads the four row results into scalars.
template <int CTRL> __device__ __forceinline__ int dpp_lane(int x) {
    return __builtin_amdgcn_update_dpp(x, x, CTRL, 0xf, 0xf, false);
}
// the value of lane l ^ M, M = 1, 2, 4 or 8 (xor 4: the mirrored half row, then the reversed quads)
template <int M> __device__ __forceinline__ float lane_xor(float x) {
    const int v = __builtin_bit_cast(int, x);
    if constexpr (M == 1) return __builtin_bit_cast(float, dpp_lane<0xb1>(v));
    else if constexpr (M == 2) return __builtin_bit_cast(float, dpp_lane<0x4e>(v));
    else if constexpr (M == 4) return __builtin_bit_cast(float, dpp_lane<0x1b>(dpp_lane<0x141>(v)));
    else return __builtin_bit_cast(float, dpp_lane<0x128>(v));       // row_ror 8
}
// sum over aligned groups of 16 lanes in the order of a butterfly from 8 down, as __shfl_xor would add it
__device__ __forceinline__ float butterfly16(float x) {
    x += lane_xor<8>(x);
    x += lane_xor<4>(x);
    x += lane_xor<2>(x);
    return x + lane_xor<1>(x);
}
template <typename T, typename Op> __device__ __forceinline__ T group_reduce(T x, int logG, Op op) {
    static_assert(sizeof(T) == 4, "32-bit lanes");
    auto bits = [](T v) { return __builtin_bit_cast(int, v); };
    auto val = [](int v) { return __builtin_bit_cast(T, v); };
    if (logG >= 1) x = op(x, val(dpp_lane<0xb1>(bits(x))));      // quad_perm [1,0,3,2]
    if (logG >= 2) x = op(x, val(dpp_lane<0x4e>(bits(x))));      // quad_perm [2,3,0,1]
    if (logG >= 3) x = op(x, val(dpp_lane<0x141>(bits(x))));     // row_half_mirror
    if (logG >= 4) x = op(x, val(dpp_lane<0x140>(bits(x))));     // row_mirror
    if (logG == 5) x = op(x, val(__builtin_amdgcn_ds_swizzle(bits(x), 0x401f)));   // lane ^ 16 within 32 lanes
    if (logG >= 6) {
        const int xi = bits(x);
        x = op(op(val(__builtin_amdgcn_readlane(xi, 0)), val(__builtin_amdgcn_readlane(xi, 16))),
               op(val(__builtin_amdgcn_readlane(xi, 32)), val(__builtin_amdgcn_readlane(xi, 48))));
    }
    return x;
}

// Rank of the lane among the valid lanes below it that hold the same expert, and how many valid lanes hold it: one ballot
// per bit of the expert index.  (A loop over the distinct experts present is a serial chain of up to 64 ballots and
// lane reads.)
__device__ __forceinline__ int rank_in_wave(int e, bool valid, int E, int &same) {
    uint64_t m = __ballot(valid);
    for (int b = 0; (1 << b) < E; ++b) {
        const bool bit = (e >> b) & 1;
        const uint64_t bal = __ballot(valid && bit);
        m &= bit ? bal : ~bal;
    }
    same = __popcll(m);
    return __popcll(m & ((1ull << (threadIdx.x & 63)) - 1ull));
}

// What a block does once the top-k of its BT tokens (BT <= 64) lies in LDS - s_idx / s_graw [k][BT]: expert and raw
// gate value of every choice, s_col [4][E]: the four waves' column sums of the block's scores: the block's column sums
// out, gate values and indices out, then each choice's in-block ranks and per-expert histogram.  Four waves.
__device__ __forceinline__ void topk_block_tail(int BT, int S, int E, int k, int normalize, const int *s_idx,
                                                const float *s_graw, int *s_hist, const float *s_col,
                                                int32_t *__restrict__ idx, int32_t *__restrict__ lrank,
                                                float *__restrict__ gates, int32_t *__restrict__ hist,
                                                float *__restrict__ colsum, int nb) {
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b = blockIdx.x, tok0 = b * BT;
    __syncthreads();
    for (int e = tid; e < E; e += RT_THREADS)
        colsum[(size_t)b * E + e] = ((s_col[e] + s_col[E + e]) + s_col[2 * E + e]) + s_col[3 * E + e];

    // ---- gate values and indices out (threads 0..BT-1 = the block's tokens) -------------
    const int token = tok0 + tid;
    const bool tv = tid < BT && token < S;
    if (tv) {
        float denom = 0.f;
        for (int j = 0; j < k; ++j) denom += s_graw[j * BT + tid];  // left to right, fp32
        const float den = denom < FP32_EPS ? FP32_EPS : denom;
        for (int j = 0; j < k; ++j) {
            float gv = s_graw[j * BT + tid];
            if (k > 1 && normalize) gv = gv / den;
            gates[(size_t)j * S + token] = gv;
            idx[(size_t)j * S + token] = s_idx[j * BT + tid];
        }
    }

    if (hist == nullptr) return;           // (route_rank takes them from the indices)
    // ---- in-block ranks per choice (lane = token; wave w takes choices w, w + 4, ...) ------
    // Each wave works on a histogram of its own, so the choices proceed side by side without block barriers.
    int *my_hist = s_hist + w * E;
    const int ctoken = tok0 + lane;
    const bool cv = lane < BT && ctoken < S;
    for (int j = w; j < k; j += RT_THREADS / WAVE) {
        for (int e = lane; e < E; e += WAVE) my_hist[e] = 0;
        const int e = cv ? s_idx[j * BT + lane] : -1;
        int same;
        const int rank = rank_in_wave(e, cv, E, same);
        if (cv && rank == 0) my_hist[e] = same;
        if (cv) lrank[(size_t)j * S + ctoken] = rank;
        // (the histogram is written and read by this wave only: program order is enough)
        for (int e2 = lane; e2 < E; e2 += WAVE) hist[((size_t)j * E + e2) * nb + b] = my_hist[e2];
    }
}

// one wave per (choice, expert) pair: exclusive prefix over blocks, total into counts
__device__ __forceinline__ void scan_pair(int32_t *__restrict__ hist, int nb, int pair, int32_t *__restrict__ counts) {
    const int lane = threadIdx.x & 63;
    int carry = 0;
    // four chunks of 64 blocks at a time: their loads are in flight together
    for (int c0 = 0; c0 < nb; c0 += 4 * WAVE) {
        int v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int bi = c0 + u * WAVE + lane;
            v[u] = load_or_zero(hist + (size_t)pair * nb + min(bi, nb - 1), bi < nb);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const int bi = c0 + u * WAVE + lane;
            const int x = wave_scan(v[u]);
            if (bi < nb) hist[(size_t)pair * nb + bi] = carry + x - v[u];
            carry += wave_total(x);
        }
    }
    if (lane == 0) counts[pair] = carry;
}
// Blocks past the scan's own fold the per-block column sums of the scores (for l_aux) into COLSUM_SLICES rows:
// slice s adds blocks s, s + COLSUM_SLICES, ... in that order, so the single block that finishes the routing
// reads COLSUM_SLICES rows instead of one per 64 tokens (at 32768 tokens and 256 experts that loop was 40 us).
constexpr int COLSUM_SLICES = 16;
__global__ __launch_bounds__(256) void route_scan_kernel(int32_t *__restrict__ hist, int nb, int npairs,
                                                         int32_t *__restrict__ counts, int scan_blocks,
                                                         const float *__restrict__ colsum, int E,
                                                         float *__restrict__ colpart) {
    if ((int)blockIdx.x < scan_blocks) {
        const int pair = blockIdx.x * 4 + (threadIdx.x >> 6);
        if (pair < npairs) scan_pair(hist, nb, pair, counts);
        return;
    }
    const int cb = blockIdx.x - scan_blocks;
    const int slice = cb % COLSUM_SLICES, e = (cb / COLSUM_SLICES) * 256 + threadIdx.x;
    if (e >= E) return;
    float me = 0.f;
    for (int b0 = slice; b0 < nb; b0 += 8 * COLSUM_SLICES) {        // 8 loads in flight, added in block order
        float t[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int b = b0 + u * COLSUM_SLICES;
            t[u] = load_or_zero(colsum + (size_t)min(b, nb - 1) * E + e, b < nb);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (b0 + u * COLSUM_SLICES < nb) me += t[u];
    }
    colpart[slice * E + e] = me;
}

constexpr int FIN_THREADS = 1024;

// What the end of the routing needs and produces.
struct RouteEnd {
    int S, E, k, cf_sign, cap_bound, alignment, layout;
    int32_t *counts, *kept_rows, *offsets, *capacity;
    float *l_aux;
    int32_t *idx, *loc, *row;          // loc: in-block ranks in, locations out
    int32_t *token_of;                 // token of every row that is kept (null: nobody asks)
    // location l of pair p (token i) of an expert whose rows start at off
    __device__ __forceinline__ void place(size_t p, int i, int l, int cap, int off) const {
        const int at = l < cap ? off + l : -1;
        loc[p] = l;
        row[p] = at;
        if (token_of != nullptr && at >= 0) token_of[at] = i;
    }
};

// Loads of the experts (s_off [E]) -> capacity, kept rows, offsets (s_off again), l_aux (s_me [E]: column sum of the scores x count of the
// first choice).  Called by all threads of a block.  What runs over the experts - the largest load, the offsets, the loss's
// sum - is one wave's work, 64 experts at a time: by all waves of the block each of the three is a reduction between two or three
// barriers.
__device__ __forceinline__ void finish_offsets(const RouteEnd &r, const float *s_me, int *s_off, int *s_cap) {
    const int tid = threadIdx.x, E = r.E;
    if (tid < WAVE) {
        int cap = r.cap_bound;
        if (r.cf_sign <= 0) {              // uniform: the largest load, which only capacity factors <= 0 ask for
            int most = 0;
            for (int e = tid; e < E; e += WAVE) most = max(most, s_off[e]);
            cap = group_reduce(most, 6, [](int a, int c) { return max(a, c); });
            if (r.cf_sign < 0) cap = min(cap, r.cap_bound);
        }
        const int rem = cap % r.alignment;
        if (rem > 0) cap += r.alignment - rem;
        int before = 0;
        float loss = 0.f;
        for (int e0 = 0; e0 < E; e0 += WAVE) {
            const int e = e0 + tid, n = e < E ? min(s_off[e], cap) : 0;
            int off = e * cap;
            if (r.layout == MOLE_LAYOUT_RAGGED) {
                const int incl = wave_scan(n);
                off = before + incl - n;
                before += wave_total(incl);
            }
            if (r.l_aux != nullptr) loss += e < E ? s_me[e] : 0.f;
            if (e < E) {
                r.kept_rows[e] = n;
                r.offsets[e] = off;
                s_off[e] = off;
            }
        }
        if (r.l_aux != nullptr) loss = wave_sum(loss);
        if (tid == 0) {
            r.offsets[E] = r.layout == MOLE_LAYOUT_RAGGED ? before : E * cap;
            r.capacity[0] = cap;
            *s_cap = cap;
            if (r.l_aux != nullptr) r.l_aux[0] = r.S > 0 ? loss * ((float)E / ((float)r.S * (float)r.S)) : 0.f;
        }
    }
    __syncthreads();
}

// Counts -> capacity, kept rows, offsets, l_aux.  cnt: [k][E] totals (global or LDS), replaced by base(choice, expert), the rows of
// the expert's earlier choices; s_me [E]: the column sums of the scores (with l_aux).  Returns the capacity; s_off[e] = first row of
// expert e.
template <int THREADS>
__device__ __forceinline__ int finish_counts(const RouteEnd &r, int *cnt, float *s_me, int *s_off, int *s_cap) {
    const int tid = threadIdx.x, E = r.E;
    for (int e = tid; e < E; e += THREADS) {
        int tot = 0, first = 0;
        for (int j = 0; j < r.k; ++j) {
            const int c = cnt[j * E + e];
            if (j == 0) first = c;
            r.counts[j * E + e] = c;
            cnt[j * E + e] = tot;
            tot += c;
        }
        s_off[e] = tot;
        if (r.l_aux != nullptr) s_me[e] *= (float)first;
    }
    __syncthreads();
    finish_offsets(r, s_me, s_off, s_cap);
    return *s_cap;
}
// The column sums of the scores (with l_aux): thread (g, e) adds blocks g, g + groups, ... in order; later the groups in order.
__device__ __forceinline__ float column_part(const RouteEnd &r, const float *__restrict__ colsum, int nb_col) {
    float me = 0.f;
    const int E = r.E, groups = FIN_THREADS / E;
    if ((int)threadIdx.x < groups * E) {
        const int e = threadIdx.x % E, gq = threadIdx.x / E;
        for (int b0 = gq; b0 < nb_col; b0 += 8 * groups) {
            float t[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int b = b0 + u * groups;
                t[u] = load_or_zero(colsum + (size_t)min(b, nb_col - 1) * E + e, b < nb_col);
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (b0 + u * groups < nb_col) me += t[u];
        }
    }
    return me;
}
// s_part: the threads' parts; s_part[e], e < E, becomes the sum
__device__ __forceinline__ void fold_columns(const RouteEnd &r, float *s_part) {
    const int E = r.E, tid = threadIdx.x;
    if (r.l_aux == nullptr || tid >= E) return;
    float me = s_part[tid];
    for (int gq = 1; gq < FIN_THREADS / E; ++gq) me += s_part[gq * E + tid];
    s_part[tid] = me;
}

// One block.  scan_hist == NULL: counts holds the totals already (route_scan ran).  Otherwise the block scans the
// histograms itself: a thread per (choice, expert) where few blocks of tokens were counted (all its loads are in
// flight at once), a wave per pair otherwise.  last: it also writes locations and rows (small problems: a launch less).
// (256 experts, top-8, 256 tokens: 2048 pairs of four counts took a wave each and 197 us; by threads, last stage
// included, 15 us.)
constexpr int FIN_FEW = 32;            // blocks of tokens up to which a thread scans a pair on its own
__global__ __launch_bounds__(FIN_THREADS) void route_finish_kernel(const RouteEnd r, const float *__restrict__ colsum, int nb_col,
                                                                   int32_t *__restrict__ basej, int32_t *scan_hist, int nb, int bt,
                                                                   int last) {
    __shared__ int s_off[FIN_THREADS];
    __shared__ int s_cap;
    __shared__ float s_part[FIN_THREADS];
    const int tid = threadIdx.x, E = r.E, npairs = r.k * E;
    if (r.l_aux != nullptr) s_part[tid] = column_part(r, colsum, nb_col);
    if (scan_hist != nullptr) {
        if (nb <= FIN_FEW) {
            for (int pair = tid; pair < npairs; pair += FIN_THREADS) {
                int32_t *h = scan_hist + (size_t)pair * nb;
                int carry = 0;
                for (int b0 = 0; b0 < nb; b0 += 8) {
                    int v[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) v[u] = load_or_zero(h + min(b0 + u, nb - 1), b0 + u < nb);
#pragma unroll
                    for (int u = 0; u < 8; ++u)
                        if (b0 + u < nb) { h[b0 + u] = carry; carry += v[u]; }
                }
                basej[pair] = carry;
            }
        } else {
            for (int pair = tid >> 6; pair < npairs; pair += FIN_THREADS / 64) scan_pair(scan_hist, nb, pair, basej);
        }
    } else {
        for (int pair = tid; pair < npairs; pair += FIN_THREADS) basej[pair] = r.counts[pair];
    }
    __threadfence_block();
    __syncthreads();
    fold_columns(r, s_part);
    const int cap = finish_counts<FIN_THREADS>(r, basej, s_part, s_off, &s_cap);
    if (!last) return;
    __threadfence_block();
    for (int p = tid; p < r.k * r.S; p += FIN_THREADS) {
        const int j = p / r.S, i = p % r.S;
        const int e = r.idx[p];
        r.place(p, i, basej[j * E + e] + scan_hist[((size_t)j * E + e) * nb + i / bt] + r.loc[p], cap, s_off[e]);
    }
}

// The end of the routing from the chosen experts alone, in one block: no histograms through memory, no launch behind it.  The pairs
// lie in choice-major order, in chunks of 64 tokens of one choice; wave w ranks chunks w, w + 16, ... (P of them) and leaves their
// counts in LDS, an exclusive prefix over the chunks of every expert is then a pair's location but for its rank.  Bound by latency:
// one round trip for the indices, the rest is LDS.  Histograms through memory and what goes with them / here: 256 experts, top-8, 256 tokens
// 17.8 / 13.4 us; 8 experts, top-2, 777 tokens 7.6 / 5.8, 4096 tokens 12.9 / 10.4 (two launches / one); 16 experts, top-2, 2048 tokens 9.5 /
// 7.4, 3001 tokens 13.7 / 11.8.  A thread's eight pairs are as long as the launch they save: the line lies there.
constexpr int RANK_PAIRS = 8192, RANK_COUNTS = 16384;       // most pairs (P = 8) and counts (64 KB of LDS)
static bool rank_in_one_block(int S, int E, int k) {
    const long chunks = (long)k * ceil_div(S, WAVE);
    return chunks <= RANK_PAIRS / WAVE && chunks * (E | 1) <= RANK_COUNTS;
}
template <int P>
__global__ __launch_bounds__(FIN_THREADS) void route_rank_kernel(const RouteEnd r, const float *__restrict__ colsum, int nb_col) {
    constexpr int WAVES = FIN_THREADS / WAVE;
    extern __shared__ __align__(16) int s_cnt[];            // [chunks][stride]
    __shared__ int s_off[FIN_THREADS];
    __shared__ float s_part[FIN_THREADS];
    __shared__ int s_cap;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, E = r.E, S = r.S, k = r.k;
    const int per = (S + WAVE - 1) / WAVE, chunks = k * per, stride = E | 1;       // (odd: the scan walks down a column)
    int e[P], at[P];
    bool ok[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int c = p * WAVES + w, j = c / per, i = (c - j * per) * WAVE + lane;
        ok[p] = c < chunks && i < S;
        at[p] = min(j, k - 1) * S + min(i, S - 1);
        e[p] = load_or_zero(r.idx + at[p], ok[p]);
    }
    if (r.l_aux != nullptr) s_part[tid] = column_part(r, colsum, nb_col);
    for (int q = tid; q < chunks * stride; q += FIN_THREADS) s_cnt[q] = 0;
    __syncthreads();
    fold_columns(r, s_part);
    int rank[P];
#pragma unroll
    for (int p = 0; p < P; ++p) {
        int same;
        rank[p] = rank_in_wave(e[p], ok[p], E, same);
        if (ok[p] && rank[p] == 0) s_cnt[(p * WAVES + w) * stride + e[p]] = same;
    }
    __syncthreads();
    // exclusive prefix over the chunks, a wave per expert, four at a time
    for (int e0 = w; e0 < E; e0 += 4 * WAVES) {
        int run[4] = {0, 0, 0, 0};
        for (int c0 = 0; c0 < chunks; c0 += WAVE) {
            const int c = c0 + lane;
            int n[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) n[u] = load_or_zero(s_cnt + min(c, chunks - 1) * stride + min(e0 + u * WAVES, E - 1), c < chunks);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int incl = wave_scan(n[u]);
                if (c < chunks && e0 + u * WAVES < E) s_cnt[c * stride + e0 + u * WAVES] = run[u] + incl - n[u];
                run[u] += wave_total(incl);
            }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (lane == 0 && e0 + u * WAVES < E) s_off[e0 + u * WAVES] = run[u];         // all rows of the expert
    }
    __syncthreads();
    for (int q = tid; q < k * E; q += FIN_THREADS) {         // counts of a choice: where the next one starts less where it does
        const int j = q / E, ee = q - j * E;
        const int n = (j + 1 < k ? s_cnt[(j + 1) * per * stride + ee] : s_off[ee]) - s_cnt[j * per * stride + ee];
        r.counts[q] = n;
        if (j == 0 && r.l_aux != nullptr) s_part[ee] *= (float)n;
    }
    __syncthreads();
    finish_offsets(r, s_part, s_off, &s_cap);
    const int cap = s_cap;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (!ok[p]) continue;
        const int c = p * WAVES + w;
        r.place(at[p], c % per * WAVE + lane, s_cnt[c * stride + e[p]] + rank[p], cap, s_off[e[p]]);
    }
}

__global__ __launch_bounds__(256) void route_finalize_kernel(const RouteEnd r, const int32_t *__restrict__ hist, const int32_t *__restrict__ basej,
                                                             int nb, int bt /* tokens per histogram block */) {
    const size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (size_t)r.k * r.S) return;
    const int j = (int)(p / r.S), i = (int)(p % r.S);
    const int e = r.idx[p];
    const int b = i / bt;
    r.place(p, i, basej[j * r.E + e] + hist[((size_t)j * r.E + e) * nb + b] + r.loc[p], r.capacity[0], r.offsets[e]);
}

// ---- the tokens' own part ------------------------------------------------------------------------------------------
// A block of THREADS takes TOK tokens.  2^LOGG lanes own a token and hold VPL scores each (lane g: experts g, g + G, ...); with 16 lanes per token
// all the block's tokens go through their rounds at once, with a wave per token THREADS / 64 of them.  64 tokens
// a block where there are many (four waves on 64 tokens, 16 tokens a wave, four at a time, spent four times the latency of a round: 256 experts,
// top-8: 42 us for 256 tokens and 58 for 32768, now 21 and 45).  Few tokens leave the other CUs idle that way, while the rounds of a block's 16
// waves share the four SIMDs of one: they take blocks of four waves and 16 tokens, or, beyond 64 experts, of four tokens with a wave each (256
// experts, top-8, 256 tokens: 21 -> 7.8 us).
// logits != 0: `in` holds logits (without bias if one is given) and the block starts with the softmax (the sums in the order of gate_fwd_kernel's), writing
// scores; LOGITS_PARTS / LOGITS_PAIRS: `in` holds four partial sums of them, [4][S][E], to be added one after the other / in pairs.
// nb == 1: the block has seen all tokens and goes on to the end of the routing by itself.  hist null: route_rank takes it
// from the indices.
enum { LOGITS_NONE, LOGITS_WHOLE, LOGITS_PARTS, LOGITS_PAIRS };
// PARTS: partial sums may come (up to 64 tokens).  Their registers are not for the blocks of 64 tokens beyond 64 experts: three parts beside 16
// values a lane, and 54 registers instead of 18 are spilled (routing of 512 tokens, 300 experts top-8, with / without, 80.6 / 75.1 us; 16384, 512
// top-8, 91.2 / 78.9; that pass 274 / 261).
template <int VPL, int LOGG, int THREADS, int TOK, bool PARTS>
__global__ __launch_bounds__(THREADS) void route_tokens_kernel(const float *__restrict__ in, const float *__restrict__ bias,
                                                                   int logits, int normalize,
                                                                   float *__restrict__ scores, float *__restrict__ gates,
                                                                   int32_t *__restrict__ hist /* [k][E][nb] */,
                                                                   float *__restrict__ colsum /* [nb][E] */, int nb, const RouteEnd r) {
    constexpr int G = 1 << LOGG, TPP = THREADS >> LOGG, PASSES = TOK / TPP;
    constexpr int WAVES = THREADS / WAVE, PER_WAVE = (MOLE_MAX_TOPK + WAVES - 1) / WAVES;
    constexpr int ROWS = THREADS == 256 ? WAVE / G : 1;      // a small block keeps its waves' token groups' column sums apart
    extern __shared__ __align__(16) char smem[];
    const int S = r.S, E = r.E, k = r.k;
    int *s_idx = (int *)smem;                          // [k][TOK]
    float *s_graw = (float *)(s_idx + k * TOK);        // [k][TOK]
    float *s_col = (float *)(s_graw + k * TOK);        // [WAVES ROWS][E]
    int *s_hist = (int *)(s_col + WAVES * ROWS * E);          // [k][E], with hist or nb == 1
    int *s_off = s_hist + k * E;                       // [E], nb == 1
    __shared__ int s_cap;

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int b = blockIdx.x, tok0 = b * TOK;
    const int g = lane & (G - 1);
    const bool count = nb == 1 || hist != nullptr;
    if (count)
        for (int i = tid; i < k * E; i += THREADS) s_hist[i] = 0;
    float colacc[VPL];
#pragma unroll
    for (int q = 0; q < VPL; ++q) colacc[q] = 0.f;
    for (int pass = 0; pass < PASSES; ++pass) {
        const int tl = pass * TPP + (tid >> LOGG);
        const int token = tok0 + tl;
        const bool tv = tl < TOK && token < S;
        float v[VPL];
#pragma unroll
        for (int q = 0; q < VPL; ++q) v[q] = 0.f;
        if (S > 0) {
#pragma unroll
            for (int q = 0; q < VPL; ++q) v[q] = in[(size_t)min(token, S - 1) * E + min(g + (q << LOGG), E - 1)];
            if (PARTS && logits >= LOGITS_PARTS) {
                float t[3][VPL];
#pragma unroll
                for (int u = 0; u < 3; ++u)
#pragma unroll
                    for (int q = 0; q < VPL; ++q) t[u][q] = in[((size_t)(u + 1) * S + min(token, S - 1)) * E + min(g + (q << LOGG), E - 1)];
#pragma unroll
                for (int q = 0; q < VPL; ++q) v[q] = logits == LOGITS_PARTS ? v[q] + t[0][q] + t[1][q] + t[2][q] : (v[q] + t[0][q]) + (t[1][q] + t[2][q]);
            }
        }
        if (logits) {
            float mx = -INFINITY;
#pragma unroll
            for (int q = 0; q < VPL; ++q) {
                if (bias) v[q] += bias[min(g + (q << LOGG), E - 1)];
                v[q] = g + (q << LOGG) < E ? v[q] : -INFINITY;
                mx = fmaxf(mx, v[q]);
            }
            mx = group_reduce(mx, LOGG, [](float a, float c) { return fmaxf(a, c); });
            float sum = 0.f;
#pragma unroll
            for (int q = 0; q < VPL; ++q) v[q] = g + (q << LOGG) < E ? expf(v[q] - mx) : 0.f;
            // the sums of the kernels that do the softmax alone, term for term: up to 64 experts gate_fwd_kernel's, beyond
            // softmax_fwd_kernel's, whose wave holds experts l, l + 64, .. in lane l (four of them are lane g's here)
            if constexpr (LOGG == 4 && VPL > 4) {
                float part[4];
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    part[c] = 0.f;
#pragma unroll
                    for (int q = c; q < VPL; q += 4) part[c] += v[q];
                    part[c] = group_reduce(part[c], 4, [](float a, float d) { return a + d; });
                }
                sum = (part[0] + part[1]) + (part[2] + part[3]);
            } else {
#pragma unroll
                for (int q = 0; q < VPL; ++q) sum += v[q];
                if constexpr (LOGG == 4) {
                    sum = butterfly16(sum);
                } else {
                    sum = group_reduce(sum, LOGG, [](float a, float d) { return a + d; });
                }
            }
#pragma unroll
            for (int q = 0; q < VPL; ++q) {
                const int e = g + (q << LOGG);
                v[q] = v[q] / sum;
                if (tv && e < E) scores[(size_t)token * E + e] = v[q];
            }
        }
        uint32_t key[VPL];
#pragma unroll
        for (int q = 0; q < VPL; ++q) {
            const bool ok = tv && g + (q << LOGG) < E;
            const float sv = __uint_as_float(__float_as_uint(v[q]) & (ok ? 0xffffffffu : 0u));
            colacc[q] += sv;
            key[q] = ok ? topk_key(sv) : 0u;
        }
        for (int j = 0; j < k; ++j) {
            // the best score of the token, then the lowest expert index among those that hold it
            uint32_t best = key[0];
#pragma unroll
            for (int q = 1; q < VPL; ++q) best = max(best, key[q]);
            const uint32_t top = group_reduce(best, LOGG, [](uint32_t a, uint32_t c) { return max(a, c); });
            int cand = INT_MAX;
#pragma unroll
            for (int q = VPL - 1; q >= 0; --q)
                if (key[q] == top) cand = g + (q << LOGG);             // ends on the lane's lowest such expert
            if (top == 0u) cand = INT_MAX;                             // nothing available (a token past the end)
            const int bi = group_reduce(cand, LOGG, [](int a, int c) { return min(a, c); });
            const bool mine = bi != INT_MAX && (bi & (G - 1)) == g;
#pragma unroll
            for (int q = 0; q < VPL; ++q)
                if (mine && (bi >> LOGG) == q) key[q] = 0u;
            if (g == 0 && tv) {
                s_idx[j * TOK + tl] = bi;
                s_graw[j * TOK + tl] = topk_unkey(top);
            }
        }
    }
    // column sums of the scores (for l_aux): the tokens of a wave, then (below) the waves in order
#pragma unroll
    for (int q = 0; q < VPL; ++q) {
        float c = colacc[q];
        if constexpr (ROWS == 1)
            for (int m = G; m < WAVE; m <<= 1) c += __shfl_xor(c, m, WAVE);
        const int e = g + (q << LOGG);
        if ((ROWS > 1 || lane < G) && e < E) s_col[(w * ROWS + (ROWS > 1 ? lane >> LOGG : 0)) * E + e] = c;
    }
    __syncthreads();
    for (int e = tid; e < E; e += THREADS) {
        float me = 0.f;
#pragma unroll
        for (int q = 0; q < WAVES * ROWS; ++q) me += s_col[q * E + e];
        if (nb > 1) colsum[(size_t)b * E + e] = me;
        else s_col[e] = me;
    }
    // gate values and indices out: thread t < TOK is token t
    if (tid < TOK && tok0 + tid < S) {
        float denom = 0.f;
        for (int j = 0; j < k; ++j) denom += s_graw[j * TOK + tid];  // left to right, fp32
        const float den = denom < FP32_EPS ? FP32_EPS : denom;
        for (int j = 0; j < k; ++j) {
            float gv = s_graw[j * TOK + tid];
            if (k > 1 && normalize) gv = gv / den;
            gates[(size_t)j * S + tok0 + tid] = gv;
            r.idx[(size_t)j * S + tok0 + tid] = s_idx[j * TOK + tid];
        }
    }
    if (!count) return;
    // in-block ranks: wave w ranks choices w, w + WAVES, ..., lane = token
    const int token = tok0 + lane;
    int my_e[PER_WAVE], rank[PER_WAVE];
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int j = q * WAVES + w;
        if (j >= k) break;
        const bool cv = lane < TOK && token < S;
        my_e[q] = cv ? s_idx[j * TOK + lane] : 0;
        int same;
        rank[q] = rank_in_wave(my_e[q], cv, E, same);
        if (cv && rank[q] == 0) s_hist[j * E + my_e[q]] = same;
        if (nb > 1) {
            if (cv) r.loc[(size_t)j * S + token] = rank[q];
            // written and read by this wave: program order is enough
            for (int e = lane; e < E; e += WAVE) hist[((size_t)j * E + e) * nb + b] = s_hist[j * E + e];
        }
    }
    if (nb > 1) return;
    __syncthreads();
    const int cap = finish_counts<THREADS>(r, s_hist, s_col, s_off, &s_cap);
#pragma unroll
    for (int q = 0; q < PER_WAVE; ++q) {
        const int j = q * WAVES + w;
        if (j >= k || lane >= TOK || token >= S) break;
        r.place((size_t)j * S + token, token, s_hist[j * E + my_e[q]] + rank[q], cap, s_off[my_e[q]]);
    }
}

static size_t align256(size_t v) { return (v + 255) & ~(size_t)255; }

}  // namespace mole

using namespace mole;

// Up to FEW_TOKENS tokens in small blocks: 16 tokens of up to 64 experts, 16 lanes each, or 4 tokens, a wave each.
constexpr int FEW_TOKENS = 512;
static int few_block(int E) { return E <= 64 ? 16 : 4; }

// Scratch of the routing by histograms, with which mole_route does any call, and the column sums of small blocks, which are more where the blocks are
// many and the choices few: mole_route takes small blocks where the workspace holds them.
static size_t route_hist_bytes(int S, int E, int k) {
    const size_t nb = (size_t)ceil_div(S > 0 ? S : 1, RT_TOKENS);
    return align256(nb * k * E * sizeof(int32_t)) + align256((size_t)k * E * sizeof(int32_t)) +
           align256(nb * E * sizeof(float)) + align256((size_t)COLSUM_SLICES * E * sizeof(float));
}
static size_t few_bytes(int S, int E) { return S <= FEW_TOKENS ? align256((size_t)ceil_div(S, few_block(E)) * E * sizeof(float)) : 0; }
extern "C" size_t mole_route_workspace_bytes(int S, int E, int k) {
    if (S < 0 || E <= 0 || k <= 0) return 0;
    return std::max(route_hist_bytes(S, E, k), few_bytes(S, E));
}

// The stages of the routing behind the tokens' own: scan of the histograms over blocks, counts / capacity / offsets /
// l_aux, then locations and destination rows.  nb blocks of bt tokens each were counted.
static int route_after_topk(const RouteEnd &r, int32_t *hist, int32_t *basej, float *colsum, float *colpart, int nb, int bt,
                            hipStream_t st) {
    const int npairs = r.k * r.E;
    // small enough for the finishing block (saves a launch): a thread per pair up to FIN_FEW blocks of tokens and 2^16
    // counts, a wave per pair up to 2^13 counts
    const bool scan_in_finish = (long long)npairs * nb <= (nb <= FIN_FEW ? 65536 : 8192);
    const bool last_in_finish = scan_in_finish && (long long)r.k * r.S <= 4 * FIN_THREADS;
    if (!scan_in_finish) {
        const int scan_blocks = ceil_div(npairs, 4);
        hipLaunchKernelGGL(route_scan_kernel, dim3(scan_blocks + COLSUM_SLICES * ceil_div(r.E, 256)), dim3(256), 0, st, hist,
                           nb, npairs, r.counts, scan_blocks, colsum, r.E, colpart);
        MOLE_LAUNCH_CHECK();
    }
    // (when the scan kernel ran, it also folded the column sums: the finish then adds its COLSUM_SLICES rows)
    hipLaunchKernelGGL(route_finish_kernel, dim3(1), dim3(FIN_THREADS), 0, st, r, scan_in_finish ? colsum : colpart,
                       scan_in_finish ? nb : min(nb, COLSUM_SLICES), basej, scan_in_finish ? hist : (int32_t *)nullptr, nb, bt,
                       (int)last_in_finish);
    MOLE_LAUNCH_CHECK();
    if (r.S > 0 && !last_in_finish) {
        const size_t n = (size_t)r.k * r.S;
        hipLaunchKernelGGL(route_finalize_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, r, hist, basej, nb, bt);
        MOLE_LAUNCH_CHECK();
    }
    return 0;
}

static RouteEnd route_end(int S, int E, int k, double capacity_factor, int alignment, int layout, int32_t *idx, int32_t *loc,
                          int32_t *row, int32_t *counts, int32_t *kept_rows, int32_t *offsets, int32_t *capacity, float *l_aux,
                          int32_t *token_of = nullptr) {
    const int spe = (S + E - 1) / E;
    const int cf_sign = capacity_factor > 0. ? 1 : (capacity_factor < 0. ? -1 : 0);
    // int(cf * spe) of the Python reference: the product is taken in double precision
    const double prod = (capacity_factor < 0. ? -capacity_factor : capacity_factor) * (double)spe;
    // (held to what leaves room for the alignment in 32 bits: a factor that overflowed them made the capacity negative)
    const int limit = (INT_MAX - alignment) / k;
    return RouteEnd{S, E, k, cf_sign, k * (prod < (double)limit ? (int)prod : limit), alignment, layout, counts, kept_rows, offsets, capacity, l_aux, idx, loc, row, token_of};
}

template <int VPL, int LOGG, int THREADS, int TOK, bool PARTS>
static int launch_tokens_as(const float *in, const float *bias, int logits, int normalize, float *scores, float *gates, int32_t *hist, float *colsum,
                            int nb, const RouteEnd &r, hipStream_t st) {
    constexpr int COLS = THREADS / WAVE * (THREADS == 256 ? WAVE >> LOGG : 1);
    const size_t lds = (size_t)r.k * TOK * 8 + (size_t)COLS * r.E * 4 + (nb == 1 || hist != nullptr ? (size_t)(r.k + 1) * r.E * 4 : 0);
    auto kern = route_tokens_kernel<VPL, LOGG, THREADS, TOK, PARTS>;
    MOLE_REQUIRE(PARTS || logits < LOGITS_PARTS, "routing: partial logits for a kernel that takes whole ones (S=%d E=%d k=%d)", r.S, r.E, r.k);
    if (lds > 48 * 1024)               // hundreds of experts and a long top-k: beyond the default limit together with the static part
        MOLE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(kern, dim3(nb), dim3(THREADS), lds, st, in, bias, logits, normalize, scores, gates, hist, colsum, nb, r);
    MOLE_LAUNCH_CHECK();
    return 0;
}
// few: at most FEW_TOKENS tokens, in blocks of few_block(E)
static int launch_tokens(bool few, const float *in, const float *bias, int logits, int normalize, float *scores, float *gates, int32_t *hist, float *colsum,
                         int nb, const RouteEnd &r, hipStream_t st) {
#define MOLE_LT(VPL, LOGG, THREADS, TOK, PARTS) launch_tokens_as<VPL, LOGG, THREADS, TOK, PARTS>(in, bias, logits, normalize, scores, gates, hist, colsum, nb, r, st)
    const int E = r.E;
    if (few) {
        if (E <= 16) return MOLE_LT(1, 4, 256, 16, true);
        if (E <= 32) return MOLE_LT(2, 4, 256, 16, true);
        if (E <= 64) return MOLE_LT(4, 4, 256, 16, true);
        if (E <= 128) return MOLE_LT(2, 6, 256, 4, true);
        if (E <= 256) return MOLE_LT(4, 6, 256, 4, true);
        return MOLE_LT(16, 6, 256, 4, true);
    }
    // 16 lanes per token; beyond 256 experts a lane would hold more than 16 values, so the whole wave takes a token
    if (E <= 16) return MOLE_LT(1, 4, 1024, 64, true);
    if (E <= 32) return MOLE_LT(2, 4, 1024, 64, true);
    if (E <= 64) return MOLE_LT(4, 4, 1024, 64, true);
    if (E <= 128) return MOLE_LT(8, 4, 1024, 64, false);
    if (E <= 256) return MOLE_LT(16, 4, 1024, 64, false);
    return MOLE_LT(16, 6, 1024, 64, false);
#undef MOLE_LT
}
template <int P> static int launch_rank(const float *colsum, int nb_col, const RouteEnd &r, hipStream_t st) {
    const size_t lds = (size_t)r.k * ceil_div(r.S, WAVE) * (r.E | 1) * 4;
    auto kern = route_rank_kernel<P>;
    if (lds > 48 * 1024) MOLE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, RANK_COUNTS * 4));
    hipLaunchKernelGGL(kern, dim3(1), dim3(FIN_THREADS), lds, st, r, colsum, nb_col);
    MOLE_LAUNCH_CHECK();
    return 0;
}
static int route_rank(const float *colsum, int nb_col, const RouteEnd &r, hipStream_t st) {
    const int p = ceil_div(r.k * ceil_div(r.S, WAVE), FIN_THREADS / WAVE);
    if (p <= 1) return launch_rank<1>(colsum, nb_col, r, st);
    if (p <= 2) return launch_rank<2>(colsum, nb_col, r, st);
    if (p <= 4) return launch_rank<4>(colsum, nb_col, r, st);
    return launch_rank<RANK_PAIRS / FIN_THREADS>(colsum, nb_col, r, st);
}

// The whole routing of scores (or of logits, to which bias is added if given and whose softmax then goes to `scores`).
static int route_from(const float *in, const float *bias, int logits, int normalize, float *scores, float *gates, const RouteEnd &r, void *workspace,
                      size_t workspace_bytes, hipStream_t st) {
    const int nb = ceil_div(r.S > 0 ? r.S : 1, RT_TOKENS);
    char *ws = (char *)workspace;
    if (r.S <= few_block(r.E)) return launch_tokens(true, in, bias, logits, normalize, scores, gates, nullptr, nullptr, 1, r, st);
    const bool few = r.S <= FEW_TOKENS && workspace_bytes >= few_bytes(r.S, r.E), rank = rank_in_one_block(r.S, r.E, r.k);
    if (nb == 1 && !(few && rank && r.E > 64)) return launch_tokens(false, in, bias, logits, normalize, scores, gates, nullptr, nullptr, 1, r, st);
    if (rank) {
        float *colsum = (float *)ws;
        const int blocks = few ? ceil_div(r.S, few_block(r.E)) : nb;
        if (int rc = launch_tokens(few, in, bias, logits, normalize, scores, gates, nullptr, colsum, blocks, r, st)) return rc;
        return route_rank(colsum, blocks, r, st);
    }
    int32_t *hist = (int32_t *)ws;
    ws += align256((size_t)nb * r.k * r.E * sizeof(int32_t));
    int32_t *basej = (int32_t *)ws;
    ws += align256((size_t)r.k * r.E * sizeof(int32_t));
    float *colsum = (float *)ws;
    ws += align256((size_t)nb * r.E * sizeof(float));
    float *colpart = (float *)ws;
    if (int rc = launch_tokens(false, in, bias, logits, normalize, scores, gates, hist, colsum, nb, r, st)) return rc;
    return route_after_topk(r, hist, basej, colsum, colpart, nb, RT_TOKENS, st);
}

extern "C" int mole_route(const float *scores, int S, int E, int k, double capacity_factor, int normalize_gate,
                          int alignment, int layout, int32_t *idx, int32_t *loc, float *gates, int32_t *row,
                          int32_t *counts, int32_t *kept_rows, int32_t *offsets, int32_t *capacity,
                          float *l_aux, void *workspace, size_t workspace_bytes, mole_stream_t stream) {
    MOLE_REQUIRE(S >= 0 && E >= 1 && E <= MOLE_MAX_EXPERTS, "mole_route: need S >= 0 and 1 <= E <= %d (S=%d E=%d)",
                 MOLE_MAX_EXPERTS, S, E);
    MOLE_REQUIRE(k >= 1 && k <= MOLE_MAX_TOPK && k <= E, "mole_route: need 1 <= k <= min(E, %d) (k=%d E=%d)",
                 MOLE_MAX_TOPK, k, E);
    MOLE_REQUIRE(alignment >= 1, "mole_route: alignment must be >= 1");
    MOLE_REQUIRE(layout == MOLE_LAYOUT_PADDED || layout == MOLE_LAYOUT_RAGGED, "mole_route: bad layout %d", layout);
    MOLE_REQUIRE(counts && kept_rows && offsets && capacity && workspace, "mole_route: null output pointer");
    MOLE_REQUIRE(S == 0 || (scores && idx && loc && gates && row), "mole_route: null token buffer");
    MOLE_REQUIRE((long long)S * k < INT_MAX && (long long)S * E < (1ll << 40), "mole_route: S*k too large");
    if (workspace_bytes < route_hist_bytes(S, E, k)) {
        set_error("mole_route: workspace of %zu bytes, need %zu", workspace_bytes, mole_route_workspace_bytes(S, E, k));
        return MOLE_E_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    ScopedTiming timing(MOLE_K_ROUTE, st);
    const RouteEnd r = route_end(S, E, k, capacity_factor, alignment, layout, idx, loc, row, counts, kept_rows, offsets, capacity, l_aux);
    return route_from(scores, nullptr, LOGITS_NONE, normalize_gate, nullptr, gates, r, workspace, workspace_bytes, st);
}

// ---------------------------------------------------------------------------------------------
// mole_route without a workspace argument and without any allocation: the per-block histograms, the per-choice
// bases and the column sums of the scores live in a file-scope device array.  Each GPU the library runs on holds
// its own copy of the array until the process ends.  The array's name is only a host-side handle; the address
// the kernels get is looked up once per device with hipGetSymbolAddress and kept.
// ---------------------------------------------------------------------------------------------
#define MOLE_ROUTE_SCRATCH_BYTES (8u << 20)
static __device__ __align__(256) unsigned char scratch[MOLE_ROUTE_SCRATCH_BYTES];

namespace mole {
constexpr int MAX_SCRATCH_DEVICES = 64;
static void *g_scratch_ptr[MAX_SCRATCH_DEVICES];
static std::mutex g_scratch_mu;

// device address of `scratch` on the current device
static int route_scratch(void **out) {
    int dev = 0;
    MOLE_HIP(hipGetDevice(&dev));
    MOLE_REQUIRE(dev >= 0 && dev < MAX_SCRATCH_DEVICES, "mole_route_static: device %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev] == nullptr) {
        void *p = nullptr;
        MOLE_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        MOLE_REQUIRE(p != nullptr, "mole_route_static: hipGetSymbolAddress returned no address");
        g_scratch_ptr[dev] = p;
    }
    *out = g_scratch_ptr[dev];
    return 0;
}
}  // namespace mole

extern "C" size_t mole_route_static_max_bytes(void) { return MOLE_ROUTE_SCRATCH_BYTES; }

extern "C" int mole_route_static(const float *scores, int S, int E, int k, double capacity_factor, int normalize_gate,
                                 int alignment, int layout, int32_t *idx, int32_t *loc, float *gates, int32_t *row,
                                 int32_t *counts, int32_t *kept_rows, int32_t *offsets, int32_t *capacity, float *l_aux,
                                 mole_stream_t stream) {
    const size_t need = mole_route_workspace_bytes(S, E, k);
    if (need == 0 || need > MOLE_ROUTE_SCRATCH_BYTES) {
        set_error("mole_route_static: S=%d E=%d k=%d needs %zu bytes of scratch, the static array holds %zu "
                  "(use mole_route with a workspace of your own)", S, E, k, need, (size_t)MOLE_ROUTE_SCRATCH_BYTES);
        return need == 0 ? MOLE_E_INVALID : MOLE_E_WORKSPACE;
    }
    void *ptr = nullptr;
    if (int rc = route_scratch(&ptr)) return rc;
    // every word of the scratch that a kernel of the route reads has been written by an earlier kernel of the
    // same call (the histograms by the top-k blocks, the bases and column sums by the scan / finish kernels), so
    // nothing needs clearing between calls; calls that overlap on one GPU would race on it
    return mole_route(scores, S, E, k, capacity_factor, normalize_gate, alignment, layout, idx, loc, gates, row, counts,
                      kept_rows, offsets, capacity, l_aux, ptr, MOLE_ROUTE_SCRATCH_BYTES, stream);
}

// ---------------------------------------------------------------------------------------------
// softmax over experts (MOLE/utils/Ugate.py:13) and the backward from dgates to dlogits
// ---------------------------------------------------------------------------------------------
namespace mole {

// One group of G lanes per token, VPL values per lane.
template <int VPL>
__global__ __launch_bounds__(256) void softmax_fwd_kernel(const float *__restrict__ logits,
                                                          const float *__restrict__ bias, int S, int E, int logG,
                                                          float *__restrict__ scores) {
    const int lane = threadIdx.x & 63;
    const int G = 1 << logG;
    const int g = lane & (G - 1), tg = lane >> logG;
    const int tpw = 64 >> logG;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int token = wave * tpw + tg;
    const bool tv = token < S;
    float v[VPL];
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        const bool ok = tv && e < E;
        // (an unconditional load from a clamped address; entries that do not exist become -inf)
        const float lg = load_or_zero(logits + (size_t)min(token, S - 1) * E + min(e, E - 1), ok);
        v[r] = lg + (ok ? (bias ? bias[e] : 0.f) : -INFINITY);
        mx = fmaxf(mx, v[r]);
    }
    mx = group_reduce(mx, logG, [](float a, float c) { return fmaxf(a, c); });
    float sum = 0.f;
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        v[r] = (tv && e < E) ? expf(v[r] - mx) : 0.f;
        sum += v[r];
    }
    sum = group_reduce(sum, logG, [](float a, float c) { return a + c; });
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        if (tv && e < E) scores[(size_t)token * E + e] = v[r] / sum;
    }
}

// Softmax backward on its own (the gate used outside the fused layer node): dlogits = s * (ds - sum_e ds s).
template <int VPL>
__global__ __launch_bounds__(256) void softmax_bwd_kernel(const float *__restrict__ dscores,
                                                          const float *__restrict__ scores, int S, int E, int logG,
                                                          float *__restrict__ dlogits) {
    const int lane = threadIdx.x & 63;
    const int G = 1 << logG;
    const int g = lane & (G - 1), tg = lane >> logG;
    const int tpw = 64 >> logG;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int token = wave * tpw + tg;
    const bool tv = token < S;
    float s[VPL], ds[VPL];
    float dot = 0.f;
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        const size_t at = (size_t)min(token, S - 1) * E + min(e, E - 1);
        s[r] = load_or_zero(scores + at, tv && e < E);
        ds[r] = load_or_zero(dscores + at, tv && e < E);
        dot += ds[r] * s[r];
    }
    dot = group_reduce(dot, logG, [](float a, float c) { return a + c; });
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        if (tv && e < E) dlogits[(size_t)token * E + e] = s[r] * (ds[r] - dot);
    }
}

// dlogits[i,e] = s[i,e] * (dscore[i,e] - sum_e' dscore[i,e'] s[i,e']), dscore scattered from dgates
// through gate_j = graw_j / max(sum graw, eps).  The token's group of lanes shares the k-sized part, then
// writes the row.  With counts0 and d_l_aux given, dscore also carries the load-balancing loss
// l_aux = E/S^2 sum_e (sum_i s[i,e]) counts0[e]: d l_aux / d s[i,e] = E/S^2 counts0[e], the same for every token
// (the counts are integers and carry no gradient).
template <int VPL>
__global__ __launch_bounds__(256) void gate_bwd_kernel(const float *__restrict__ dgates,
                                                       const float *__restrict__ scores,
                                                       const int32_t *__restrict__ idx, int S, int E, int k,
                                                       int logG, int normalize, int through_softmax,
                                                       const int32_t *__restrict__ counts0,
                                                       const float *__restrict__ d_l_aux,
                                                       float *__restrict__ dlogits) {
    const int lane = threadIdx.x & 63;
    const int G = 1 << logG;
    const int g = lane & (G - 1), tg = lane >> logG;
    const int tpw = 64 >> logG;
    const int wave = blockIdx.x * 4 + (threadIdx.x >> 6);
    const int token = wave * tpw + tg;
    const bool tv = token < S;
    float s[VPL], ds[VPL];
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        s[r] = load_or_zero(scores + (size_t)min(token, S - 1) * E + min(e, E - 1), tv && e < E);
        ds[r] = 0.f;
    }
    if (counts0 != nullptr) {       // uniform over the grid
        const float scale = d_l_aux[0] * ((float)E / ((float)S * (float)S));
#pragma unroll
        for (int r = 0; r < VPL; ++r) ds[r] = scale * (float)counts0[min(g + (r << logG), E - 1)];
    }
    // Lane j < k of the token's group fetches choice j (index, incoming gradient, raw gate value), the sums over
    // the k choices are lane reductions, and each choice is then handed round the group.  (With every lane walking
    // the k choices itself the token paid 2 k dependent memory latencies.)
    const bool has = tv && g < k;
    const int tokc = min(token, S - 1), jc = min(g, k - 1);
    const int my_e = idx[(size_t)jc * S + tokc];
    const float my_dg = load_or_zero(dgates + (size_t)jc * S + tokc, has);
    const float my_gr = load_or_zero(scores + (size_t)tokc * E + min(max(my_e, 0), E - 1), has);
    const float denom = group_reduce(my_gr, logG, [](float a, float c) { return a + c; });
    const float dotg = group_reduce(my_dg * my_gr, logG, [](float a, float c) { return a + c; });
    const bool norm = k > 1 && normalize;
    const bool clamped = denom < FP32_EPS;
    const float den = clamped ? FP32_EPS : denom;
    const float sub = (norm && !clamped) ? dotg / (den * den) : 0.f;
    const float my_dgraw = norm ? my_dg / den - sub : my_dg;
    const int group_base = lane & ~(G - 1);
    for (int j = 0; j < k; ++j) {
        int e;
        float dgraw;
        if (logG >= 6) {       // the group is the wave: lane j is a scalar read
            e = __builtin_amdgcn_readlane(my_e, j);
            dgraw = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, my_dgraw), j));
        } else {
            e = __shfl(my_e, group_base + j, WAVE);
            dgraw = __shfl(my_dgraw, group_base + j, WAVE);
        }
        if ((e & (G - 1)) == g) {
            const int rr = e >> logG;
#pragma unroll
            for (int r = 0; r < VPL; ++r)
                if (r == rr) ds[r] += dgraw;
        }
    }
    float dot = 0.f;
#pragma unroll
    for (int r = 0; r < VPL; ++r) dot += ds[r] * s[r];
    dot = group_reduce(dot, logG, [](float a, float c) { return a + c; });
#pragma unroll
    for (int r = 0; r < VPL; ++r) {
        const int e = g + (r << logG);
        if (tv && e < E) dlogits[(size_t)token * E + e] = through_softmax ? s[r] * (ds[r] - dot) : ds[r];
    }
}


// ---- the gate for fp32 tokens and small gates (E <= 32): one wave per token ------------------------------
// Lane l holds 4 columns of the token per pass (M / 256 passes) and accumulates its share of all E logits in
// registers against the matching columns of Wg (16-64 KB in all: L1/L2 hits); the E sums are reduced over the
// wave with lane patterns, lane e keeps logit e, and the softmax runs over the wave.  fp32 FMAs throughout.
// (The two-kernel path spends 44 us on a 4096 x 512 x 8 product: one 128 x 128 tile of the GEMM kernel per 128
// tokens leaves most of the chip idle.)
template <int EB>
__global__ __launch_bounds__(256) void gate_fwd_f32_kernel(const float *__restrict__ x, const float *__restrict__ wg,
                                                           const float *__restrict__ bias, int S, int E, int M,
                                                           float *__restrict__ scores) {
    const int lane = threadIdx.x & 63;
    const int token = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (token >= S) return;                       // a whole wave
    float acc[EB];
#pragma unroll
    for (int e = 0; e < EB; ++e) acc[e] = 0.f;
    const float *xr = x + (size_t)token * M;
    for (int c = lane * 4; c < M; c += 256) {
        const float4 xv = *reinterpret_cast<const float4 *>(xr + c);
#pragma unroll
        for (int e = 0; e < EB; ++e) {            // rows past the gate repeat its last row and are not used
            const float4 wv = *reinterpret_cast<const float4 *>(wg + (size_t)min(e, E - 1) * M + c);
            acc[e] = fmaf(xv.w, wv.w, fmaf(xv.z, wv.z, fmaf(xv.y, wv.y, fmaf(xv.x, wv.x, acc[e]))));
        }
    }
    float mine = -INFINITY;
#pragma unroll
    for (int e = 0; e < EB; ++e) {
        const float sum = group_reduce(acc[e], 6, [](float a, float c) { return a + c; });
        if (lane == e && e < E) mine = sum + (bias ? bias[e] : 0.f);
    }
    const float mx = group_reduce(mine, 6, [](float a, float c) { return fmaxf(a, c); });
    const float ex = lane < E ? expf(mine - mx) : 0.f;
    const float den = group_reduce(ex, 6, [](float a, float c) { return a + c; });
    if (lane < E) scores[(size_t)token * E + lane] = ex / den;
}

// ---- fused gate: scores = softmax(x . Wg^T + bias) for bf16 tokens ------------------------------------
// A block of four waves owns 16 tokens; wave w contracts the w-th quarter of the model dimension with
// v_mfma_f32_16x16x32_bf16 (16 tokens x 16 experts x 32 of k per instruction), operands straight from
// global memory in the instruction's layout - lane l supplies 8 consecutive k (k slice l / 16) of token or
// expert l % 16 - with the fp32 gate weights rounded to bf16 on the fly, as the separate GEMM did.  The
// four partial logit tiles meet in LDS, then 16 lanes per token do the softmax.  EG = groups of 16 experts.
typedef __bf16 gate_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gate_f32x4 __attribute__((ext_vector_type(4)));

// STAGE: the token rows of a round reach the fragments by way of LDS.  Straight from memory, a load instruction of
// the instruction's layout touches 16 rows with 64 bytes each; staged, it fetches 512-byte pieces of two rows (at
// KSTEPS 8), and the fragments are 16-byte LDS reads (rows 16 bytes longer than their data: the 16 rows of a read
// fall into distinct banks).  A wave stages and reads its own rows only.
// ROUTE: the block goes on to the first stage of the routing for its 16 TG tokens - top-k, gate values, in-block
// ranks and per-expert histograms, the block's column sums for l_aux - while a token's scores are still in the 16
// lanes that formed them (the layout route_tokens_kernel works in: lane j of the group holds experts j, 16 + j, ...).
// The scores are written out as well (the backward needs them) but not read back: one kernel and 4 S E bytes less.
struct GateRoute {
    int k, normalize, nb;
    int32_t *idx, *lrank, *hist;
    float *gates, *colsum;
};
template <int EG, int KSTEPS, int TG, bool STAGE, bool ROUTE = false>   // TG groups of 16 tokens per block: Wg is read once for all of them
__global__ __launch_bounds__(256) void gate_fwd_kernel(const bf16_t *__restrict__ x, const float *__restrict__ wg,
                                                       const float *__restrict__ bias, int S, int E, int M,
                                                       float *__restrict__ scores, const GateRoute rt) {
    constexpr int RB = KSTEPS * 64, RS = RB + 16;               // staged row: bytes of data, bytes of stride
    constexpr int LPR = RB / 16, RPI = 64 / LPR;                // lanes per row, rows per load instruction
    constexpr int PART_BYTES = 4 * 16 * TG * (EG * 16 + 1) * 4;
    constexpr int STAGE_BYTES = STAGE ? 4 * 16 * TG * RS : 0;
    static_assert(!STAGE || STAGE_BYTES >= PART_BYTES, "the launch sizes the dynamic LDS for the staged rows");
    __shared__ __align__(16) char s_static[STAGE ? 16 : PART_BYTES];
    extern __shared__ __align__(16) char s_dyn[];               // STAGE: max(PART_BYTES, STAGE_BYTES), given at launch
    char *s_all = STAGE ? s_dyn : s_static;
    float (*part)[16 * TG][EG * 16 + 1] = reinterpret_cast<float (*)[16 * TG][EG * 16 + 1]>(s_all);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r16 = lane & 15, kq = lane >> 4;
    const int tok0 = blockIdx.x * 16 * TG;
    const int kbase = wave * (M >> 2) + 8 * kq;
    const bf16_t *xp[TG];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) xp[tg] = x + (size_t)min(tok0 + 16 * tg + r16, S - 1) * M + kbase;
    gate_f32x4 acc[TG][EG];
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
        for (int g = 0; g < EG; ++g) acc[tg][g] = gate_f32x4{0.f, 0.f, 0.f, 0.f};
    const int nsteps = M >> 7;                    // 32 of k per step, a quarter of M per wave
    // All loads of a round of KSTEPS steps go out first, unconditionally (a step past the end repeats the last
    // one and is masked below): under a condition each load would be waited for before the next is issued.  For
    // small gates the weights of the round are fetched ahead as well.
    constexpr bool W_AHEAD = EG * KSTEPS <= 16;
    for (int s0 = 0; s0 < nsteps; s0 += KSTEPS) {
        uint4 a[TG][KSTEPS];
        float4 wa[W_AHEAD ? KSTEPS : 1][W_AHEAD ? EG : 1][2];
        if constexpr (STAGE) {
            // load j of the round: rows RPI j + lane / LPR of the block's 16 TG, 16 bytes at (lane % LPR) 16 of the
            // round's RB; columns past the wave's quarter (steps past the end) repeat its last 16 bytes
            const int cb = min(s0 * 32 + (lane % LPR) * 8, (M >> 2) - 8);
#pragma unroll
            for (int j = 0; j < TG * KSTEPS; ++j) {
                const int rr = RPI * j + lane / LPR;
                const uint4 v = *reinterpret_cast<const uint4 *>(x + (size_t)min(tok0 + rr, S - 1) * M + wave * (M >> 2) + cb);
                a[j / KSTEPS][j % KSTEPS] = v;
            }
        }
#pragma unroll
        for (int i = 0; i < KSTEPS; ++i) {
            const int sc = min(s0 + i, nsteps - 1);
            if constexpr (!STAGE) {
#pragma unroll
                for (int tg = 0; tg < TG; ++tg) a[tg][i] = *reinterpret_cast<const uint4 *>(xp[tg] + sc * 32);
            }
            if constexpr (W_AHEAD) {
#pragma unroll
                for (int g = 0; g < EG; ++g) {
                    const float *wp = wg + (size_t)min(g * 16 + r16, E - 1) * M + kbase + sc * 32;
                    wa[i][g][0] = *reinterpret_cast<const float4 *>(wp);
                    wa[i][g][1] = *reinterpret_cast<const float4 *>(wp + 4);
                }
            }
        }
        __builtin_amdgcn_sched_barrier(0);       // or the scheduler moves each load down to its use again
        if constexpr (STAGE) {
            char *mine = s_all + wave * (16 * TG * RS);
#pragma unroll
            for (int j = 0; j < TG * KSTEPS; ++j)
                *reinterpret_cast<uint4 *>(mine + (RPI * j + lane / LPR) * RS + (lane % LPR) * 16) = a[j / KSTEPS][j % KSTEPS];
            // (written and read by this wave only: program order is enough)
#pragma unroll
            for (int i = 0; i < KSTEPS; ++i)
#pragma unroll
                for (int tg = 0; tg < TG; ++tg)
                    a[tg][i] = *reinterpret_cast<const uint4 *>(mine + (16 * tg + r16) * RS + i * 64 + kq * 16);
        }
#pragma unroll
        for (int i = 0; i < KSTEPS; ++i) {
            // (no branch here, so that the round stays one block of code and its loads stay ahead of it: a step
            // past the end multiplies zeros)
            const uint32_t keep = s0 + i < nsteps ? 0xffffffffu : 0u;
#pragma unroll
            for (int tg = 0; tg < TG; ++tg)
                a[tg][i] = make_uint4(a[tg][i].x & keep, a[tg][i].y & keep, a[tg][i].z & keep, a[tg][i].w & keep);
#pragma unroll
            for (int g = 0; g < EG; ++g) {
                float4 w0, w1;
                if constexpr (W_AHEAD) {
                    w0 = wa[i][g][0];
                    w1 = wa[i][g][1];
                } else {
                    const float *wp = wg + (size_t)min(g * 16 + r16, E - 1) * M + kbase + min(s0 + i, nsteps - 1) * 32;
                    w0 = *reinterpret_cast<const float4 *>(wp);
                    w1 = *reinterpret_cast<const float4 *>(wp + 4);
                }
                const gate_bf16x8 b = {(bf16_t)w0.x, (bf16_t)w0.y, (bf16_t)w0.z, (bf16_t)w0.w,
                                       (bf16_t)w1.x, (bf16_t)w1.y, (bf16_t)w1.z, (bf16_t)w1.w};
#pragma unroll
                for (int tg = 0; tg < TG; ++tg)
                    acc[tg][g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_bf16x8, a[tg][i]), b, acc[tg][g], 0, 0, 0);
            }
        }
    }
    // acc[tg][g][r] = partial logit of token 16 tg + 4 kq + r, expert 16 g + r16
    if constexpr (STAGE) __syncthreads();         // the partial sums take the place of the staged rows
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
        for (int g = 0; g < EG; ++g)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][16 * tg + 4 * kq + r][g * 16 + r16] = acc[tg][g][r];
    __syncthreads();
    const int j = threadIdx.x & 15;               // 16 lanes per token
    constexpr int BT = 16 * TG;
    // routing: [k][BT] experts and raw gate values, four histograms, four rows of column sums - behind the staging area
    int *s_idx = reinterpret_cast<int *>(s_dyn + STAGE_BYTES);
    float *s_graw = reinterpret_cast<float *>(s_idx + (ROUTE ? rt.k : 0) * BT);
    int *s_hist = reinterpret_cast<int *>(s_graw + (ROUTE ? rt.k : 0) * BT);
    float *s_col = reinterpret_cast<float *>(s_hist + 4 * E);
    float colacc[EG];
#pragma unroll
    for (int g = 0; g < EG; ++g) colacc[g] = 0.f;
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
        const int t = 16 * tg + (threadIdx.x >> 4);
        const int token = tok0 + t;
        float v[EG];
        float mx = -INFINITY;
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            const int e = g * 16 + j;
            v[g] = e < E ? part[0][t][e] + part[1][t][e] + part[2][t][e] + part[3][t][e] + (bias ? bias[e] : 0.f) : -INFINITY;
            mx = fmaxf(mx, v[g]);
        }
        for (int m = 8; m >= 1; m >>= 1) mx = fmaxf(mx, __shfl_xor(mx, m, WAVE));
        float sum = 0.f;
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            v[g] = g * 16 + j < E ? expf(v[g] - mx) : 0.f;
            sum += v[g];
        }
        for (int m = 8; m >= 1; m >>= 1) sum += __shfl_xor(sum, m, WAVE);
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            const int e = g * 16 + j;
            v[g] = v[g] / sum;
            if (token < S && e < E) scores[(size_t)token * E + e] = v[g];
        }
        if constexpr (ROUTE) {
            // the k rounds of route_tokens_kernel on the token's scores (the same keys, the same tie rule)
            uint32_t key[EG];
#pragma unroll
            for (int g = 0; g < EG; ++g) {
                const bool ok = token < S && g * 16 + j < E;
                const float sv = __uint_as_float(__float_as_uint(v[g]) & (ok ? 0xffffffffu : 0u));
                colacc[g] += sv;
                key[g] = ok ? topk_key(sv) : 0u;
            }
            for (int c = 0; c < rt.k; ++c) {
                uint32_t best = key[0];
#pragma unroll
                for (int g = 1; g < EG; ++g) best = max(best, key[g]);
                const uint32_t top = group_reduce(best, 4, [](uint32_t a, uint32_t b2) { return max(a, b2); });
                int cand = INT_MAX;
#pragma unroll
                for (int g = EG - 1; g >= 0; --g)
                    if (key[g] == top) cand = j + (g << 4);                // ends on the lane's lowest such expert
                if (top == 0u) cand = INT_MAX;                             // nothing available (a token past the end)
                const int bi = group_reduce(cand, 4, [](int a, int b2) { return min(a, b2); });
                const bool mine = bi != INT_MAX && (bi & 15) == j;
#pragma unroll
                for (int g = 0; g < EG; ++g)
                    if (mine && (bi >> 4) == g) key[g] = 0u;
                if (j == 0 && token < S) {
                    s_idx[c * BT + t] = bi;
                    s_graw[c * BT + t] = topk_unkey(top);
                }
            }
        }
    }
    if constexpr (ROUTE) {
        // column sums of the scores: fold the wave's four token groups, then (in the tail) the four waves
#pragma unroll
        for (int g = 0; g < EG; ++g) {
            float c = colacc[g];
            c += __shfl_xor(c, 16, WAVE);
            c += __shfl_xor(c, 32, WAVE);
            const int e = g * 16 + j;
            if (lane < 16 && e < E) s_col[wave * E + e] = c;
        }
        topk_block_tail(BT, S, E, rt.k, rt.normalize, s_idx, s_graw, s_hist, s_col, rt.idx, rt.lrank, rt.gates, rt.hist,
                        rt.colsum, rt.nb);
    }
}

// ---- logits alone, for few tokens ------------------------------------------------------------------------------------
// A block owns 16 TG tokens x 16 experts; its four waves take a quarter of the model dimension each, in the order of
// gate_fwd_kernel (whose logits these equal bit for bit where it applies: bf16, M a multiple of 128).  One block per
// 16-expert group instead of one that reads all of Wg: 512 KB of Wg for one token is then 4 blocks' work side by side
// instead of one block's 20 us, and 256 tokens x 256 experts x 2048 are 256 blocks (10 us; one 256 x 256 tile: 54).
// Fragments come straight from memory.  Steps past a wave's share repeat its last one and are not multiplied; of a step
// that M ends in, the lanes past the end are zero on both sides (an infinite weight times zero would be NaN).
// fp32: every step of a round and every component of its 16 bytes has sums of its own, added up in pairs at the end, as are
// the waves'.  A single running sum per wave is a chain of M / 4 additions, which left the logits 1.9 (M = 256) to 3.6 times
// (M = 4096) as far off as gate_fwd_f32_kernel's 64 lanes do, and with them the gate values; this way they are as close or
// closer.
// QUARTERS: a block is one of the four waves and writes its partial logits, [4][S][E], which route_tokens adds up in the same order.  A
// handful of tokens has so few blocks that each pulls its share of Wg through one CU (1 token, 64 experts of 2048: four blocks
// of 128 KB, 6.2 us; now 3.6); see gate_quarters.
template <typename T, int TG, bool QUARTERS>
__global__ __launch_bounds__(QUARTERS ? 64 : 256, QUARTERS ? 1 : 2) void gate_logits_kernel(const T *__restrict__ x, const float *__restrict__ wg,
                                                          const float *__restrict__ bias, int S, int E, int M,
                                                          float *__restrict__ logits) {
    constexpr int EPC = 16 / sizeof(T), KSTEP = 4 * EPC, U = QUARTERS && sizeof(T) == 2 ? 16 : TG == 1 ? 8 : 4, NA = sizeof(T) == 2 ? 1 : 4 * U;
    __shared__ float part[4][16 * TG][17];
    const int lane = threadIdx.x & 63, wave = QUARTERS ? blockIdx.z : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r16 = lane & 15, kq = lane >> 4;
    const int tok0 = blockIdx.x * 16 * TG, e0 = blockIdx.y * 16;
    const int steps = (M + KSTEP - 1) / KSTEP, s_lo = wave * steps / 4, s_hi = (wave + 1) * steps / 4;
    const T *xp[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) xp[t] = x + (size_t)min(tok0 + 16 * t + r16, S - 1) * M;
    const float *wp = wg + (size_t)min(e0 + r16, E - 1) * M;
    gate_f32x4 acc[TG][NA];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int i = 0; i < NA; ++i) acc[t][i] = gate_f32x4{0.f, 0.f, 0.f, 0.f};
    for (int s = s_lo; s < s_hi; s += U) {
        uint4 a[TG][U];
        float4 w[U][EPC / 4];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(min(s + u, s_hi - 1) * KSTEP + kq * EPC, M - EPC);
#pragma unroll
            for (int t = 0; t < TG; ++t) a[t][u] = *reinterpret_cast<const uint4 *>(xp[t] + k);
#pragma unroll
            for (int h = 0; h < EPC / 4; ++h) w[u][h] = *reinterpret_cast<const float4 *>(wp + k + 4 * h);
        }
        __builtin_amdgcn_sched_barrier(0);       // all loads of the round first
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= s_hi) break;
            if ((s + u + 1) * KSTEP > M && (s + u) * KSTEP + kq * EPC >= M) {
#pragma unroll
                for (int t = 0; t < TG; ++t) a[t][u] = make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
                for (int h = 0; h < EPC / 4; ++h) w[u][h] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int t = 0; t < TG; ++t) {
                const uint4 v = a[t][u];
                if constexpr (sizeof(T) == 2) {
                    const float4 w0 = w[u][0], w1 = w[u][EPC / 4 - 1];
                    const gate_bf16x8 b = {(bf16_t)w0.x, (bf16_t)w0.y, (bf16_t)w0.z, (bf16_t)w0.w,
                                           (bf16_t)w1.x, (bf16_t)w1.y, (bf16_t)w1.z, (bf16_t)w1.w};
                    acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(gate_bf16x8, v), b, acc[t][0], 0, 0, 0);
                } else {
                    gate_f32x4 (&c)[NA] = acc[t];
                    c[4 * u] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v.x), w[u][0].x, c[4 * u], 0, 0, 0);
                    c[4 * u + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v.y), w[u][0].y, c[4 * u + 1], 0, 0, 0);
                    c[4 * u + 2] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v.z), w[u][0].z, c[4 * u + 2], 0, 0, 0);
                    c[4 * u + 3] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(v.w), w[u][0].w, c[4 * u + 3], 0, 0, 0);
                }
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TG; ++t) {
#pragma unroll
        for (int half = NA / 2; half >= 1; half /= 2)
#pragma unroll
            for (int i = 0; i < half; ++i) acc[t][i] += acc[t][i + half];
        if constexpr (QUARTERS) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int token = tok0 + 16 * t + 4 * kq + r;
                if (token < S && e0 + r16 < E) logits[((size_t)wave * S + token) * E + e0 + r16] = acc[t][0][r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) part[wave][16 * t + 4 * kq + r][r16] = acc[t][0][r];
        }
    }
    if constexpr (QUARTERS) return;
    __syncthreads();
    const int e = e0 + (threadIdx.x & 15);
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        const int tl = 16 * t + (threadIdx.x >> 4);
        const float p0 = part[0][tl][e - e0], p1 = part[1][tl][e - e0], p2 = part[2][tl][e - e0], p3 = part[3][tl][e - e0];
        const float sum = sizeof(T) == 2 ? p0 + p1 + p2 + p3 : (p0 + p1) + (p2 + p3);
        if (tok0 + tl < S && e < E) logits[(size_t)(tok0 + tl) * E + e] = sum + (bias ? bias[e] : 0.f);
    }
}

// Wg in the operand type of the GEMM path
__global__ __launch_bounds__(256) void f32_to_bf16_kernel(const float *__restrict__ in, bf16_t *__restrict__ out, size_t n4) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n4) return;
    const float4 v = reinterpret_cast<const float4 *>(in)[i];
    typedef __bf16 bf16x4_ __attribute__((ext_vector_type(4)));
    reinterpret_cast<uint2 *>(out)[i] = __builtin_bit_cast(uint2, bf16x4_{(bf16_t)v.x, (bf16_t)v.y, (bf16_t)v.z, (bf16_t)v.w});
}

}  // namespace mole

#define MOLE_VPL_DISPATCH(vpl, KERNEL, grid, st, ...)                                              \
    do {                                                                                           \
        if ((vpl) <= 1) hipLaunchKernelGGL(KERNEL<1>, grid, dim3(256), 0, st, __VA_ARGS__);         \
        else if ((vpl) <= 2) hipLaunchKernelGGL(KERNEL<2>, grid, dim3(256), 0, st, __VA_ARGS__);    \
        else if ((vpl) <= 4) hipLaunchKernelGGL(KERNEL<4>, grid, dim3(256), 0, st, __VA_ARGS__);    \
        else if ((vpl) <= 8) hipLaunchKernelGGL(KERNEL<8>, grid, dim3(256), 0, st, __VA_ARGS__);    \
        else hipLaunchKernelGGL(KERNEL<16>, grid, dim3(256), 0, st, __VA_ARGS__);                   \
    } while (0)

extern "C" int mole_softmax_fwd(const float *logits, const float *logit_bias, int S, int E, float *scores,
                                mole_stream_t stream) {
    MOLE_REQUIRE(S >= 0 && E >= 1 && E <= MOLE_MAX_EXPERTS, "mole_softmax_fwd: bad sizes S=%d E=%d", S, E);
    if (S == 0) return 0;
    MOLE_REQUIRE(logits && scores, "mole_softmax_fwd: null pointer");
    int logG = 0;
    while ((1 << logG) < E && logG < 6) ++logG;       // (16-lane groups as in the top-k: 18.1 against 17.1 us at 256 experts)
    const int vpl = ceil_div(E, 1 << logG);
    const int tpw = 64 >> logG;
    const dim3 grid(ceil_div(S, 4 * tpw));
    ScopedTiming timing(MOLE_K_GATE_FWD, (hipStream_t)stream);
    MOLE_VPL_DISPATCH(vpl, softmax_fwd_kernel, grid, (hipStream_t)stream, logits, logit_bias, S, E, logG, scores);
    MOLE_LAUNCH_CHECK();
    return 0;
}

// dynamic LDS of gate_fwd_kernel<1, 4, 2, true>: the staged token rows (four waves x 32 rows of 4 x 64 + 16 bytes)
static constexpr unsigned GATE_STAGE_LDS = 4 * 32 * (4 * 64 + 16);
// tokens per block of the fused gate + routing kernels (TG = 2)
static constexpr int GATE_ROUTE_TOKENS = 32;

static size_t gate_route_fused_bytes(int S, int E, int k) {
    const size_t nb = (size_t)ceil_div(S > 0 ? S : 1, GATE_ROUTE_TOKENS);
    return align256(nb * k * E * sizeof(int32_t)) + align256((size_t)k * E * sizeof(int32_t)) +
           align256(nb * E * sizeof(float)) + align256((size_t)COLSUM_SLICES * E * sizeof(float));
}

// How the gate and the routing of a call run.
//   FUSED   the gate kernel does the tokens' part of the routing as well: bf16, gates of up to 64 experts, many tokens
//           (a block of 32 tokens reads all of Wg, so with few tokens few blocks read it one after the other:
//           1 token, 64 experts of 2048: 21 + 17 + 4 us in three kernels against 4 + 7 us)
//   FEW     logits by 16 x 16 tiles, then softmax and routing: up to 2048 tokens (2048 blocks at 256 experts; beyond, the
//           re-reads of x and Wg by the tiles cost more than the GEMM's tiles), in fp32, whose GEMM tiles are 128 x 128 of one
//           block's walk over M, up to 3072 blocks (2977 tokens, 200 experts of 1536: 139 / 69 us; 8192, 40 of 2048: 167 / 52; 16384, 64
//           of 1032: 97 / 66; 16384, 128 of 512, 4096 blocks: 64 / 71; 32768, 80 of 1032: 111 / 137)
//   SCORES  fp32, up to 32 experts: mole_gate_fwd's wave per token, then the routing of the scores
//   GEMM    logits on the grouped-GEMM tiles, then softmax and routing
enum { GR_FUSED, GR_FEW, GR_SCORES, GR_GEMM };
// The logits of FEW by quarters of the model dimension: while four times the blocks are at most one for every CU, and where the routing adds
// them up (all but 5 to 64 tokens over 1024 experts, top-16, whose pairs route_rank does not hold: see route_from).
static bool gate_quarters(int S, int E, int k) {
    return S <= RT_TOKENS && ceil_div(S, 16) * ceil_div(E, 16) <= 64 && (E <= 64 || S <= few_block(E) || rank_in_one_block(S, E, k));
}
static int gate_route_path(int dtype, int S, int E, int M) {
    if (dtype == MOLE_BF16 && M % 128 == 0 && E <= 64 && S > RT_TOKENS) return GR_FUSED;
    if (S <= 2048 || (dtype == MOLE_F32 && E > 32 && (long)ceil_div(S, 32) * ceil_div(E, 16) <= 3072)) return GR_FEW;
    return dtype == MOLE_F32 && E <= 32 ? GR_SCORES : GR_GEMM;
}

// small: with the routing's small blocks and the logits by quarters; otherwise the least that the call does with
static size_t gate_route_bytes(int dtype, int S, int E, int M, int k, bool small) {
    const int path = gate_route_path(dtype, S, E, M);
    if (path == GR_FUSED) return gate_route_fused_bytes(S, E, k);
    size_t n = small ? mole_route_workspace_bytes(S, E, k) : route_hist_bytes(S, E, k);
    if (path != GR_SCORES) n += align256((small && path == GR_FEW && gate_quarters(S, E, k) ? 4 : 1) * (size_t)S * E * sizeof(float));
    if (path == GR_GEMM && dtype == MOLE_BF16) n += align256((size_t)E * M * sizeof(bf16_t));
    return n;
}
extern "C" size_t mole_gate_route_shape_workspace_bytes(int dtype, int S, int E, int M, int k) {
    return S < 0 || E <= 0 || M <= 0 || k <= 0 ? 0 : gate_route_bytes(dtype, S, E, M, k, true);
}
namespace mole {
size_t gate_route_least_bytes(int dtype, int S, int E, int M, int k) { return gate_route_bytes(dtype, S, E, M, k, false); }
}

extern "C" size_t mole_gate_route_workspace_bytes(int S, int E, int k) {
    if (S < 0 || E <= 0 || k <= 0) return 0;
    return S > RT_TOKENS ? gate_route_fused_bytes(S, E, k)
                         : std::max(gate_route_fused_bytes(S, E, k), mole_gate_route_shape_workspace_bytes(MOLE_BF16, S, E, 128, k));
}

namespace mole {
// mole_gate_route, which also writes down the token of every kept row (null: it does not)
int gate_route(const void *x, int dtype, const float *wg, const float *logit_bias, int S, int E, int M, int k, double capacity_factor,
               int normalize_gate, int alignment, int layout, float *scores, int32_t *idx, int32_t *loc, float *gates, int32_t *row, int32_t *counts,
               int32_t *kept_rows, int32_t *offsets, int32_t *capacity, float *l_aux, int32_t *token_of, void *workspace, size_t workspace_bytes,
               mole_stream_t stream) {
    MOLE_REQUIRE(dtype == MOLE_BF16 || dtype == MOLE_F32, "mole_gate_route: bad dtype %d", dtype);
    const int epc = dtype == MOLE_BF16 ? 8 : 4;
    MOLE_REQUIRE(S >= 1 && E >= 1 && E <= MOLE_MAX_EXPERTS && M >= epc && M % epc == 0,
                 "mole_gate_route: needs S >= 1, 1 <= E <= %d and M a multiple of %d (S=%d E=%d M=%d dtype=%d)", MOLE_MAX_EXPERTS,
                 epc, S, E, M, dtype);
    MOLE_REQUIRE(k >= 1 && k <= MOLE_MAX_TOPK && k <= E, "mole_gate_route: need 1 <= k <= min(E, %d) (k=%d E=%d)", MOLE_MAX_TOPK, k, E);
    MOLE_REQUIRE(alignment >= 1, "mole_gate_route: alignment must be >= 1");
    MOLE_REQUIRE(layout == MOLE_LAYOUT_PADDED || layout == MOLE_LAYOUT_RAGGED, "mole_gate_route: bad layout %d", layout);
    MOLE_REQUIRE(x && wg && scores && idx && loc && gates && row && counts && kept_rows && offsets && capacity && workspace,
                 "mole_gate_route: null pointer");
    // (fp32 as in the entry points it joins; bf16 kernels read the fp32 weights, and small gates the tokens, at any alignment
    // of their elements: a gate's weight may be a view into a flat parameter buffer)
    const bool any_x = dtype == MOLE_BF16 && E <= 64 && M % 128 == 0, any_wg = dtype == MOLE_BF16;
    MOLE_REQUIRE((any_x || ((uintptr_t)x & 15) == 0) && (any_wg || ((uintptr_t)wg & 15) == 0),
                 "mole_gate_route: x and wg must be 16-byte aligned");
    MOLE_REQUIRE((long long)S * k < INT_MAX, "mole_gate_route: S*k too large");
    const size_t need = mole_gate_route_shape_workspace_bytes(dtype, S, E, M, k);
    const bool small = workspace_bytes >= need;
    if (workspace_bytes < gate_route_least_bytes(dtype, S, E, M, k)) {
        set_error("mole_gate_route: workspace of %zu bytes, need %zu", workspace_bytes, need);
        return MOLE_E_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    const RouteEnd r = route_end(S, E, k, capacity_factor, alignment, layout, idx, loc, row, counts, kept_rows, offsets, capacity, l_aux, token_of);
    const int path = gate_route_path(dtype, S, E, M);
    char *ws = (char *)workspace;
    if (path != GR_FUSED) {
        void *route_ws = ws;
        const size_t route_bytes = small ? mole_route_workspace_bytes(S, E, k) : route_hist_bytes(S, E, k);
        ws += route_bytes;
        if (path == GR_SCORES) {
            if (int rc = mole_gate_fwd(x, dtype, wg, logit_bias, S, E, M, scores, stream)) return rc;
            ScopedTiming timing(MOLE_K_ROUTE, st);
            return route_from(scores, nullptr, LOGITS_NONE, normalize_gate, nullptr, gates, r, route_ws, route_bytes, st);
        }
        float *logits = (float *)ws;
        if (small && path == GR_FEW && gate_quarters(S, E, k)) {
            const dim3 grid(ceil_div(S, 16), ceil_div(E, 16), 4);
            if (dtype == MOLE_BF16) timed_launch(MOLE_K_GATE_FWD, gate_logits_kernel<bf16_t, 1, true>, grid, dim3(64), 0, st, (const bf16_t *)x, wg, nullptr, S, E, M, logits);
            else timed_launch(MOLE_K_GATE_FWD, gate_logits_kernel<float, 1, true>, grid, dim3(64), 0, st, (const float *)x, wg, nullptr, S, E, M, logits);
            MOLE_LAUNCH_CHECK();
            ScopedTiming timing(MOLE_K_ROUTE, st);
            return route_from(logits, logit_bias, dtype == MOLE_BF16 ? LOGITS_PARTS : LOGITS_PAIRS, normalize_gate, scores, gates, r, route_ws, route_bytes, st);
        }
        ws += align256((size_t)S * E * sizeof(float));
        if (path == GR_FEW) {
            // Wg is read once for 16 or 32 tokens.  fp32 gates of one or two groups of experts have the blocks to spare
            // (2048 tokens, 16 experts of 4096, with the routing: 32 us in 16s, 38 in 32s); wide ones do not (2000, 256 of 2048: 97 / 86).
            const int tg = S <= 512 || (dtype == MOLE_F32 && E <= 32) ? 1 : 2;
            const dim3 grid(ceil_div(S, 16 * tg), ceil_div(E, 16));
#define MOLE_GL(T, TG) timed_launch(MOLE_K_GATE_FWD, gate_logits_kernel<T, TG, false>, grid, dim3(256), 0, st, (const T *)x, wg, logit_bias, S, E, M, logits)
            if (dtype == MOLE_BF16) { if (tg == 1) MOLE_GL(bf16_t, 1); else MOLE_GL(bf16_t, 2); }
            else { if (tg == 1) MOLE_GL(float, 1); else MOLE_GL(float, 2); }
#undef MOLE_GL
            MOLE_LAUNCH_CHECK();
            ScopedTiming timing(MOLE_K_ROUTE, st);
            return route_from(logits, nullptr, LOGITS_WHOLE, normalize_gate, scores, gates, r, route_ws, route_bytes, st);
        }
        const void *w = wg;
        if (dtype == MOLE_BF16) {
            const size_t n4 = (size_t)E * M / 4;
            hipLaunchKernelGGL(f32_to_bf16_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, st, wg, (bf16_t *)ws, n4);
            MOLE_LAUNCH_CHECK();
            w = ws;
        }
        if (int rc = mole_gemm_nt(x, w, dtype, S, E, M, logits, stream)) return rc;
        ScopedTiming timing(MOLE_K_ROUTE, st);
        return route_from(logits, logit_bias, LOGITS_WHOLE, normalize_gate, scores, gates, r, route_ws, route_bytes, st);
    }
    const int nb = ceil_div(S, GATE_ROUTE_TOKENS);
    int32_t *hist = (int32_t *)ws;
    ws += align256((size_t)nb * k * E * sizeof(int32_t));
    int32_t *basej = (int32_t *)ws;
    ws += align256((size_t)k * E * sizeof(int32_t));
    float *colsum = (float *)ws;
    ws += align256((size_t)nb * E * sizeof(float));
    float *colpart = (float *)ws;
    const bool ranks = rank_in_one_block(S, E, k);
    const GateRoute rt{k, normalize_gate, nb, idx, loc, ranks ? nullptr : hist, gates, colsum};
    const unsigned route_lds = (unsigned)((size_t)k * GATE_ROUTE_TOKENS * 8 + (size_t)E * 4 * 4 * 2);
    const bf16_t *xb = (const bf16_t *)x;
    if (E <= 16)
        timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<1, 4, 2, true, true>, dim3(nb), dim3(256), GATE_STAGE_LDS + route_lds, st, xb, wg,
                     logit_bias, S, E, M, scores, rt);
    else if (E <= 32)
        timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<2, 4, 2, false, true>, dim3(nb), dim3(256), route_lds, st, xb, wg, logit_bias, S,
                     E, M, scores, rt);
    else
        timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<4, 4, 2, false, true>, dim3(nb), dim3(256), route_lds, st, xb, wg, logit_bias, S,
                     E, M, scores, rt);
    MOLE_LAUNCH_CHECK();
    ScopedTiming timing(MOLE_K_ROUTE, st);
    return ranks ? route_rank(colsum, nb, r, st) : route_after_topk(r, hist, basej, colsum, colpart, nb, GATE_ROUTE_TOKENS, st);
}
}  // namespace mole

extern "C" int mole_gate_route(const void *x, int dtype, const float *wg, const float *logit_bias, int S, int E, int M,
                               int k, double capacity_factor, int normalize_gate, int alignment, int layout, float *scores,
                               int32_t *idx, int32_t *loc, float *gates, int32_t *row, int32_t *counts,
                               int32_t *kept_rows, int32_t *offsets, int32_t *capacity, float *l_aux, void *workspace,
                               size_t workspace_bytes, mole_stream_t stream) {
    return gate_route(x, dtype, wg, logit_bias, S, E, M, k, capacity_factor, normalize_gate, alignment, layout, scores, idx, loc, gates, row, counts,
                      kept_rows, offsets, capacity, l_aux, nullptr, workspace, workspace_bytes, stream);
}

extern "C" int mole_gate_fwd(const void *x, int dtype, const float *wg, const float *logit_bias, int S, int E, int M,
                             float *scores, mole_stream_t stream) {
    MOLE_REQUIRE(S >= 0 && E >= 1 &&
                     ((dtype == MOLE_BF16 && E <= 256 && M >= 128 && M % 128 == 0) || (dtype == MOLE_F32 && E <= 32 && M >= 4 && M % 4 == 0)),
                 "mole_gate_fwd: needs bf16 tokens with M a multiple of 128 and at most 256 experts, or fp32 tokens with M a "
                 "multiple of 4 and at most 32 experts (S=%d E=%d M=%d dtype=%d)", S, E, M, dtype);
    if (S == 0) return 0;
    MOLE_REQUIRE(x && wg && scores, "mole_gate_fwd: null pointer");
    hipStream_t st = (hipStream_t)stream;
    if (dtype == MOLE_F32) {
        MOLE_REQUIRE((((uintptr_t)x | (uintptr_t)wg) & 15) == 0, "mole_gate_fwd: x and wg must be 16-byte aligned");
        const dim3 grid4(ceil_div(S, 4));
        const float *xf = (const float *)x;
        if (E <= 8) timed_launch(MOLE_K_GATE_FWD, gate_fwd_f32_kernel<8>, grid4, dim3(256), 0, st, xf, wg, logit_bias, S, E, M, scores);
        else if (E <= 16) timed_launch(MOLE_K_GATE_FWD, gate_fwd_f32_kernel<16>, grid4, dim3(256), 0, st, xf, wg, logit_bias, S, E, M, scores);
        else timed_launch(MOLE_K_GATE_FWD, gate_fwd_f32_kernel<32>, grid4, dim3(256), 0, st, xf, wg, logit_bias, S, E, M, scores);
        MOLE_LAUNCH_CHECK();
        return 0;
    }
    const bf16_t *xb = (const bf16_t *)x;
    const int eg = ceil_div(E, 16);
    // small gates: 32 tokens per block (Wg, which every block reads in full, is then read half as often)
    const dim3 grid(ceil_div(S, eg <= 2 ? 32 : 16));
    // (16 experts or fewer: staged, 34 KB of LDS; 10.6 against 11.6 us straight from memory at 16384 x 1024, and 11.1
    // with the whole quarter row in one round of eight steps)
    const GateRoute none{};
    if (eg == 1) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<1, 4, 2, true>, grid, dim3(256), GATE_STAGE_LDS, st, xb, wg, logit_bias, S, E, M, scores, none);
    else if (eg == 2) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<2, 4, 2, false>, grid, dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    // (33-64 experts: Wg is 4 times as large, so more tokens share a block's pass over it: 8192 x 2048 x 64: 35.6 us
    // with 16 tokens per block, 22.5 with 32, 27.7 with 64 (128 blocks); 16384 x 1024 x 64: 35.5 / 23.6 / 18.5 us)
    else if (eg <= 4 && S >= 64 * 256) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<4, 4, 4, false>, dim3(ceil_div(S, 64)), dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    else if (eg <= 4 && S >= 32 * 128) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<4, 4, 2, false>, dim3(ceil_div(S, 32)), dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    else if (eg <= 4) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<4, 4, 1, false>, grid, dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    else if (eg <= 8) timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<8, 4, 1, false>, grid, dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    else timed_launch(MOLE_K_GATE_FWD, gate_fwd_kernel<16, 2, 1, false>, grid, dim3(256), 0, st, xb, wg, logit_bias, S, E, M, scores, none);
    MOLE_LAUNCH_CHECK();
    return 0;
}

extern "C" int mole_softmax_bwd(const float *dscores, const float *scores, int S, int E, float *dlogits,
                                mole_stream_t stream) {
    MOLE_REQUIRE(S >= 0 && E >= 1 && E <= MOLE_MAX_EXPERTS, "mole_softmax_bwd: bad sizes S=%d E=%d", S, E);
    if (S == 0) return 0;
    MOLE_REQUIRE(dscores && scores && dlogits, "mole_softmax_bwd: null pointer");
    int logG = 0;
    while ((1 << logG) < E && logG < 6) ++logG;
    const int vpl = ceil_div(E, 1 << logG);
    const int tpw = 64 >> logG;
    const dim3 grid(ceil_div(S, 4 * tpw));
    ScopedTiming timing(MOLE_K_GATE_BWD, (hipStream_t)stream);
    MOLE_VPL_DISPATCH(vpl, softmax_bwd_kernel, grid, (hipStream_t)stream, dscores, scores, S, E, logG, dlogits);
    MOLE_LAUNCH_CHECK();
    return 0;
}

extern "C" int mole_gate_bwd(const float *dgates, const float *scores, const int32_t *idx, int S, int E, int k,
                             int normalize_gate, int through_softmax, const int32_t *counts0, const float *d_l_aux,
                             float *dlogits, mole_stream_t stream) {
    MOLE_REQUIRE(S >= 0 && E >= 1 && E <= MOLE_MAX_EXPERTS && k >= 1 && k <= MOLE_MAX_TOPK && k <= E,
                 "mole_gate_bwd: bad sizes S=%d E=%d k=%d", S, E, k);
    if (S == 0) return 0;
    MOLE_REQUIRE(dgates && scores && idx && dlogits, "mole_gate_bwd: null pointer");
    MOLE_REQUIRE((counts0 == nullptr) == (d_l_aux == nullptr), "mole_gate_bwd: counts0 and d_l_aux go together");
    int logG = 0;
    while ((1 << logG) < E && logG < 6) ++logG;
    const int vpl = ceil_div(E, 1 << logG);
    const int tpw = 64 >> logG;
    const dim3 grid(ceil_div(S, 4 * tpw));
    ScopedTiming timing(MOLE_K_GATE_BWD, (hipStream_t)stream);
    MOLE_VPL_DISPATCH(vpl, gate_bwd_kernel, grid, (hipStream_t)stream, dgates, scores, idx, S, E, k, logG,
                      normalize_gate, through_softmax, counts0, d_l_aux, dlogits);
    MOLE_LAUNCH_CHECK();
    return 0;
}
