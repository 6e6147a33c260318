// Row-ragged products of experts with few rows (decode batches, short training batches): the expert's weights are
// read once, straight from memory into MFMA fragments, and everything else is arranged around keeping those loads
// in flight.
//
// With a handful of rows per expert a product is a stream over its weights (2 x 16.8 MB for an expert of 2048 x 8192),
// and the big-tile kernels have too few blocks to pull it: a contraction over 8192 with 2048 result columns is 8 tiles
// of 256 columns per active expert, each a serial walk over 8192 of K by one CU (about 60 GB/s a CU).  Here the waves of
// a block split the contraction, and blocks split it further (ksplit) where the result is too narrow to give every CU a
// block; partial results meet in LDS, or as fp32 planes in a workspace that plane_reduce_kernel adds up in plane order
// (deterministic, no atomics).
//
// Tokens take the MFMA's B side (16 rows), weights its A side (16 result columns), so a lane ends up with 4 consecutive
// columns of one row.  A lane supplies EPC = 16 bytes worth of consecutive k (8 bf16: one 16x16x32 MFMA; 4 fp32: four
// 16x16x4 MFMAs, one per component), lane group l / 16 the k-run l / 16 of a 64-byte step.
//   KC  (weights [N][K], h = xd.w1^T and t = go.w2^T): a 16-byte load per lane is a fragment as it comes.
//   KS  (weights [K][N], out = a.w2 and gx = t.w1): a lane loads EPC rows of EPC consecutive columns and transposes
//       the EPC x EPC block in registers (bf16: byte permutes; fp32: a renaming); fragment j is then column EPC i + j
//       of the tile's 16 EPC columns for lane i, and a row's results are EPC consecutive columns per lane.
// No LDS on the way in, no barrier before the partial sums meet.
#include "gemm.h"

namespace mole {

typedef float sk_f32x4 __attribute__((ext_vector_type(4)));

constexpr int SK_WAVES = 8, SK_THREADS = 64 * SK_WAVES;
static_assert(HEAD_PAIRS <= SK_THREADS, "a thread per pair");

template <typename T> struct SkElem;
template <> struct SkElem<bf16_t> { static constexpr int EPC = 8; };
template <> struct SkElem<float> { static constexpr int EPC = 4; };

template <typename T> __device__ __forceinline__ sk_f32x4 sk_mma(uint4 w, uint4 x, sk_f32x4 acc) {
    if constexpr (sizeof(T) == 2) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), acc, 0, 0, 0);
    } else {
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.x), __uint_as_float(x.x), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.y), __uint_as_float(x.y), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.z), __uint_as_float(x.z), acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w.w), __uint_as_float(x.w), acc, 0, 0, 0);
    }
}

__device__ __forceinline__ void sk_mask(uint4 &v, uint32_t keep) {
    v = make_uint4(v.x & keep, v.y & keep, v.z & keep, v.w & keep);
}

// q[kk] = EPC consecutive columns of k-row kk; f[j] = the EPC k of column j
__device__ __forceinline__ void sk_transpose(const uint4 (&q)[8], uint4 (&f)[8]) {
    const uint32_t w[8][4] = {{q[0].x, q[0].y, q[0].z, q[0].w}, {q[1].x, q[1].y, q[1].z, q[1].w},
                              {q[2].x, q[2].y, q[2].z, q[2].w}, {q[3].x, q[3].y, q[3].z, q[3].w},
                              {q[4].x, q[4].y, q[4].z, q[4].w}, {q[5].x, q[5].y, q[5].z, q[5].w},
                              {q[6].x, q[6].y, q[6].z, q[6].w}, {q[7].x, q[7].y, q[7].z, q[7].w}};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
        f[j] = make_uint4(__builtin_amdgcn_perm(w[1][j >> 1], w[0][j >> 1], sel), __builtin_amdgcn_perm(w[3][j >> 1], w[2][j >> 1], sel),
                          __builtin_amdgcn_perm(w[5][j >> 1], w[4][j >> 1], sel), __builtin_amdgcn_perm(w[7][j >> 1], w[6][j >> 1], sel));
    }
}
__device__ __forceinline__ void sk_transpose(const uint4 (&q)[4], uint4 (&f)[4]) {
    f[0] = make_uint4(q[0].x, q[1].x, q[2].x, q[3].x);
    f[1] = make_uint4(q[0].y, q[1].y, q[2].y, q[3].y);
    f[2] = make_uint4(q[0].z, q[1].z, q[2].z, q[3].z);
    f[3] = make_uint4(q[0].w, q[1].w, q[2].w, q[3].w);
}

// The `target`-th group of at most RG rows, counted over the experts in order: its expert, its number within the expert,
// the expert's rows and first row.  Every wave looks it up for itself (rows and offsets of 256 experts per pass come in
// one go); false when there are fewer groups.
template <int RG>
__device__ __forceinline__ bool sk_find_group(const GemmArgs &g, int target, int &e, int &grp, int &rows, long &row0) {
    const int lane = threadIdx.x & 63;
    int run = 0;
    for (int base = 0; base < g.E; base += 4 * WAVE) {
        int r[4], o[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const int ee = min(base + c * WAVE + lane, g.E - 1);
            r[c] = g.kept[ee];
            o[c] = g.offsets[ee];
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (base + c * WAVE >= g.E) break;
            const int cnt = base + c * WAVE + lane < g.E ? (r[c] + RG - 1) / RG : 0;
            const int incl = wave_scan(cnt);
            const unsigned long long hit = __ballot(run + incl > target);
            if (hit) {
                const int src = __ffsll(hit) - 1;
                e = __builtin_amdgcn_readfirstlane(base + c * WAVE + src);
                grp = target - (run + __builtin_amdgcn_readlane(incl - cnt, src));
                rows = __builtin_amdgcn_readlane(r[c], src);
                row0 = __builtin_amdgcn_readlane(o[c], src);
                return true;
            }
            run += wave_total(incl);
        }
    }
    return false;
}

template <typename T> __device__ __forceinline__ void sk_store4(T *p, const float (&v)[4]) {
    if constexpr (sizeof(T) == 2) {
        typedef __bf16 bf16x4_ __attribute__((ext_vector_type(4)));
        *reinterpret_cast<uint2 *>(p) = __builtin_bit_cast(uint2, bf16x4_{(bf16_t)v[0], (bf16_t)v[1], (bf16_t)v[2], (bf16_t)v[3]});
    } else {
        *reinterpret_cast<float4 *>(p) = make_float4(v[0], v[1], v[2], v[3]);
    }
}
template <typename T> __device__ __forceinline__ void sk_load4(const T *p, float (&v)[4]) {
    if constexpr (sizeof(T) == 2) {
        const uint2 u = *reinterpret_cast<const uint2 *>(p);
        v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
        v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
    } else {
        const float4 u = *reinterpret_cast<const float4 *>(p);
        v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
    }
}

// 16 bytes of a weight.  ONCE: no other block reads them, so they leave no copy behind (non-temporal): a plain stream of
// 1 GB runs at 6.4 instead of 5.8 TB/s that way on this chip.  Only for KS, whose loads cover whole 128-byte lines: a KC
// load takes 64 bytes of a row and the next one the other half of the line, which a non-temporal load has let go of by
// then (123 experts of 448 -> 1344, fp32, 2 rows each: KS 59 -> 53 us, KC 57 -> 80).
template <bool ONCE> __device__ __forceinline__ uint4 sk_weight(const void *p) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    if constexpr (ONCE) {
        const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(p));
        return make_uint4(v[0], v[1], v[2], v[3]);
    } else {
        return *reinterpret_cast<const uint4 *>(p);
    }
}

// Four consecutive columns n .. n+3 (all inside the result: N is a multiple of 4) of row `row` of expert e.
template <typename T, int EPI>
__device__ __forceinline__ void sk_epilogue4(const GemmArgs &g, int e, long row, int n, float (&v)[4]) {
    if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) {
        float b[4];
        sk_load4<T>((const T *)g.bias + (long)e * g.N + n, b);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] += b[j];
    }
    const long at = row * g.ldc + n;
    const bool fitted = sizeof(T) == 2 && g.K % 32 == 0;      // (the fitted polynomials or the closed forms: see gemm.h)
    if constexpr (EPI == EPI_DGELU) {
        float h[4];
        sk_load4<T>((const T *)g.H + at, h);
        if (fitted) {
            DGeluCoef d;
            d.select(g.gelu_bwd == MOLE_GELU_BWD_TANH);
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] *= d(h[j]);
        } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] *= g.gelu_bwd == MOLE_GELU_BWD_TANH ? d_gelu_tanh(h[j]) : d_gelu_exact(h[j]);
        }
    }
    if constexpr (EPI == EPI_BIAS_GELU) {
        if (g.C != nullptr) sk_store4<T>((T *)g.C + at, v);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = fitted ? fast_gelu_erf(v[j]) : gelu_erf(v[j]);
        sk_store4<T>((T *)g.C2 + at, v);
    } else {
        sk_store4<T>((T *)g.C + at, v);
    }
}

// ---- weights [N][K] ---------------------------------------------------------------------------------------------
// A block owns 16 NA result columns of one group of up to 16 MB rows; its eight waves split the contraction.  A wave has the
// weights of two steps (2 NA loads of 1 KiB) in flight and waits for them before it asks for more: sixteen waves to a
// CU, out of step with each other, keep the memory busier than eight waves with two rounds in flight each (the
// registers allow one or the other; 256 experts of eight rows, 2048 -> 1024: 215 against 250 us, 1.07 GB of weights).  Two
// steps also with 32 columns, where four would keep as many loads in flight: what a wave's share lacks of them is loaded all the
// same (see launch_kc).
template <typename T, int MB, int NA, int EPI>
__device__ __forceinline__ void skinny_kc_run(const GemmArgs &g, sk_f32x4 (&red)[SK_WAVES][NA][WAVE], const int *token, int e,
                                              int rows, long row0, int m0, int n0) {
    constexpr int EPC = SkElem<T>::EPC, KSTEP = 4 * EPC, U = 2;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int steps = (g.K + KSTEP - 1) / KSTEP;
    const int s_lo = wave * steps / SK_WAVES, s_hi = (wave + 1) * steps / SK_WAVES;
    const T *wp[NA], *xp[MB];
#pragma unroll
    for (int a = 0; a < NA; ++a) wp[a] = (const T *)g.B + (long)e * g.strideB + (long)min(n0 + 16 * a + i16, g.N - 1) * g.ldb;
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int m = min(m0 + 16 * b + i16, rows - 1);
        xp[b] = (const T *)g.A + (EPI == EPI_BIAS_GELU && g.pair_row != nullptr ? (long)min((unsigned)token[m - m0], (unsigned)g.tokens - 1u) : row0 + m) * g.lda;
    }
    sk_f32x4 acc[NA][MB];
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[a][b] = sk_f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 w[U][NA], x[U][MB];
    // (steps past the wave's share repeat its last one and are not multiplied; of a step that the contraction ends in, the lanes
    // past its end are masked on both sides: a weight that is no number times zero would be none)
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = min(min(s + u, s_hi - 1) * KSTEP + kg * EPC, g.K - EPC);
#pragma unroll
            for (int a = 0; a < NA; ++a) w[u][a] = *reinterpret_cast<const uint4 *>(wp[a] + k);
#pragma unroll
            for (int b = 0; b < MB; ++b) x[u][b] = *reinterpret_cast<const uint4 *>(xp[b] + k);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    auto use = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (s + u >= s_hi) break;
            if ((s + u + 1) * KSTEP > g.K) {
                const uint32_t keep = (s + u) * KSTEP + kg * EPC < g.K ? 0xffffffffu : 0u;
#pragma unroll
                for (int a = 0; a < NA; ++a) sk_mask(w[u][a], keep);
#pragma unroll
                for (int b = 0; b < MB; ++b) sk_mask(x[u][b], keep);
            }
#pragma unroll
            for (int b = 0; b < MB; ++b)
#pragma unroll
                for (int a = 0; a < NA; ++a) acc[a][b] = sk_mma<T>(w[u][a], x[u][b], acc[a][b]);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int s = s_lo; s < s_hi; s += U) {
        fetch(s);
        use(s);
    }
    // per 16-row block the waves' partial tiles meet in LDS; wave a adds up 16-column cell a in wave order
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        if (b > 0) __syncthreads();
#pragma unroll
        for (int a = 0; a < NA; ++a) red[wave][a][lane] = acc[a][b];
        __syncthreads();
        const int m = m0 + 16 * b + i16, n = n0 + 16 * wave + 4 * kg;
        if (wave < NA && m < rows && n < g.N) {
            sk_f32x4 s = red[0][wave][lane];
#pragma unroll
            for (int q = 1; q < SK_WAVES; ++q) s += red[q][wave][lane];
            float v[4] = {s[0], s[1], s[2], s[3]};
            sk_epilogue4<T, EPI>(g, e, row0 + m, n, v);
        }
    }
}

// MB: 16-row blocks of a group; a group with fewer live ones runs the code for those.  With g.pair_row every block finds the tokens
// of its rows for itself, a pair per thread: the pairs' rows arrive while the block looks its group up, where a launch in front of
// this one is 2 us of latency for a few kilobytes.  Passes with a dispatch / without: 1 token, 64 experts of 2048 -> 8192, 47.9 /
// 45.7 us; 8 tokens, 8 of 1024 -> 4096, 37.4 / 35.5; 256 tokens top-2, 32 of 512 -> 1024, 512 pairs, 39.7 / 37.6; fp32, 1 token, 8 of
// 1024 -> 4096, 28.9 / 26.3, 128 tokens top-2, 32 of 512 -> 1024, 49.8 / 48.1.
template <typename T, int MB, int NA, int EPI>
__global__ __launch_bounds__(SK_THREADS, 4) void skinny_kc_kernel(const GemmArgs g) {
    __shared__ __align__(16) sk_f32x4 red[SK_WAVES][NA][WAVE];
    __shared__ int token[16 * MB];
    const int chunks = (g.N + 16 * NA - 1) / (16 * NA);
    int e, grp, rows;
    long row0;
    int pair = -1;
    if constexpr (EPI == EPI_BIAS_GELU)
        if (g.pair_row != nullptr && threadIdx.x < (unsigned)g.pairs) pair = g.pair_row[threadIdx.x];
    if (!sk_find_group<16 * MB>(g, blockIdx.x / chunks, e, grp, rows, row0)) return;
    if constexpr (EPI == EPI_BIAS_GELU) {
        if (g.pair_row != nullptr) {
            const long r = pair - (row0 + grp * (16 * MB));
            if (pair >= 0 && r >= 0 && r < 16 * MB) token[r] = threadIdx.x % (unsigned)g.tokens;
            __syncthreads();
        }
    }
    const int n0 = (blockIdx.x % chunks) * (16 * NA), m0 = grp * (16 * MB), live = rows - m0;
    if (MB == 1 || live <= 16) skinny_kc_run<T, 1, NA, EPI>(g, red, token, e, rows, row0, m0, n0);
    else skinny_kc_run<T, MB, NA, EPI>(g, red, token, e, rows, row0, m0, n0);
}

// ---- weights [K][N] ---------------------------------------------------------------------------------------------
// A block owns 16 EPC result columns (256 bytes of a weight row) of one group of up to 16 MB rows and 1 / ksplit of the
// contraction, which its eight waves split again; a wave has the weights of one step (EPC loads of 1 KiB) in flight.
template <typename T, int MB, bool ONCE, int EPI>
__device__ __forceinline__ void skinny_ks_run(const GemmArgs &g, sk_f32x4 (&red)[SK_WAVES][SkElem<T>::EPC][WAVE], int e, int rows,
                                              long row0, int m0, int n0, int split) {
    constexpr int EPC = SkElem<T>::EPC, KSTEP = 4 * EPC;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i16 = lane & 15, kg = lane >> 4;
    const int steps = (g.K + KSTEP - 1) / KSTEP, parts = g.ksplit * SK_WAVES, part = split * SK_WAVES + wave;
    const int s_lo = (int)((long)part * steps / parts), s_hi = (int)((long)(part + 1) * steps / parts);
    const T *wp = (const T *)g.B + (long)e * g.strideB + min(n0 + i16 * EPC, g.N - EPC);
    const T *xp[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) xp[b] = (const T *)g.A + (row0 + min(m0 + 16 * b + i16, rows - 1)) * g.lda;
    sk_f32x4 acc[EPC][MB];
#pragma unroll
    for (int j = 0; j < EPC; ++j)
#pragma unroll
        for (int b = 0; b < MB; ++b) acc[j][b] = sk_f32x4{0.f, 0.f, 0.f, 0.f};
    uint4 w[EPC], x[MB];
    auto fetch = [&](int s) __attribute__((always_inline)) {
        const int k = min(s * KSTEP + kg * EPC, g.K - EPC);
        const T *wk = wp + (long)k * g.ldb;
#pragma unroll
        for (int q = 0; q < EPC; ++q) w[q] = sk_weight<ONCE>(wk + (long)q * g.ldb);
#pragma unroll
        for (int b = 0; b < MB; ++b) x[b] = *reinterpret_cast<const uint4 *>(xp[b] + k);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto use = [&](int s) __attribute__((always_inline)) {
        if ((s + 1) * KSTEP > g.K) {       // the step that the contraction ends in: as for the other layout
            const uint32_t keep = s * KSTEP + kg * EPC < g.K ? 0xffffffffu : 0u;
#pragma unroll
            for (int q = 0; q < EPC; ++q) sk_mask(w[q], keep);
#pragma unroll
            for (int b = 0; b < MB; ++b) sk_mask(x[b], keep);
        }
        uint4 f[EPC];
        sk_transpose(w, f);
#pragma unroll
        for (int b = 0; b < MB; ++b)
#pragma unroll
            for (int j = 0; j < EPC; ++j) acc[j][b] = sk_mma<T>(f[j], x[b], acc[j][b]);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int s = s_lo; s < s_hi; ++s) {
        fetch(s);
        use(s);
    }
    // acc[j][b][r] of lane (i16, kg) is row m0 + 16 b + i16, column n0 + EPC (4 kg + r) + j.  Per 16-row block the waves'
    // partial tiles meet in LDS; a thread adds up four consecutive columns (j = 4 q .. 4 q + 3) of one lane and r.
    constexpr int QJ = EPC / 4;          // quadruples of columns per (lane, r)
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        if (b > 0) __syncthreads();
#pragma unroll
        for (int j = 0; j < EPC; ++j) red[wave][j][lane] = acc[j][b];
        __syncthreads();
        const int r = wave & 3;
        const int m = m0 + 16 * b + i16;
        if (wave < 4 * QJ && m < rows) {
            const int q = wave >> 2;
            const int n = n0 + EPC * (4 * kg + r) + 4 * q;
            if (n < g.N) {
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float s = red[0][4 * q + j][lane][r];
#pragma unroll
                    for (int ww = 1; ww < SK_WAVES; ++ww) s += red[ww][4 * q + j][lane][r];
                    v[j] = s;
                }
                if (g.ksplit == 1) {
                    sk_epilogue4<T, EPI>(g, e, row0 + m, n, v);
                } else {
                    *reinterpret_cast<float4 *>(g.part + ((long)split * g.part_rows + row0 + m) * g.N + n) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
    }
}

template <typename T, int MB, int EPI>
__global__ __launch_bounds__(SK_THREADS, 4) void skinny_ks_kernel(const GemmArgs g) {
    constexpr int BN = 16 * SkElem<T>::EPC;
    __shared__ __align__(16) sk_f32x4 red[SK_WAVES][SkElem<T>::EPC][WAVE];
    const int chunks = (g.N + BN - 1) / BN;
    int e, grp, rows;
    long row0;
    const int per_group = chunks * g.ksplit;
    if (!sk_find_group<16 * MB>(g, blockIdx.x / per_group, e, grp, rows, row0)) return;
    const int in_group = blockIdx.x % per_group;
    const int n0 = (in_group % chunks) * BN, split = in_group / chunks, m0 = grp * (16 * MB), live = rows - m0;
    if (rows <= 16 && g.once) skinny_ks_run<T, 1, true, EPI>(g, red, e, rows, row0, m0, n0, split);
    else if (MB == 1 || live <= 16) skinny_ks_run<T, 1, false, EPI>(g, red, e, rows, row0, m0, n0, split);
    else skinny_ks_run<T, MB, false, EPI>(g, red, e, rows, row0, m0, n0, split);
}

// out[row][n] = bias[n] + sum over the planes of part[plane][row][n], for the rows of the launch's experts
// only: the rows between them belong to experts of other launches (offloaded experts run in chunks).
constexpr int RED_ROWS = 4;
template <typename T>
__global__ __launch_bounds__(256) void plane_reduce_kernel(const GemmArgs g) {
    int e, grp, rows;
    long row0;
    const int chunks = (g.N + 1023) / 1024;
    if (!sk_find_group<RED_ROWS>(g, blockIdx.x / chunks, e, grp, rows, row0)) return;
    const int n = (blockIdx.x % chunks * 256 + threadIdx.x) * 4;
    if (n >= g.N) return;
    const long plane = g.part_rows * g.N;
    const int m0 = grp * RED_ROWS;
    float4 s[RED_ROWS];
    const float *p[RED_ROWS];
#pragma unroll
    for (int i = 0; i < RED_ROWS; ++i) {            // (rows past the expert's end repeat its last one and are not stored)
        p[i] = g.part + (row0 + min(m0 + i, rows - 1)) * g.N + n;
        s[i] = *reinterpret_cast<const float4 *>(p[i]);
    }
    // five planes' loads in flight (with one, 16 planes are 16 round trips to memory: 2 rows of 2048 took 7.9 us)
    constexpr int PF = 5;
    for (int k = 1; k < g.ksplit; k += PF) {
        float4 t[PF][RED_ROWS];
#pragma unroll
        for (int j = 0; j < PF; ++j)                // (planes past the last repeat it and are not added)
#pragma unroll
            for (int i = 0; i < RED_ROWS; ++i) t[j][i] = *reinterpret_cast<const float4 *>(p[i] + (long)min(k + j, g.ksplit - 1) * plane);
#pragma unroll
        for (int j = 0; j < PF; ++j)
            if (k + j < g.ksplit)
#pragma unroll
                for (int i = 0; i < RED_ROWS; ++i) { s[i].x += t[j][i].x; s[i].y += t[j][i].y; s[i].z += t[j][i].z; s[i].w += t[j][i].w; }
    }
    float b[4] = {0.f, 0.f, 0.f, 0.f};
    if (g.bias != nullptr) sk_load4<T>((const T *)g.bias + (long)e * g.N + n, b);
#pragma unroll
    for (int i = 0; i < RED_ROWS; ++i) {
        float v[4] = {s[i].x + b[0], s[i].y + b[1], s[i].z + b[2], s[i].w + b[3]};
        if (m0 + i < rows) sk_store4<T>((T *)g.C + (row0 + m0 + i) * g.ldc + n, v);
    }
}

// The same with the combine behind it: y[i] = sum over the k choices of gate x out, a block per token and 1024 columns.  Every kept
// row belongs to one token and choice, so the planes are read once as above; out - rounded to T first, as the combine reads
// it - need not pass through memory (keep_out: a backward pass reads it) and the combine needs no launch.  Bound by the planes'
// bytes, for few tokens by latency.  Forward passes of 1 token (64 experts of 2048 -> 8192) 51.4 -> 48.2 us, 61 tokens (16 of
// 1024 -> 4096) 72.8 -> 70.0, 3001 tokens 180.5 -> 173, 777 tokens in fp32 (8 of 512 -> 2048) 95.2 -> 92.1.
template <typename T, int K>
__global__ __launch_bounds__(256) void combine_planes_kernel(const float *__restrict__ part, int ksplit, long plane, const T *__restrict__ bias,
                                                             const int32_t *__restrict__ row, const int32_t *__restrict__ idx,
                                                             const float *__restrict__ gates, int S, int N, int k, T *__restrict__ out,
                                                             T *__restrict__ y) {
    const int cols = blockDim.x * 4, chunks = (N + cols - 1) / cols;
    const int i = blockIdx.x / chunks, n = (blockIdx.x % chunks * blockDim.x + threadIdx.x) * 4;
    int r[K], e[K];
    float gt[K];
    uint32_t keep[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const size_t at = (size_t)min(j, k - 1) * S + i;
        r[j] = row[at];
        e[j] = idx[at];
        gt[j] = gates[at];
    }
    if (n >= N) return;
    const float *p[K];
#pragma unroll
    for (int j = 0; j < K; ++j) {              // (a dropped pair reads row 0, and a choice past k the last one; neither counts)
        keep[j] = j < k && r[j] >= 0 ? 0xffffffffu : 0u;
        r[j] &= (int)keep[j];
        p[j] = part + (long)r[j] * N + n;
    }
    float4 s[K];
    float b[K][4];
#pragma unroll
    for (int j = 0; j < K; ++j) s[j] = *reinterpret_cast<const float4 *>(p[j]);
#pragma unroll
    for (int j = 0; j < K; ++j) sk_load4<T>(bias + (long)e[j] * N + n, b[j]);
    constexpr int PF = K >= 8 ? 1 : K == 4 ? 3 : 5;      // planes in flight
    for (int q = 1; q < ksplit; q += PF) {
        float4 t[PF][K];
#pragma unroll
        for (int u = 0; u < PF; ++u)
#pragma unroll
            for (int j = 0; j < K; ++j) t[u][j] = *reinterpret_cast<const float4 *>(p[j] + (long)min(q + u, ksplit - 1) * plane);
#pragma unroll
        for (int u = 0; u < PF; ++u)
            if (q + u < ksplit)
#pragma unroll
                for (int j = 0; j < K; ++j) { s[j].x += t[u][j].x; s[j].y += t[u][j].y; s[j].z += t[u][j].z; s[j].w += t[u][j].w; }
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < K; ++j) {
        const float v[4] = {s[j].x + b[j][0], s[j].y + b[j][1], s[j].z + b[j][2], s[j].w + b[j][3]};
        if (out != nullptr && keep[j]) sk_store4<T>(out + (long)r[j] * N + n, v);
        const float gj = __uint_as_float(__float_as_uint(gt[j]) & keep[j]);
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] += gj * __uint_as_float(__float_as_uint(to_f32(from_f32<T>(v[c]))) & keep[j]);
    }
    sk_store4<T>(y + (long)i * N + n, acc);
}

template <typename T>
static int launch_combine_planes(const GemmArgs &g, CombineTail &c, hipStream_t st) {
    const int threads = g.N >= 1024 ? 256 : ceil_div(g.N, 256) * 64;
    const dim3 grid((unsigned)c.S * (unsigned)ceil_div(g.N, threads * 4)), block(threads);
    T *out = c.keep_out ? (T *)g.C : nullptr;
#define MOLE_COMBINE_PLANES(K)                                                                                                    \
    timed_launch(MOLE_K_COMBINE_FWD, combine_planes_kernel<T, K>, grid, block, 0, st, (const float *)g.part, g.ksplit, g.part_rows * g.N, \
                 (const T *)g.bias, c.row, c.idx, c.gates, c.S, g.N, c.k, out, (T *)c.y)
    if (c.k <= 1) MOLE_COMBINE_PLANES(1);
    else if (c.k <= 2) MOLE_COMBINE_PLANES(2);
    else if (c.k <= 4) MOLE_COMBINE_PLANES(4);
    else if (c.k <= 8) MOLE_COMBINE_PLANES(8);
    else MOLE_COMBINE_PLANES(16);
#undef MOLE_COMBINE_PLANES
    MOLE_LAUNCH_CHECK();
    c.done = true;
    return 0;
}

// ---- which products come here, and how they are cut ------------------------------------------------------------
// avg: rows of an expert if the rows spread evenly; tiles: blocks the big-tile kernel of the type would have; tiles_split:
// whether those can split the contraction as they would, or have no need to.
struct SkinnyPlan { int mb, ksplit; };
static bool skinny_plan(int dtype, bool b_ks, int E, int est_rows, int N, int K, bool tiles_split, SkinnyPlan &p) {
    if (est_rows <= 0) return false;
    const bool bf16 = dtype == MOLE_BF16;
    const int epc = bf16 ? 8 : 4;
    const int active = E < est_rows ? E : est_rows;
    const int avg = ceil_div(est_rows, active);
    // bf16: with a CU's worth of tiles or more (192 of 256) the 256-column tiles of gemm256.hip stream the weights as
    // fast or faster (16 experts of 1024 -> 4096, 61 rows: 27 against 30 us); with fewer they leave CUs without work
    // (2 rows of 64 experts, 2048 -> 8192: h 24 against 17.5 us, out 66 against 13).  KC stops at 24 rows per expert,
    // where the token loads, one per four weight loads and 16 rows, begin to cost (8 experts of 512 -> 2048, 600 rows:
    // 18 against 14 us).  KS, eight weight loads for every 16 rows, against tiles that split the contraction as well: with
    // fewer than 32 tiles up to 64 rows per expert, below 48 up to 24, beyond up to 12 (and up to 64 where no workspace lets the
    // tiles split).  Forward pass, weights in no cache, here / on tiles: 4 experts of 2048 -> 2048, 32 tiles, 20 / 40 / 60 rows
    // 53 / 71 / 77 against 54 / 68 / 73 us; 20 of 512 -> 2048, 40 tiles, 20 / 40 / 60 rows 59 / 62 / 67 against 56 / 56 / 61, under Zipf
    // loads 58 / 67 / 71 against 61 / 66 / 71; 32 of 768 -> 2304, 96 tiles, 9 / 16 / 40 / 60 rows 97 / 104 / 131 / 151 against 92 / 93 / 98 /
    // 105, Zipf 80 / 91 / 116 / 127 against 77 / 88 / 114 / 113; 24 of 520 -> 1416, 72 tiles, 9 / 16 / 40 rows 53 / 61 / 77 against 52 /
    // 54 / 61, Zipf 47 / 56 / 81 against 50 / 55 / 79.  (Weights in the caches: 2 of 2048 -> 8192, 16 tiles, 16 / 62 rows 55 / 60
    // against 64 / 74.)
    // fp32: the 64 x 128 tiles of gemm_f32.hip, with their planes, from 48 rows per expert on, where also evenly spread rows
    // need more than one group of 32 and the fuller experts of a skewed routing many, each reading the weights again
    // (16 experts of 1024 -> 4096, forward pass, tiles / here: 800 rows 190 / 225 us, skewed 295 / 318; 960 rows 302 / 329;
    // 640 rows here 204, skewed 277).  KC: 244 / 400 rows 69 / 84 against 75 / 78 us.
    bool takes;
    if (bf16) {
        const long tiles = (long)active * ceil_div(avg, 256) * ceil_div(N, 256);
        takes = tiles < 192 && avg <= (!b_ks ? 24 : tiles < 32 || !tiles_split ? 64 : tiles < 48 ? 24 : 12);
        // every group of 16 rows reads the expert's weights again, from memory where they are more than the 256 MB last-level
        // cache holds: there the tiles take what is more than one group (20 experts of 2264 -> 9056, 20 rows: out 304 us here
        // against 153, planes added)
        if (b_ks && avg > 16 && (size_t)active * N * K * sizeof(bf16_t) > (size_t)256 << 20) takes = false;
    } else {
        takes = avg <= (b_ks ? 48 : 20);
    }
    if (!takes) return false;
    // rows per group: KC shares a block's weight loads among 32 rows once experts hold more than eight; KS in bf16 has
    // eight accumulators per 16 rows and runs better on more waves (groups of 16 re-read the weights out of the caches)
    p.mb = b_ks ? (bf16 ? 1 : 2) : (avg > 8 ? 2 : 1);
    // KS: about two blocks of eight waves per CU, every wave with at least two steps
    const int blocks = active * ceil_div(avg, 16 * p.mb) * ceil_div(N, 16 * epc);
    int ks = b_ks ? ceil_div(512, blocks) : 1;
    const int most = ceil_div(K, 4 * epc) / (2 * SK_WAVES);
    if (ks > most) ks = most;
    if (ks > 16) ks = 16;
    p.ksplit = ks < 1 ? 1 : ks;
    return true;
}

static bool tiles_split(int dtype, int E, int max_rows, int est_rows, int N, int K, size_t ws_bytes) {
    if (dtype != MOLE_BF16) return true;
    const int ks = gemm256_ksplit(E, est_rows, N, K);
    return ks <= 1 || (planes_allowed(ks, max_rows, est_rows, N) == ks && ws_bytes >= (size_t)ks * max_rows * N * sizeof(float));
}

bool gemm_skinny_takes_tokens(int E, int max_rows, int est_rows, int N, int K, int dtype) {
    const int epc = dtype == MOLE_BF16 ? 8 : 4;
    SkinnyPlan p;
    return max_rows > 0 && N % epc == 0 && K % epc == 0 && skinny_plan(dtype, false, E, est_rows, N, K, true, p);
}

int gemm_skinny_ksplit(int E, int max_rows, int est_rows, int N, int K, int dtype) {
    SkinnyPlan p;
    return skinny_plan(dtype, true, E, est_rows, N, K, tiles_split(dtype, E, max_rows, est_rows, N, K, SIZE_MAX), p) ? p.ksplit : 0;
}

int launch_plane_reduce(const GemmArgs &g, int dtype, int max_rows, hipStream_t st) {
    if (g.tail != nullptr) return dtype == MOLE_BF16 ? launch_combine_planes<bf16_t>(g, *g.tail, st) : launch_combine_planes<float>(g, *g.tail, st);
    // (the row groups are counted in x: y ends at 65535 blocks, which 262144 rows of a narrow layer reach)
    const dim3 grid((unsigned)((g.E < max_rows ? g.E : max_rows) + max_rows / RED_ROWS) * (unsigned)ceil_div(g.N, 1024));
    if (dtype == MOLE_BF16) hipLaunchKernelGGL(plane_reduce_kernel<bf16_t>, grid, dim3(256), 0, st, g);
    else hipLaunchKernelGGL(plane_reduce_kernel<float>, grid, dim3(256), 0, st, g);
    MOLE_LAUNCH_CHECK();
    return 0;
}

template <typename T, int MB, int NA>
static int launch_kc_na(const GemmArgs &g, int epi, int groups, hipStream_t st, int kid) {
    const dim3 grid((unsigned)(groups * ceil_div(g.N, 16 * NA)));
    if (epi == EPI_BIAS_GELU) timed_launch(kid, skinny_kc_kernel<T, MB, NA, EPI_BIAS_GELU>, grid, dim3(SK_THREADS), 0, st, g);
    else if (epi == EPI_DGELU) timed_launch(kid, skinny_kc_kernel<T, MB, NA, EPI_DGELU>, grid, dim3(SK_THREADS), 0, st, g);
    else return -100;
    MOLE_LAUNCH_CHECK();
    return 0;
}
// 32 columns a block instead of 64: 46 registers and 16 KB of LDS, four blocks to a CU where 64 columns run three, and twice
// the blocks where those leave CUs without one.  What counts against them is that every block loads its tokens for half of the
// columns, which shows where a wave has so few steps that its last pair repeats one; there 64 columns keep the launches that fill
// the chip with them.  h alone, weights in no cache, experts of one to eight rows, us with 64 / 32 columns (64-column blocks):
//   bf16, K = 2048: 12.5 / 7.5 (32), 18.4 / 18.0 (256), 30.1 / 27.2 (512), 40.6 / 32.9 (640);  K = 512: 5.4 / 4.5 (32), 11.3 / 11.0
//   (512), 14.5 / 13.3 (640), 14.5 / 14.5 (704);  K = 768, 8 rows: 22.2 / 21.4 (640), 22.4 / 24.3 (704);  K = 128: 4.2 / 4.0 (32), 5.6 /
//   5.9 (384), 6.6 / 7.1 (512), 9.0 / 9.8 (704).
//   fp32, K = 1024: 11.9 / 7.4 (32), 32.3 / 28.8 (512), 56 / 50.5 (1024), 230 / 223 (4096);  K = 384, 8 rows: 22.8 / 21.3 (640), 30.6 /
//   32.3 (1024);  K = 128: 5.3 / 4.2 (32), 9.7 / 10.2 (512), 20.7 / 23.1 (1536).
// (With four steps of 32 columns in flight a share of fewer steps loads them all the same: K = 512, 12.1 us for 320 blocks of 64
// columns, 19.4 for 640.)  Not with groups of 32 rows, whose token loads double (24 tokens, 4 of 4096 -> 4096: 71 / 80 us, the pass).
template <typename T, int MB>
static int launch_kc(const GemmArgs &g, int epi, int groups, hipStream_t st, int kid) {
    if constexpr (MB == 1) {
        const int steps = ceil_div(g.K, SK_WAVES * 4 * SkElem<T>::EPC);      // a wave's
        const long blocks = (long)(g.E < g.est_rows ? g.E : g.est_rows) * ceil_div(g.N, 64);
        if (steps >= 4 || blocks < (steps >= 2 ? 641 : 512)) return launch_kc_na<T, MB, 2>(g, epi, groups, st, kid);
    }
    return launch_kc_na<T, MB, 4>(g, epi, groups, st, kid);
}

template <typename T, int MB>
static int launch_ks(const GemmArgs &g, int epi, int groups, int max_rows, hipStream_t st, int kid) {
    const dim3 grid((unsigned)(groups * ceil_div(g.N, 16 * SkElem<T>::EPC) * g.ksplit));
    if (epi == EPI_BIAS) timed_launch(kid, skinny_ks_kernel<T, MB, EPI_BIAS>, grid, dim3(SK_THREADS), 0, st, g);
    else if (epi == EPI_STORE) timed_launch(kid, skinny_ks_kernel<T, MB, EPI_STORE>, grid, dim3(SK_THREADS), 0, st, g);
    else return -100;
    MOLE_LAUNCH_CHECK();
    if (g.ksplit > 1) return launch_plane_reduce(g, sizeof(T) == 2 ? MOLE_BF16 : MOLE_F32, max_rows, st);
    return 0;
}

static bool plan_launch(const GemmArgs &g, int dtype, bool b_ks, int max_rows, void *ws, size_t ws_bytes, SkinnyPlan &p) {
    const int epc = dtype == MOLE_BF16 ? 8 : 4;
    if (max_rows <= 0 || g.offsets == nullptr || g.kept == nullptr || g.token_of != nullptr) return false;
    const bool split = !b_ks || tiles_split(dtype, g.E, max_rows, g.est_rows, g.N, g.K, ws != nullptr ? ws_bytes : 0);
    if (!skinny_plan(dtype, b_ks, g.E, g.est_rows, g.N, g.K, split, p)) return false;
    return !(g.K % epc || g.N % epc || g.lda % epc || g.ldb % epc || g.ldc % epc || g.strideB % epc);
}
bool gemm_skinny_takes(const GemmArgs &g, int dtype, bool b_ks, int max_rows, void *ws, size_t ws_bytes) {
    SkinnyPlan p;
    return plan_launch(g, dtype, b_ks, max_rows, ws, ws_bytes, p);
}

int launch_gemm_skinny(const GemmArgs &g0, int dtype, bool b_ks, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid) {
    GemmArgs g = g0;
    SkinnyPlan p;
    if (!plan_launch(g, dtype, b_ks, max_rows, ws, ws_bytes, p)) return -100;
    const int groups = (g.E < max_rows ? g.E : max_rows) + max_rows / (16 * p.mb);     // as many as max_rows rows can need
    g.ksplit = 1;
    p.ksplit = planes_allowed(p.ksplit, max_rows, g.est_rows, g.N);
    if (p.ksplit > 1 && ws != nullptr && ws_bytes >= (size_t)p.ksplit * max_rows * g.N * sizeof(float)) {
        g.ksplit = p.ksplit;
        g.part = (float *)ws;
        g.part_rows = max_rows;
    }
    if (dtype == MOLE_BF16) {
        if (b_ks) return launch_ks<bf16_t, 1>(g, epi, groups, max_rows, st, kid);
        return p.mb == 1 ? launch_kc<bf16_t, 1>(g, epi, groups, st, kid) : launch_kc<bf16_t, 2>(g, epi, groups, st, kid);
    }
    if (b_ks) return launch_ks<float, 2>(g, epi, groups, max_rows, st, kid);
    return p.mb == 1 ? launch_kc<float, 1>(g, epi, groups, st, kid) : launch_kc<float, 2>(g, epi, groups, st, kid);
}

}  // namespace mole
