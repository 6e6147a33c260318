// Weight-gradient tiles of experts with few rows, inside the large-tile kernels (gemm256.hip): C_e[M, N] = sum over the
// expert's rows r of A[r, M]^T . B[r, N], up to 64 rows.
//
// Such a tile is one or two matrix instructions deep; what it costs is its results' way to memory (bound: a stream of stores, 5.8
// TB/s).  By way of the operand ring and the LDS slabs of the large tiles a block of one stage spends 6.5 us, most of it waits and
// barriers one after the other, on the storing of 128 KB.  Here a wave is on its own: operands come straight from memory into fragments,
// results leave straight from the accumulators, and there is no LDS and no barrier.  By way of the ring / here, us a launch: 64 experts
// of 1024 x 2048, 16 rows (268 MB), 70.5 / 58, added to 111 / 91; 16 of 1024 x 4096, 4 rows, 35 / 27 and 58 / 47; 200 of 384 x 768, 16
// rows, 32 / 25 and 51 / 43; 64 of 2048 x 8192, 32 rows, 546 / 501.
//
// Neither operand is contiguous along the rows that are summed over.  A lane loads V consecutive columns (16, 8 or 4 bytes) of the
// eight rows 8 kg .. 8 kg + 7 (kg = lane / 16) of a step of 32 and turns the 8 x V block in registers; fragment j then holds column
// V i + j for lane i of 16.  The m-side (VM columns) feeds the instruction's first slot, so that a lane ends up with VN consecutive
// columns of row VM (4 kg + r) + j in the VN products of m-fragment j: with VN = 8 a store writes whole 256-byte pieces of four rows
// (128-byte pieces, VN = 4: 440 -> 530 us for 2.1 GB).
// The first 32 rows are summed first and the rest follows; the large tiles begin with what whole stages of 32 leave over, so with 33 to 63 rows their
// results may be the neighbouring ones.
#pragma once
#include "gemm.h"

namespace mole {

// eight rows of V columns; rows past the expert's last one repeat it and are cleared when they are turned
template <int V> struct FewRows {
    uint32_t w[8][V / 2];
    __device__ __forceinline__ void fetch(const bf16_t *col, long ld, int k0, int rows) {
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const bf16_t *p = col + (long)min(k0 + u, rows - 1) * ld;
            if constexpr (V == 8) {
                const uint4 v = *reinterpret_cast<const uint4 *>(p);
                w[u][0] = v.x; w[u][1] = v.y; w[u][2] = v.z; w[u][3] = v.w;
            } else if constexpr (V == 4) {
                const uint2 v = *reinterpret_cast<const uint2 *>(p);
                w[u][0] = v.x; w[u][1] = v.y;
            } else {
                w[u][0] = *reinterpret_cast<const uint32_t *>(p);
            }
        }
    }
    // f[j] = the eight rows' values of column j
    __device__ __forceinline__ void turn(int k0, int rows, bool partial, bf16x8 (&f)[V]) {
        if (partial) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const uint32_t keep = k0 + u < rows ? 0xffffffffu : 0u;
#pragma unroll
                for (int c = 0; c < V / 2; ++c) w[u][c] &= keep;
            }
        }
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;
            const int c = j >> 1;
            f[j] = __builtin_bit_cast(bf16x8, make_uint4(__builtin_amdgcn_perm(w[1][c], w[0][c], sel), __builtin_amdgcn_perm(w[3][c], w[2][c], sel),
                                                         __builtin_amdgcn_perm(w[5][c], w[4][c], sel), __builtin_amdgcn_perm(w[7][c], w[6][c], sel)));
        }
    }
};

// The sums of a wave's columns.  side 2: sums[c] holds column n0 + V i + c in every register of lane i; side 1: register r of a lane
// of group kg holds column m0 + V (4 kg + r) + c.
template <int V, int SIDE, bool ACC> __device__ __forceinline__ void few_store_sums(const f32x4 (&sums)[V], bf16_t *out, int first, int ext) {
    const int lane = threadIdx.x & 63, i = lane & 15, kg = lane >> 4;
    constexpr int R = SIDE == 1 ? 4 : 1;
    const bool mine = SIDE == 1 ? i == 0 : kg == 0;
    float old[V][R];
    auto at = [&](int c, int r) { return first + (SIDE == 1 ? V * (4 * kg + r) : V * i) + c; };
#pragma unroll
    for (int c = 0; c < V; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r) old[c][r] = ACC ? (float)out[min(at(c, r), ext - 1)] : 0.f;
#pragma unroll
    for (int c = 0; c < V; ++c)
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (mine && at(c, r) < ext) out[at(c, r)] = (bf16_t)(ACC ? sums[c][r] + old[c][r] : sums[c][r]);
}

// The 16 VM x 16 VN results at (m0, n0) of an expert with 1 .. 32 KS rows.  C: the expert's matrix; sums: where this wave puts the sums
// of its m-side (side 1) or n-side (side 2) columns.
template <int VM, int VN, int KS, bool ACC>
__device__ __forceinline__ void few_rows_tile(const GemmArgs &g, const bf16_t *Ap, const bf16_t *Bp, bf16_t *C, bf16_t *colsum, int side, int m0, int n0, int rows) {
    typedef uint32_t piece_t __attribute__((ext_vector_type(VN / 2)));
    typedef __attribute__((address_space(1))) char gchar;
    typedef __attribute__((address_space(1))) piece_t gpiece;
    const int lane = threadIdx.x & 63, i = lane & 15, kg = lane >> 4;
    if (m0 >= g.M || n0 >= g.N) return;
    const bf16_t *ac = Ap + min(m0 + VM * i, g.M - VM), *bc = Bp + min(n0 + VN * i, g.N - VN);
    FewRows<VM> qa[KS];
    FewRows<VN> qb[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qb[s].fetch(bc, g.ldb, 32 * s + 8 * kg, rows);
        qa[s].fetch(ac, g.lda, 32 * s + 8 * kg, rows);
    }
    // this lane's VN columns of row VM r + j: a wave-uniform base and a 32-bit offset of the lane's
    const uint32_t pitch = (uint32_t)g.ldc * 2;
    gchar *const base = (gchar *)((char *)C + ((long)m0 * g.ldc + n0) * 2);
    const uint32_t lane_off = (uint32_t)(4 * VM * kg) * pitch + (uint32_t)(VN * i) * 2;
    const int rows_left = n0 + VN * i < g.N ? g.M - m0 - 4 * VM * kg : 0;
    auto at = [&](int row) { return reinterpret_cast<gpiece *>(base + (size_t)row * pitch + lane_off); };
    piece_t old[VM][4];
    if constexpr (ACC) {
        // (rows past the end: the tile's first, which exists; columns past the end: the tile's first)
        const uint32_t safe = n0 + VN * i < g.N ? lane_off : (uint32_t)(4 * VM * kg) * pitch;
#pragma unroll
        for (int j = 0; j < VM; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool in = VM * r + j < g.M - m0 - 4 * VM * kg;
                old[j][r] = __builtin_nontemporal_load(reinterpret_cast<const gpiece *>(in ? base + (size_t)(VM * r + j) * pitch + safe : base));
            }
    }
    __builtin_amdgcn_sched_barrier(0);           // all loads first
    bf16x8 fa[KS][VM], fb[KS][VN];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        qb[s].turn(32 * s + 8 * kg, rows, 32 * (s + 1) > rows, fb[s]);
        qa[s].turn(32 * s + 8 * kg, rows, 32 * (s + 1) > rows, fa[s]);
    }
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    if (side != 0) {
        const bf16_t one = (bf16_t)1.0f;
        const bf16x8 ones = {one, one, one, one, one, one, one, one};
        if (side == 1) {
            f32x4 sums[VM];
#pragma unroll
            for (int c = 0; c < VM; ++c) {
                sums[c] = zero;
#pragma unroll
                for (int s = 0; s < KS; ++s) sums[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[s][c], ones, sums[c], 0, 0, 0);
            }
            few_store_sums<VM, 1, ACC>(sums, colsum, m0, g.M);
        } else {
            f32x4 sums[VN];
#pragma unroll
            for (int c = 0; c < VN; ++c) {
                sums[c] = zero;
#pragma unroll
                for (int s = 0; s < KS; ++s) sums[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, fb[s][c], sums[c], 0, 0, 0);
            }
            few_store_sums<VN, 2, ACC>(sums, colsum, n0, g.N);
        }
    }
#pragma unroll
    for (int j = 0; j < VM; ++j) {
        f32x4 acc[VN];
#pragma unroll
        for (int c = 0; c < VN; ++c) {
            acc[c] = zero;
#pragma unroll
            for (int s = 0; s < KS; ++s) acc[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[s][j], fb[s][c], acc[c], 0, 0, 0);
        }
        // (nothing of this launch reads them again: non-temporal, as on the large tiles)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            piece_t p;
#pragma unroll
            for (int c = 0; c < VN / 2; ++c) {
                float lo = acc[2 * c][r], hi = acc[2 * c + 1][r];
                if constexpr (ACC) {
                    lo += __uint_as_float(old[j][r][c] << 16);
                    hi += __uint_as_float(old[j][r][c] & 0xffff0000u);
                }
                const bf16_t b0 = (bf16_t)lo, b1 = (bf16_t)hi;
                p[c] = (uint32_t)__builtin_bit_cast(uint16_t, b0) | ((uint32_t)__builtin_bit_cast(uint16_t, b1) << 16);
            }
            if (VM * r + j < rows_left) __builtin_nontemporal_store(p, at(VM * r + j));
        }
    }
}

}  // namespace mole
