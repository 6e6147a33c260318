// bf16 grouped GEMM for gfx950: the fast path of the six expert-FFN products.
//
// A block of 8 waves (2 wave rows x 4 wave columns, two waves per SIMD) owns a BM (m) x 256 (n) output tile, BM =
// 256 or up to 320; a wave covers BM/2 rows and 64 columns (BM/32 x 4 MFMA 16x16x32 blocks, fp32 accumulators).
// One block per CU.  Launches too small to give most CUs such a tile run 128 x 128 tiles of four waves, two blocks to a
// CU.  (A build with -DMOLE_TUNING also reads the launch orders that were measured against these and lost.)
// Operand tiles go from HBM/L2 straight into LDS (global_load_lds_dwordx4, no staging registers)
// through a ring of stages of 32 of K, several stages of loads in flight while one is consumed: with
// a single stage of look-ahead the loop ran at the memory latency, not at the MFMA rate.  One
// barrier per stage.  Each 16-byte piece is placed at a swizzled LDS position by choosing which
// global address the lane that owns the slot fetches:
//   * K-contiguous operand  -> LDS [row][4 x 16 B]; fragments read with ds_read_b128
//   * K-strided operand     -> LDS [k][rows x 2 B] as it lies in HBM; fragments read with
//                              ds_read_b64_tr_b16, the LDS transpose read
// The MFMA "A" slot is fed with the n-side operand and the "B" slot with the m-side operand, so the
// four consecutive accumulator rows a lane holds are four consecutive n; results leave through LDS
// as whole 128-byte rows.  A ragged m-tile runs only the 32-row blocks it has rows for.
#include "gemm.h"
#include "lds_dma.h"
#include "mole_hip_probe.h"
#include "wgrad_few.h"

#include <stdlib.h>

#include <type_traits>

namespace mole {

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

constexpr int Q_BK = 32;
// Rows of an expert up to which a weight-gradient tile goes by way of few_rows_tile: two steps of 32, whose fragments fit the registers
// beside the results' old values.  (Up to 32 / up to 64: 8 experts of 2048 x 4096, 48 rows, 35.4 / 30.1 us; 64 of 1024 x 2048 81 / 75.)
constexpr int FEW_ROWS = 64;

// Geometry of a BM x BN tile of TMB 32-row m-blocks computed by WM x WN waves: WM wave rows of TMB/WM m-blocks
// each, WN wave columns of 64 columns each.  Eight waves put two on every SIMD: while one waits for
// the memory pipeline to accept a load or for a barrier, the other issues MFMAs.
template <int TMB, int WM, int WN> struct Tile {
    static constexpr int NW = WM * WN, THREADS = 64 * NW, TMW = TMB / WM;
    static constexpr int BM = TMB * 32, BN = 64 * WN;
    static constexpr int M_ROWS = (BM + 16 * NW - 1) / (16 * NW) * (16 * NW);   // rows the waves' loads cover
    static constexpr int M_OPERAND = M_ROWS * Q_BK * 2, N_OPERAND = BN * Q_BK * 2;   // bytes of one stage
    static constexpr int STAGE = M_OPERAND + N_OPERAND;
    static constexpr bool WHOLE_CU = TMB >= 8 && WN == 4;
    static constexpr int LDS_BUDGET = TMB >= 4 ? 80 * 1024 : 40 * 1024;   // two or four blocks per CU
    static constexpr int NSTAGE = WHOLE_CU ? 4 : (LDS_BUDGET / STAGE < 6 ? LDS_BUDGET / STAGE : 6);
    static constexpr int SLABS = NW * TMW * 32 * 128;                // the waves' epilogue staging areas
    static constexpr int LDS_BYTES = NSTAGE * STAGE > SLABS ? NSTAGE * STAGE : SLABS;
    static constexpr int WAVES_PER_SIMD = TMB >= 4 ? 2 : 4;
};

// One stage of the operand ring for a tile of which the first TMC 32-row blocks are live.  Of a K-contiguous
// m-side tile only the 64-row groups that hold live blocks are fetched and stored, so a light tile has
// smaller stages and its ring, in the same LDS, is deeper: light tiles do little arithmetic per stage and
// run at the memory latency divided by the stages in flight.
// NS: stages of a full tile that the ring has room for.
template <int TMB, int WM, int WN, bool M_KS, int TMC, int NS = Tile<TMB, WM, WN>::NSTAGE> struct Stage {
    typedef Tile<TMB, WM, WN> TL;
    static constexpr int RPL = 16 * TL::NW;                                       // rows (or 16-byte slot groups) one load of every wave covers
    static_assert(!M_KS || TL::BM % RPL == 0, "a K-strided m-side tile must be whole load rounds wide");
    static constexpr int LM = M_KS ? TL::BM / RPL : (TMC * 32 + RPL - 1) / RPL;  // m-side loads per wave
    static constexpr int LN = TL::BN / RPL;
    static constexpr int L = LM + LN;                                             // loads per wave
    static constexpr int M_OPERAND = LM * RPL * Q_BK * 2;
    static constexpr int BYTES = M_OPERAND + TL::N_OPERAND;
    static constexpr int FIT = NS * TL::STAGE / BYTES;
    static constexpr int NSTAGE = FIT > 6 ? 6 : FIT;
};

// ---- operand tiles in LDS -------------------------------------------------------------------------
// A stage holds 32 of K.  Every lane always issues its load (no divergent branches in the K loop):
// rows past the operand's extent are clamped to the last valid row / 16-byte piece.  What lands in
// LDS for them is real, finite data that only contributes to output rows or columns the epilogue
// does not store - except along a ragged contraction length, which the zero_*_tail functions repair.
//
// K-contiguous operand, element (r, k) at p[r*ld + k]: LDS [ROWS][4 x 16 B], the chunk index XORed
// with swz16(row).  A fragment read has lane l at row l % 16, chunk l / 16; one pass of ds_read_b128 serves 16 lanes, either
// 16 neighbours or (0-3, 12-15, 20-27) and its like, and with this swizzle both kinds fall into distinct bank groups of the
// 64-bank LDS.
// With NW waves, wave w's load i fills LDS bytes [(NW i + w)*1024, +1024) = rows 16(NW i + w) .. +16.
// Per-lane byte offsets of the ROWS/(16 NW) loads a wave issues for one stage of an operand tile, relative to
// the tile's first element at the stage's first k (what the scalar base points at).  r_left = rows of the
// operand from the tile's first row on.
__device__ __forceinline__ int swz16(int row) { return ((row >> 3) & 1) | (((row >> 1) ^ (row >> 2)) & 2); }
// src: the operand's rows are those of a matrix of n_src rows that src names, and the base is that matrix (null: they lie there in order).
template <int ROWS, int NW> struct OffKC {
    uint32_t off[ROWS / (16 * NW)];
    __device__ __forceinline__ void init(long ld, int r_left, const int32_t *src, int n_src) {
        uint32_t at[ROWS / (16 * NW)];
#pragma unroll
        for (int i = 0; i < ROWS / (16 * NW); ++i) {
            at[i] = (uint32_t)min((NW * i + (int)(threadIdx.x >> 6)) * 16 + ((int)threadIdx.x >> 2 & 15), r_left - 1);
            if (src != nullptr) at[i] = min((uint32_t)src[at[i]], (uint32_t)n_src - 1u);
        }
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
        for (int i = 0; i < ROWS / (16 * NW); ++i) {
            const int row = (NW * i + w) * 16 + (lane >> 2);
            off[i] = (uint32_t)(at[i] * ld * 2 + ((lane & 3) ^ swz16(row)) * 16);
        }
    }
    // of a stage with k_left (a multiple of 8) of k: the last 16-byte piece instead of those past it
    __device__ __forceinline__ void clamp(int k_left, long) {
        const int lane = threadIdx.x & 63;
        const uint32_t past = (uint32_t)max(((lane & 3) ^ swz16(lane >> 2)) - ((k_left >> 3) - 1), 0) * 16;      // (the swizzle goes by the row's place among 16)
#pragma unroll
        for (int i = 0; i < ROWS / (16 * NW); ++i) off[i] -= past;
    }
};
// K-strided operand, element (r, k) at p[k*ld + r]: LDS [32 k][ROWS x 2 B] as it lies in HBM, the
// 32-byte granule index XORed with swz_ks(k) (conflict-free transpose reads, see frag_ks).
// A k-row has ROWS/8 slots of 16 bytes; a wave load of 1 KiB covers 512/ROWS k-rows.
__device__ __forceinline__ int swz_ks(int k) { return ((k & 3) << 1) | ((k >> 3) & 1); }
template <int ROWS, int NW> struct OffKS {
    uint32_t off[ROWS / (16 * NW)];
    static constexpr int SPR = ROWS / 8;          // 16-byte slots per k-row
    static constexpr int KPL = 64 / SPR;          // k-rows per wave load
    __device__ __forceinline__ void init(long ld, int r_left, const int32_t *, int) {
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
        for (int i = 0; i < ROWS / (16 * NW); ++i) {
            const int kr = (NW * i + w) * KPL + lane / SPR;
            const int pc = lane % SPR;                                        // physical 16-byte slot in the k-row
            const int c = ((((pc >> 1) ^ swz_ks(kr)) << 1) | (pc & 1));  // logical 16-byte chunk
            off[i] = (uint32_t)(kr * ld * 2 + min(c * 8, r_left - 8) * 2);
        }
    }
    // of a stage with k_left k-rows: the last one instead of those past it
    __device__ __forceinline__ void clamp(int k_left, long ld) {
#pragma unroll
        for (int i = 0; i < ROWS / (16 * NW); ++i)
            off[i] -= (uint32_t)(max((NW * i + (int)(threadIdx.x >> 6)) * KPL + (int)(threadIdx.x & 63) / SPR - (k_left - 1), 0) * ld * 2);
    }
};
template <int ROWS, int NW, bool KS> struct Off;
template <int ROWS, int NW> struct Off<ROWS, NW, false> : OffKC<ROWS, NW> {};
template <int ROWS, int NW> struct Off<ROWS, NW, true> : OffKS<ROWS, NW> {};
// zero the chunks of k from k_valid (a multiple of 8) on of a K-contiguous tile
template <int ROWS, int THREADS> __device__ __forceinline__ void zero_kc_tail(char *lds, int k_valid) {
    for (int idx = threadIdx.x; idx < ROWS * 4; idx += THREADS) {
        const int row = idx >> 2, c = idx & 3;
        if (c * 8 >= k_valid) *reinterpret_cast<uint4 *>(lds + row * 64 + ((c ^ swz16(row)) << 4)) = make_uint4(0, 0, 0, 0);
    }
}
// zero the k-rows [k_valid, 32) of a K-strided tile
template <int ROWS, int THREADS> __device__ __forceinline__ void zero_k_tail(char *lds, int k_valid) {
    for (int idx = threadIdx.x; idx < (Q_BK - k_valid) * (ROWS / 8); idx += THREADS)
        *reinterpret_cast<uint4 *>(lds + k_valid * (ROWS * 2) + idx * 16) = make_uint4(0, 0, 0, 0);
}

// ---- MFMA fragments: 8 bf16 of k (8 (lane / 16) on) for row lane % 16 of 16-row block tb; one covers the stage's 32 of k --
// v_mfma_f32_16x16x32_bf16 and not the 32x32x16 shape of the same rate: the chip runs matrix work against its power limit,
// and per flop the smaller shape moves half of the accumulator bytes.  Back to back on random operands held in registers
// (mole_probe_mfma, 256 blocks of eight waves; the same probe with either shape, in turn on one box) it sustains 1661-1686 TFLOP/s
// against 1520-1536, on zeros 2274-2298 against 2212-2234; the K loop of h at 16384 x 1024 -> 4096 takes 112-114 us against 121-124.
__device__ __forceinline__ bf16x8 frag_kc(const char *lds, int tb) {
    const int lane = threadIdx.x & 63;
    const int row = lane & 15;
    const int chunk = (lane >> 4) ^ swz16(row);
    return __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(lds + tb * 1024 + row * 64 + chunk * 16));
}
// ds_read_b64_tr_b16: in a group of 16 lanes, lane 4r+q supplies the address of 4 consecutive values
// of k-row r, and lane i receives column i of that 4 x 16 block.  Two reads give 8 of k.
template <int ROWS> __device__ __forceinline__ bf16x8 frag_ks(const char *lds, int tb) {
    const int lane = threadIdx.x & 63;
    const int l = lane & 15;
    const int k = 8 * (lane >> 4) + (l >> 2);                           // + 4 for the second read
    const int gran = tb ^ swz_ks(k);                                    // (the same for k + 4)
    const char *a0 = lds + k * (ROWS * 2) + gran * 32 + (l & 3) * 8;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(a0));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3))) *)(a0 + 4 * ROWS * 2));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    return __builtin_bit_cast(bf16x8, v);
}
template <bool KS, int ROWS> __device__ __forceinline__ bf16x8 frag(const char *lds, int tb) {
    if constexpr (KS) return frag_ks<ROWS>(lds, tb); else return frag_kc(lds, tb);
}

// first index of part P when N items are dealt to NP consecutive parts
template <int P, int NP, int N> constexpr int part_lo() { return P * N / NP; }

// The fragments one wave needs for a stage: its 2 TMCW 16-row m-blocks (those from 2 wm TMCW on of the tile, of which
// the tile's first 2 TMC are fetched) in two halves, and its four 16-column n-blocks.  A stage is consumed in two halves of
// four parts: part P of half H multiplies n-block P with the TMCW m-blocks of half H.  The other half of the m-side is read
// meanwhile, and in the second half the next stage's first: n-block P has been used for the last time after part P of that
// half and is read again in the part that follows, so that the n-side needs no second set of registers.
template <int TMB, int WM, int WN, bool M_KS, bool N_KS, int TMC, int TMCW> struct Frags {
    typedef Tile<TMB, WM, WN> TL;
    bf16x8 m[2][TMCW ? TMCW : 1], n[4];
    __device__ __forceinline__ void read_n(const char *stage, int wn, int j) {
        n[j] = frag<N_KS, TL::BN>(stage + Stage<TMB, WM, WN, M_KS, TMC>::M_OPERAND, wn * 4 + j);
    }
    template <int H> __device__ __forceinline__ void read_m(const char *stage, int wm, int i) {
        m[H][i] = frag<M_KS, TL::BM>(stage, wm * 2 * TMCW + H * TMCW + i);
    }
    // the reads that go with part P of half H (H 0: from the stage that is being consumed, H 1: from the next one).  The
    // m-side goes into the first three parts, as the half that follows needs all of it at once.
    template <int H, int P> __device__ __forceinline__ void read_part(const char *stage, int wm, int wn) {
        if constexpr (TMCW > 0) {
            if constexpr (H == 0 && P == 0) read_n(stage, wn, 3);
            if constexpr (P < 3) {
#pragma unroll
                for (int i = part_lo<P, 3, TMCW>(); i < part_lo<P + 1, 3, TMCW>(); ++i) read_m<1 - H>(stage, wm, i);
            }
            if constexpr (H == 1 && P > 0) read_n(stage, wn, P - 1);
        }
    }
    // what part 0 of half 0 finds already read
    __device__ __forceinline__ void read_first(const char *stage, int wm, int wn) {
        if constexpr (TMCW > 0) {
#pragma unroll
            for (int i = 0; i < TMCW; ++i) read_m<0>(stage, wm, i);
#pragma unroll
            for (int j = 0; j < 3; ++j) read_n(stage, wn, j);
        }
    }
    // the MFMAs of part P of half H.  SUM adds MFMAs against a block of ones, which sum an operand's blocks over k: of the
    // m-side (SUM 1; wave column i takes the wave row's m-blocks 2 i and 2 i + 1) or of the n-side (SUM 2; wave row j takes
    // the wave column's n-blocks 2 j and 2 j + 1).
    template <int H, int P, int SUM> __device__ __forceinline__ void mma_part(f32x4 (&acc)[2 * TL::TMW][4], f32x4 (&sums)[2], int wm, int wn) const {
#pragma unroll
        for (int i = 0; i < TMCW; ++i)
            acc[H * TMCW + i][P] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(n[P], m[H][i], acc[H * TMCW + i][P], 0, 0, 0);
        if constexpr (SUM != 0) {
            static_assert(SUM != 1 || TMCW <= WN, "the wave columns share out a wave row's m-blocks");
            const bf16_t one = (bf16_t)1.0f;
            const bf16x8 ones = {one, one, one, one, one, one, one, one};
            if constexpr (SUM == 1 && P == 3) {
#pragma unroll
                for (int i = 0; i < TMCW; ++i)
                    if (wn == (H * TMCW + i) >> 1) sums[(H * TMCW + i) & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, m[H][i], sums[(H * TMCW + i) & 1], 0, 0, 0);
            } else if constexpr (SUM == 2 && H == 0) {
                if (wm == P >> 1) sums[P & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(n[P], ones, sums[P & 1], 0, 0, 0);
            }
        }
    }
};

// Issues the asynchronous loads of the operand stages of one tile.  The two operand tiles are addressed
// by a scalar base (advanced by one stage of K after a stage's last load) plus per-lane offsets that stay
// fixed for the whole K loop.  Stages are fetched in order.
// Of a K-contiguous m-side tile only the 64-row groups that hold live 32-row blocks (the first TMC) are fetched.
// KT: the contraction may not be whole stages (weight gradients; row-ragged products when K is not a multiple of 32).  The loads of what is
// left over are clamped to what exists, and main_loop zeroes the rest of its stage.  A weight gradient takes it first, as stage 0, and its loop then
// meets whole stages only.  As the last stage it had every iteration choose between two sets of offsets and ask
// whether its stage was that one, 47 ns of a stage's 230 on 128 x 128 tiles.  us, left over last / first: 64
// experts of 1024 x 2048, 100 rows, 78.8 / 73.4, 200 rows 98 / 95, 500 rows 167 / 164; 16 of 1024 x 4096, 500 rows, 80.1 / 78.0;
// 59 of 568 x 2272, 100 rows, 53.0 / 50.4.  A row-ragged product takes it last, so that its sums are in the order of k whatever the
// width: the offsets are changed once, in the iteration that issues the first of that stage's loads (first: 0.6 % of a training pass less, 19 passes of such
// widths; loops that stop between iterations for it: no faster).
// ONCE: no other tile reads this tile's n-side panel (the weights of an expert with a single m-tile).
template <int TMB, int WM, int WN, bool M_KS, bool N_KS, bool KT, int TMC, bool ONCE> struct Feeder {
    typedef Tile<TMB, WM, WN> TL;
    typedef Stage<TMB, WM, WN, M_KS, TMC> SG;
    static constexpr int LM = SG::LM, L = SG::L;
    Off<TL::M_ROWS, TL::NW, M_KS> om;
    Off<TL::BN, TL::NW, N_KS> on;
    const char *bm, *bn;
    long step_m, step_n;
    uint32_t lds_w;      // LDS address of ring buffer 0 + this wave's 1 KiB lane
    int nk;
    int left, tail;      // KT: k of the stage that is not a whole one (0: there is none), and its number (otherwise one that no stage has)
    __device__ __forceinline__ void init(const bf16_t *Mp, long ldm, int m0, int m_ext, const bf16_t *Np, long ldn, int n0,
                                         int n_ext, int k_ext, char *smem, int wave, const int32_t *src, int n_src) {
        om.init(ldm, m_ext - m0, src, n_src);
        on.init(ldn, n_ext - n0, nullptr, 0);
        bm = uniform_ptr(src != nullptr ? Mp : M_KS ? Mp + m0 : Mp + (long)m0 * ldm);
        bn = uniform_ptr(N_KS ? Np + n0 : Np + (long)n0 * ldn);
        step_m = M_KS ? ldm * (Q_BK * 2) : Q_BK * 2;
        step_n = N_KS ? ldn * (Q_BK * 2) : Q_BK * 2;
        lds_w = lds_offset_of(smem) + __builtin_amdgcn_readfirstlane(wave * 1024);
        nk = (k_ext + Q_BK - 1) / Q_BK;
        left = KT ? __builtin_amdgcn_readfirstlane(k_ext & (Q_BK - 1)) : 0;
        tail = __builtin_amdgcn_readfirstlane(!left ? -1 : M_KS ? 0 : nk - 1);
    }
    // the loads are those of the stage that is not a whole one from here on
    __device__ __forceinline__ void clamp() {
        om.clamp(left, step_m / (Q_BK * 2));
        on.clamp(left, step_n / (Q_BK * 2));
    }
    __device__ __forceinline__ void load(int j, uint32_t o, uint32_t dst) const {
        if (j < LM) dma16s(bm, o, dst + j * (TL::NW * 1024));
        else if constexpr (ONCE) dma16s_nt(bn, o, dst + SG::M_OPERAND + (j - LM) * (TL::NW * 1024));
        else dma16s(bn, o, dst + SG::M_OPERAND + (j - LM) * (TL::NW * 1024));
    }
    // weight gradients: the loads of stage 0, into ring buffer 0
    __device__ __forceinline__ void issue_first() {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_w);
        Feeder f = *this;
        const long ahead = left ? nk - 1 : 0;         // stages before what is left over
        f.bm += ahead * step_m;
        f.bn += ahead * step_n;
        if (left) f.clamp();
#pragma unroll
        for (int j = 0; j < L; ++j) f.load(j, j < LM ? f.om.off[j < LM ? j : 0] : f.on.off[j < LM ? 0 : j - LM], dst);
        if (!left && nk > 1) { bm += step_m; bn += step_n; }
    }
    // loads [J0, J1) of stage s (the m-side tile's loads come first) into ring buffer buf; past the last stage that one's again
    template <int J0, int J1> __device__ __forceinline__ void issue(int s, int buf) {
        const uint32_t dst = __builtin_amdgcn_readfirstlane(lds_w + buf * SG::BYTES);
#pragma unroll
        for (int j = J0; j < J1; ++j) load(j, j < LM ? om.off[j < LM ? j : 0] : on.off[j < LM ? 0 : j - LM], dst);
        if (J1 == L && s + 1 < nk) { bm += step_m; bn += step_n; }
    }
};

__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
    const bf16x4 v = {(bf16_t)a, (bf16_t)b, (bf16_t)c, (bf16_t)d};
    return __builtin_bit_cast(uint2, v);
}
__device__ __forceinline__ void unpack4(uint2 u, float *f) {
    f[0] = __uint_as_float(u.x << 16);
    f[1] = __uint_as_float(u.x & 0xffff0000u);
    f[2] = __uint_as_float(u.y << 16);
    f[3] = __uint_as_float(u.y & 0xffff0000u);
}

// Waits until at most `behind` whole stages of L loads each (behind <= B; below 0 counts as 0), and X more loads if
// `extra`, are in flight (the instruction takes its count as an immediate, hence the chain).
template <int B, int L, int X> __device__ __forceinline__ void wait_stages_behind(int behind, bool extra) {
    if constexpr (B <= 0) {
        if (extra) __builtin_amdgcn_s_waitcnt(waitcnt_vm(X));
        else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    } else {
        if (behind >= B) {
            if (extra) __builtin_amdgcn_s_waitcnt(waitcnt_vm(B * L + X));
            else __builtin_amdgcn_s_waitcnt(waitcnt_vm(B * L));
        } else {
            wait_stages_behind<B - 1, L, X>(behind, extra);
        }
    }
}

// The K loop.  Stage s (32 of K) lives in ring buffer s mod NSTAGE and is fetched NSTAGE-1 stages ahead.
// A wave cannot issue MFMAs while one of its loads waits for the memory pipeline to take it, so the loads
// of a stage are not issued in one burst: each half of an iteration is cut into parts, and a part issues
// its share of the loads, then its share of the fragment reads for the next sub-step, then its MFMAs.
// The second half of iteration s issues the first half of the loads of stage s+AHEAD, the first half of
// iteration s+1 the rest, into the buffer that stage s-1 has left.  One synchronisation point per
// iteration, between the halves: wait until this wave's share of stage s+1 has landed (newer stages may
// still be in flight), then the barrier.
// PART (measurement only, results are then meaningless): 1 leaves out the operand loads, 2 the fragment reads of the
// loop (the first stage's fragments are used throughout), 3 the barriers, 4 all three.
// BIAS: the accumulators start from the bias of their columns instead of zero (bias_raw: the 4 x 4 columns a lane
// holds, fetched before the operand loads and therefore landed when the first stage has), so that the epilogue adds
// nothing.
template <int TMB, int WM, int WN, int NS, bool M_KS, bool N_KS, bool KT, int TMC, int TMCW, int SUM, bool ONCE = false, int PART = 0, bool BIAS = false>
__device__ __forceinline__ void main_loop(const bf16_t *Mp, long ldm, int m0, int m_ext, const bf16_t *Np, long ldn,
                                          int n0, int n_ext, int k_ext, char *smem, int wave, int wm, int wn,
                                          f32x4 (&acc)[2 * Tile<TMB, WM, WN>::TMW][4], f32x4 (&sums)[2], const uint2 (&bias_raw)[4], const int32_t *src, int n_src) {
    typedef Tile<TMB, WM, WN> TL;
    typedef Stage<TMB, WM, WN, M_KS, TMC, NS> SG;
    constexpr int AHEAD = SG::NSTAGE - 1, NP = 4;
    typedef Feeder<TMB, WM, WN, M_KS, N_KS, KT, TMC, ONCE> FD;
    constexpr int L = FD::L, LH = L / 2;      // loads per wave per stage; the halves are LH and L - LH
    constexpr bool LAST = KT && !M_KS;        // what whole stages leave of the contraction comes last (weight gradients: first)
    const int nk = __builtin_amdgcn_readfirstlane((k_ext + Q_BK - 1) / Q_BK);
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2 * Tile<TMB, WM, WN>::TMW; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    };
    if (M_KS || nk == 0) clear();
    if (nk == 0) return;
    FD fd;
    fd.init(Mp, ldm, m0, m_ext, Np, ldn, n0, n_ext, k_ext, smem, wave, src, n_src);
    // SPLIT: with three or more stages in flight a stage's loads are spread over two halves (one iteration
    // of look-ahead is lost for the later half); with two, all of them go into the half after the barrier.
    constexpr bool SPLIT = AHEAD >= 3;
    constexpr bool NO_LOADS = PART == 1 || PART == 4, NO_READS = PART == 2 || PART == 4, NO_BARRIERS = PART == 3 || PART == 4;
    // Only stages that exist are fetched (but for one part of a stage, see below): the prologue stops at the
    // contraction's last stage, the last iterations issue nothing, and the waits count what is really in flight.
    // Fetching AHEAD stages past the end, as a loop with one kind of iteration does, costs a tile of K = 1024 a tenth
    // more loads, a one-stage tile of a nearly empty expert four times its loads, and the epilogue a wait for loads
    // that nothing reads.  The iterations without loads are a second copy of the loop body, compiled without them: the
    // same body with the loads under a (wave-uniform) condition ran 3-10 % slower, and a third copy for the one
    // iteration in between made the register allocator spill.
    constexpr int LX = SPLIT ? LH : L;        // loads of stage AHEAD - 1 that the prologue issues
    if constexpr (!NO_LOADS) {
        static_assert(AHEAD >= 2, "the prologue issues all of stage 0");
        if constexpr (M_KS) fd.issue_first();
#pragma unroll
        for (int s = M_KS ? 1 : 0; s < AHEAD - 1; ++s)
            if (s < nk) {
                if (LAST && s == fd.tail) fd.clamp();
                fd.template issue<0, L>(s, s);
            }
        if (AHEAD - 1 < nk) {
            if (LAST && AHEAD - 1 == fd.tail) fd.clamp();
            fd.template issue<0, LX>(AHEAD - 1, AHEAD - 1);
        }
    }
    if constexpr (!M_KS) clear();       // (while the loads are on their way; weight gradients are 1 % slower for it)
    // stage 0 has landed when no more is in flight than what was issued after it
    if (nk >= AHEAD) __builtin_amdgcn_s_waitcnt(waitcnt_vm((AHEAD - 2) * L + LX));
    else wait_stages_behind<AHEAD - 2, L, 0>(nk - 1, false);
    __builtin_amdgcn_s_barrier();
    if constexpr (BIAS) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            float b4[4];
            unpack4(bias_raw[c], b4);
#pragma unroll
            for (int tm = 0; tm < 2 * TMCW; ++tm)
#pragma unroll
                for (int j = 0; j < 4; ++j) acc[tm][c][j] = b4[j];
        }
    }
    // zeroes what lies past the contraction's end in the stage that is not a whole one, which has landed in buf
    auto zero_rest = [&](char *buf) __attribute__((always_inline)) {
        if constexpr (M_KS) zero_k_tail<TL::BM, TL::THREADS>(buf, fd.left);
        else zero_kc_tail<SG::M_OPERAND / 64, TL::THREADS>(buf, fd.left);
        if constexpr (N_KS) zero_k_tail<TL::BN, TL::THREADS>(buf + SG::M_OPERAND, fd.left);
        else zero_kc_tail<TL::BN, TL::THREADS>(buf + SG::M_OPERAND, fd.left);
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (and not for loads that are in flight)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    if (KT && fd.tail == 0) zero_rest(smem);
    Frags<TMB, WM, WN, M_KS, N_KS, TMC, TMCW> fr;
    fr.read_first(smem, wm, wn);
    if constexpr (NO_READS) {
        fr.template read_part<0, 0>(smem, wm, wn);
        fr.template read_part<0, 1>(smem, wm, wn);
        fr.template read_part<0, 2>(smem, wm, wn);
    }
    int cur_b = 0;                    // ring buffer of stage s
#define MOLE_PART(ISSUE, H, P, J0, N, S_LOAD, BUF, STAGE_PTR)                                    \
        if constexpr (!NO_LOADS && (ISSUE)) fd.template issue<(J0) + part_lo<P, NP, (N)>(), (J0) + part_lo<P + 1, NP, (N)>()>(S_LOAD, BUF); \
        if constexpr (!NO_READS) fr.template read_part<H, P>(STAGE_PTR, wm, wn);                            \
        fr.template mma_part<H, P, SUM>(acc, sums, wm, wn);                                               \
        __builtin_amdgcn_sched_barrier(0);
    // One iteration (stage s).  ISSUE: the first half issues the rest of stage s + AHEAD - 1, the second the first
    // loads of stage s + AHEAD; WAIT: the wait for stage s + 1.
#define MOLE_ITER(ISSUE, WAIT)                                                                            \
    {                                                                                                     \
        const int nxt_b = cur_b + 1 == SG::NSTAGE ? 0 : cur_b + 1;                                        \
        const int free_b = cur_b == 0 ? SG::NSTAGE - 1 : cur_b - 1;     /* held stage s-1, takes stage s+AHEAD */ \
        const int fill_b = free_b == 0 ? SG::NSTAGE - 1 : free_b - 1;   /* takes the rest of stage s+AHEAD-1 */   \
        const char *cur = smem + cur_b * SG::BYTES;                                                       \
        char *nxt = smem + nxt_b * SG::BYTES;                                                       \
        MOLE_PART(ISSUE, 0, 0, SPLIT ? LH : 0, SPLIT ? L - LH : 0, s + AHEAD - 1, fill_b, cur)             \
        MOLE_PART(ISSUE, 0, 1, SPLIT ? LH : 0, SPLIT ? L - LH : 0, s + AHEAD - 1, fill_b, cur)             \
        MOLE_PART(ISSUE, 0, 2, SPLIT ? LH : 0, SPLIT ? L - LH : 0, s + AHEAD - 1, fill_b, cur)             \
        MOLE_PART(ISSUE, 0, 3, SPLIT ? LH : 0, SPLIT ? L - LH : 0, s + AHEAD - 1, fill_b, cur)             \
        WAIT;                                                                                             \
        if constexpr (!NO_BARRIERS) __builtin_amdgcn_s_barrier();                                         \
        __builtin_amdgcn_sched_barrier(0);                                                                \
        if constexpr (LAST && (AHEAD < 3 || !(ISSUE))) { if (s + 1 == fd.tail) zero_rest(nxt); }  /* (the last iteration but one) */ \
        if constexpr (LAST && (ISSUE)) { if (s + AHEAD == fd.tail) fd.clamp(); }                          \
        MOLE_PART(ISSUE, 1, 0, 0, SPLIT ? LH : L, s + AHEAD, free_b, nxt)                                  \
        MOLE_PART(ISSUE, 1, 1, 0, SPLIT ? LH : L, s + AHEAD, free_b, nxt)                                  \
        MOLE_PART(ISSUE, 1, 2, 0, SPLIT ? LH : L, s + AHEAD, free_b, nxt)                                  \
        MOLE_PART(ISSUE, 1, 3, 0, SPLIT ? LH : L, s + AHEAD, free_b, nxt)                                  \
        cur_b = nxt_b;                                                                                    \
    }
    int s = 0;
    // while stage s + AHEAD - 1 exists: its rest is issued, then the first loads of stage s + AHEAD (in the last of
    // these iterations that stage does not exist: LX loads that nothing reads, the only ones of a tile)
    // the last AHEAD - 1 iterations issue nothing; in flight behind stage s + 1: the stages after it and those LX loads
    const bool extra = nk >= AHEAD;
    for (; s + AHEAD - 1 < nk; ++s) MOLE_ITER(true, __builtin_amdgcn_s_waitcnt(waitcnt_vm((AHEAD - 2) * L)))
    for (; s < nk; ++s) MOLE_ITER(false, (wait_stages_behind<AHEAD - 2, L, LX>(nk - 2 - s, extra)))
#undef MOLE_ITER
#undef MOLE_PART
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));   // nothing may still be writing LDS when the block retires
}

// The bias of the 4 x 4 columns a lane holds results for, as raw bf16 quadruples; fetched before the K loop
// so that the epilogue does not wait for it (zero bits are 0.0 in bf16).
template <int EPI> __device__ __forceinline__ void load_bias(const GemmArgs &g, int e, int n0, int lane, int wn, uint2 (&bias_raw)[4]) {
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        bias_raw[c] = make_uint2(0, 0);
        if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) {
            const int n = n0 + wn * 64 + 16 * c + 4 * (lane >> 4);
            if (n < g.N) bias_raw[c] = *reinterpret_cast<const uint2 *>((const bf16_t *)g.bias + (long)e * g.N + n);
        }
    }
}

// The epilogue of one wave, whose first TMCW 32-row blocks hold live rows.  acc[tm][tn][j] = C[m, n] with
// m = m0 + 16 tm + lane%16 (m0: the wave's first row) and n = n0 + 64 wn + 16 tn + 4 (lane/16) + j.  A wave
// owns a (32 TMW) x 64 slab of the tile.  bf16 results go through the wave's own slab of LDS (the K loop is
// done with it) so that global memory sees whole 128-byte rows: 8 bytes per lane into LDS, then 16 bytes
// per lane out, 8 rows per store instruction.  The pre-activation that GELU' needs comes in the same way,
// in the opposite direction.  TMCW is a compile-time bound so that the work of different cells can be
// interleaved.  live: the wave's live rows.
// CLOSED: GELU and its derivatives by their closed forms instead of the fitted polynomials (see gemm.h).
template <int TMB, int WM, int WN, bool WG, int EPI, int TMC, bool CLOSED>
__device__ __forceinline__ void epilogue(const GemmArgs &g, f32x4 (&acc)[2 * Tile<TMB, WM, WN>::TMW][4], char *smem, int lane, int wave,
                                         int wn, int e, long row0, int m0, int n0, int m_ext, int live,
                                         int split_k) {
    __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __syncthreads();
    if constexpr (TMC == 0) return;
    const int lm = lane & 15, h = lane >> 4;
    bf16_t *Cb = (bf16_t *)g.C;
    long crow0 = row0;
    if constexpr (WG) { crow0 = 0; Cb += (long)e * g.strideC; }
    const int nw0 = n0 + wn * 64;                   // first column of this wave's slab
    char *slab = smem + wave * (Tile<TMB, WM, WN>::TMW * 32 * 128);
    const int jr = lane >> 3, jc = lane & 7;        // row-in-group / 16-byte column of the wide accesses
    const bool col_ok = nw0 + jc * 8 < g.N;

    // 16-byte chunk of a row at chunk ^ (row >> 1) & 7: the 16 rows x 16 bytes one ds_write_b64 pass writes (a lane
    // holds half of a chunk) land in 32 distinct 8-byte bank groups
    auto slab_at = [&](int row, int chunk, int half) -> char * {
        return slab + row * 128 + ((chunk ^ ((row >> 1) & 7)) << 4) + half * 8;
    };
    // slab -> global: rows [0, live) of the slab, 128 bytes each
    // The large results - h, a, t and the weight gradients, 134-270 MB a launch, which no block of the same
    // launch reads - leave with non-temporal stores: ordinary stores let them push the operand panels of the
    // running K loops out of the L2 and the last-level cache.  Measured at 16 experts of 1024 x 4096 over 16384
    // rows (same-box A/B): h and a of the first product -11 us, the weight gradients -6 us and the GELU' product
    // that follows them -6 us, t of the GELU' product -4 us; the launches that read them later are MFMA-bound
    // and take them from HBM at no loss.  The small results (out, gx: 34 MB) stay ordinary: the row permutes
    // that read them next are memory-bound and lost more than the products gained.
    constexpr bool STREAM_OUT = EPI == EPI_BIAS_GELU || EPI == EPI_DGELU || EPI == EPI_WGRAD;
    // Addresses of the wide accesses: a wave-uniform 64-bit base (the slab's first row in the result, advanced by
    // scalar adds from row group to row group) plus a 32-bit per-lane byte offset that is computed once, so a store
    // costs no address arithmetic on the vector ALU; and the LDS reads of a batch of eight row groups are issued
    // before the first store, so that one LDS latency is waited for per batch instead of one per store.  (Written
    // row by row with the row test around the read and the store, each store waited for its own LDS read and
    // recomputed a 64-bit row * pitch product: two thirds of the epilogue's time apart from the activation.)
    const uint32_t pitch = (uint32_t)g.ldc * 2;                          // bytes between rows of the result
    const uint32_t lane_off = (uint32_t)jr * pitch + (uint32_t)jc * 16;  // this lane's 16 bytes of row jr
    // every row group and every column is stored (the same in all lanes)
    const bool full = __builtin_amdgcn_readfirstlane(live >= TMC * 32 && nw0 + 64 <= g.N) != 0;
    // LDS address of this lane's 16 bytes of row group `it` (rows 8 it + jr): with row = 8 it + jr the swizzle term
    // (row >> 1) & 7 is (jr >> 1) | ((it & 1) << 2), so two per-lane bases and a constant per row group suffice
    char *const wide0 = slab + jr * 128 + ((jc ^ (jr >> 1)) << 4);
    char *const wide1 = slab + jr * 128 + ((jc ^ (jr >> 1) ^ 4) << 4);
    auto wide_cell = [&](int it) -> char * { return ((it & 1) ? wide1 : wide0) + it * 1024; };
    typedef __attribute__((address_space(1))) char gchar;
    auto flush = [&](bf16_t *dst) __attribute__((always_inline)) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        gchar *gbase = (gchar *)((char *)dst + ((crow0 + m0) * g.ldc + nw0) * 2);
#pragma unroll
        for (int it0 = 0; it0 < TMC * 4; it0 += 8) {
            uint4 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (it0 + i < TMC * 4) v[i] = *reinterpret_cast<const uint4 *>(wide_cell(it0 + i));
            auto put = [&](int i) __attribute__((always_inline)) {
                gchar *p = gbase + (size_t)(it0 + i) * 8 * pitch + lane_off;
                typedef __attribute__((address_space(1))) u32x4 g_u32x4;
                if constexpr (STREAM_OUT) __builtin_nontemporal_store(u32x4{v[i].x, v[i].y, v[i].z, v[i].w}, reinterpret_cast<g_u32x4 *>(p));
                else *reinterpret_cast<g_u32x4 *>(p) = u32x4{v[i].x, v[i].y, v[i].z, v[i].w};
            };
            if (full) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (it0 + i < TMC * 4) put(i);
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (it0 + i < TMC * 4 && (it0 + i) * 8 + jr < live && col_ok) put(i);
            }
        }
    };
    // global -> slab, eight rows' loads in flight at a time.  Every load is issued, from an address clamped
    // into the operand (rows past the end read its last row, columns past the end its first column): what lands
    // in cells outside the live part is never written back, and a load under a condition would make the
    // compiler wait for all loads in flight at each one, so the eight would run one after the other.
    auto fill = [&](const bf16_t *src) __attribute__((always_inline)) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        // rows are counted from the slab's first row, or from the operand's last row when the slab starts past it
        const long first = min(crow0 + m0, crow0 + m_ext - 1);
        // byte offset of the last valid row, as far as the slab reaches (the row count is bounded before it meets the
        // pitch: an expert of 10^5 rows times a pitch of tens of KB does not fit 32 bits)
        const uint32_t last_off = (uint32_t)min(crow0 + m_ext - 1 - first, (long)(TMC * 32 - 1)) * pitch;
        const gchar *gbase = (const gchar *)((const char *)src + first * g.ldc * 2);
        const uint32_t col_off = col_ok ? (uint32_t)(nw0 + jc * 8) * 2 : 0u;
        const uint32_t row_off = (uint32_t)jr * pitch;
#pragma unroll
        for (int it0 = 0; it0 < TMC * 4; it0 += 8) {
            uint4 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (it0 + i >= TMC * 4) continue;
                const uint32_t ro = min(row_off + (uint32_t)(it0 + i) * 8 * pitch, last_off);
                // read once, here: a non-temporal load keeps it from displacing the K loop's operands (-4 us)
                typedef __attribute__((address_space(1))) u32x4 g_u32x4;
                const u32x4 w = __builtin_nontemporal_load(reinterpret_cast<const g_u32x4 *>(gbase + ro + col_off));
                v[i] = make_uint4(w[0], w[1], w[2], w[3]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (it0 + i < TMC * 4) *reinterpret_cast<uint4 *>(wide_cell(it0 + i)) = v[i];
        }
    };

    if constexpr (EPI >= EPI_NONE) {
        // the K loop alone (mole_probe_kloop): results leave only under a condition that never holds, which is
        // enough to keep the accumulation alive
        if (g.K < 0) {
            float s = 0.f;
#pragma unroll
            for (int tm = 0; tm < 2 * TMC; ++tm)
#pragma unroll
                for (int tn = 0; tn < 4; ++tn)
#pragma unroll
                    for (int j = 0; j < 4; ++j) s += acc[tm][tn][j];
            ((float *)g.C)[threadIdx.x] = s;
        }
        return;
    }
    if constexpr (EPI == EPI_F32) {
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) {
            const int n = nw0 + tn * 16 + 4 * h;
            if (n >= g.N) continue;
#pragma unroll
            for (int tm = 0; tm < 2 * TMC; ++tm) {
                const int m = m0 + tm * 16 + lm;
                if (m >= m_ext) continue;
                *reinterpret_cast<f32x4 *>((float *)g.C + (crow0 + m) * g.ldc + n) = acc[tm][tn];
            }
        }
        return;
    }
    if constexpr (EPI == EPI_PART) {
        // fp32, 32 columns (128 bytes) of a row at a time through the slab: results straight from the accumulators would be
        // 32-byte pieces of 32 rows per store.  Ordinary stores: the reduction reads them next.
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            float *dst = g.part + ((long)split_k * g.part_rows + crow0 + m0) * g.N + nw0 + half * 32;
#pragma unroll
            for (int q = 0; q < 2; ++q)
#pragma unroll
                for (int tm = 0; tm < 2 * TMC; ++tm) {
                    const int row = tm * 16 + lm;
                    *reinterpret_cast<f32x4 *>(slab + row * 128 + (((4 * q + h) ^ ((row >> 1) & 7)) << 4)) = acc[tm][2 * half + q];
                }
            // (the slab is this wave's own: program order is enough)
#pragma unroll
            for (int it = 0; it < TMC * 4; ++it)
                if (it * 8 + jr < live && nw0 + half * 32 + jc * 4 < g.N)
                    *reinterpret_cast<uint4 *>(dst + (long)(it * 8 + jr) * g.N + jc * 4) = *reinterpret_cast<const uint4 *>(wide_cell(it));
        }
        return;
    }
    if constexpr (EPI == EPI_DGELU) fill((const bf16_t *)g.H);
    if constexpr (EPI == EPI_WGRAD) { if (g.accumulate) fill(Cb); }

    DGeluCoef dgelu;
    if constexpr (EPI == EPI_DGELU) dgelu.select(g.gelu_bwd == MOLE_GELU_BWD_TANH);
    // pass 0 writes C; for EPI_BIAS_GELU pass 1 writes C2 = gelu(h), and without a C (no backward pass will ask for h)
    // there is no pass 0
    constexpr int PASSES = EPI == EPI_BIAS_GELU ? 2 : 1;
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
        if constexpr (EPI == EPI_BIAS_GELU) {
            if (pass == 0 && g.C == nullptr) continue;
        }
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) {
            // (the bias is in the accumulators already: the K loop started from it)
#pragma unroll
            for (int tm = 0; tm < 2 * TMC; ++tm) {
                char *cell = slab_at(tm * 16 + lm, tn * 2 + (h >> 1), h & 1);
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = acc[tm][tn][j];
                if constexpr (EPI == EPI_BIAS_GELU) {
                    if (pass == 1) {
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] = CLOSED ? gelu_erf(v[j]) : fast_gelu_erf(v[j]);
                    }
                } else if constexpr (EPI == EPI_DGELU) {
                    float hv[4];
                    unpack4(*reinterpret_cast<const uint2 *>(cell), hv);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[j] *= !CLOSED ? dgelu(hv[j]) : g.gelu_bwd == MOLE_GELU_BWD_TANH ? d_gelu_tanh(hv[j]) : d_gelu_exact(hv[j]);
                } else if constexpr (EPI == EPI_WGRAD) {
                    if (g.accumulate) {
                        float old[4];
                        unpack4(*reinterpret_cast<const uint2 *>(cell), old);
#pragma unroll
                        for (int j = 0; j < 4; ++j) v[j] += old[j];
                    }
                }
                *reinterpret_cast<uint2 *>(cell) = pack4(v[0], v[1], v[2], v[3]);
            }
        }
        flush(pass == 0 ? Cb : (bf16_t *)g.C2);
    }
}

// Writes the operand sums of a weight-gradient block (see Frags::mma_part): colsum[e][i] (+)= sum over the
// expert's rows of operand column i.  SUM 1: every register of lane l < 16 holds the sum for row l of the wave's two
// summed m-blocks (blocks 2 wn and 2 wn + 1 of wave row wm); SUM 2: register j of a lane holds the sum for column
// 4 (lane/16) + j of the wave's two summed n-blocks (blocks 2 wm and 2 wm + 1 of wave column wn).
template <int SUM, int C>
__device__ __forceinline__ void store_sums(const GemmArgs &g, const f32x4 (&sums)[2], int e, int m0, int n0, int m_ext, int wm,
                                           int wn, int lane) {
    bf16_t *out = (bf16_t *)g.colsum;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        if constexpr (SUM == 1) {
            const int m = m0 + (wm * C + wn) * 32 + 16 * b + (lane & 15);
            if (lane < 16 && wn < C && m < m_ext) {
                bf16_t *p = out + (long)e * g.M + m;
                float v = sums[b][0];
                if (g.accumulate) v += (float)*p;
                *p = (bf16_t)v;
            }
        } else if ((lane & 15) == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int n = n0 + wn * 64 + wm * 32 + 16 * b + 4 * (lane >> 4) + j;
                if (n < g.N) {
                    bf16_t *p = out + (long)e * g.N + n;
                    float v = sums[b][j];
                    if (g.accumulate) v += (float)*p;
                    *p = (bf16_t)v;
                }
            }
        }
    }
}

// Row-ragged (!WG): C[rows_e, N] = Mop[rows_e, K] . Nop_e ; Mop K-contiguous, Nop_e [N,K] or (N_KS) [K,N].
// Weight gradient (WG): C_e[M, N] = sum_{r in rows_e} Mop[r, M]^T . Nop[r, N], both K-strided.
// block: the block's number among those of the product.
template <int TMB, int WM, int WN, bool N_KS, bool WG, bool KT, int EPI, int NS = Tile<TMB, WM, WN>::NSTAGE>
__device__ __forceinline__ void gemm256_block(const GemmArgs &g, const int block, char *smem) {
    typedef Tile<TMB, WM, WN> TL;
    constexpr bool M_KS = WG;
    constexpr int Q_BM = TL::BM, Q_BN = TL::BN, TMW = TL::TMW;
    // ---- which tile am I?  Blocks are dealt round-robin to the 8 XCDs (block b runs on XCD b mod 8):
    //      give each XCD a contiguous range of the REAL tiles, so that neighbours share operands in
    //      its L2 and every XCD gets the same share.  For row-ragged products the number of real
    //      tiles is only known here (the grid is sized for the worst case), hence the device-side sum.
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int n_tiles = (g.N + Q_BN - 1) / Q_BN;
    int sum_nt = 0, sum_mt = 0;   // weight gradients: the n-tile / m-tile whose block also sums the m-side / n-side operand
    // a contraction split over blocks: the planes of an m-tile's n-tiles are numbered like more n-tiles
    const int n_units = EPI == EPI_PART ? n_tiles * g.ksplit : n_tiles;
    int split_k = 0;
    int e, mt, nt, m_ext, k_ext, tile_h = Q_BM;   // tile_h: rows of this tile's m-tiles (row-ragged products cut experts evenly)
    long row0;  // first row of the expert
    if constexpr (!WG) {
        // An expert with r rows is cut into t = ceil(r / BM) m-tiles.  Where a launch is a single round of
        // tiles (the 320-row configuration of the two K = F products) they have equal height h = r / t
        // rounded up to whole 32-row blocks, so that no expert leaves a short remainder tile behind, which
        // would run as a second, nearly empty round; elsewhere they are BM rows high and the last one is
        // the remainder, which costs fewer MFMA blocks in total and fills in among the many rounds.  The
        // m-tiles of all experts are numbered in expert order and each XCD takes a contiguous range of the
        // real (m-tile, n-tile) pairs, so that neighbours share operands in its L2 and every XCD gets the
        // same share; their number is only known here (the grid is sized for the worst case).
        const bool single = g.offsets == nullptr;
        auto rows_of = [&](int ee) { return single ? g.single_rows : g.kept[ee]; };
        const int nE = single ? 1 : g.E;
        // Rows and first row of the first 256 experts, fetched together (lane l holds experts l, l + 64, l + 128,
        // l + 192): the lookups below then need no further loads.  Fetched where they were needed, each pass of the
        // search below and the two lookups after it waited for memory in turn - four to five dependent round trips
        // per tile for experts past the 64th, half of a tile's fixed cost with 256 experts and a contraction of 1024.
        // (Beyond 256 experts the rest is read through the cache as before.)
        // A block has nothing to run beside this search: its time is the tile's.  What up to 64 experts need stands first and straight: one
        // scan a class that serves the totals and the search, one division.  On tiles of 128 x 128, 16 experts, the search 1.65 -> 1.15 us of a
        // block's 10 to 16: h of 128 rows, 512 -> 1408 11.9 -> 11.2 us, out 15.3 -> 14.8; h of 256, 512 -> 1024 12.4 -> 11.8; passes of 3001
        // tokens, top-2 of 16, 1024 -> 4096 -1 %, of 256, top-8 of 256, -1.5 %.
        constexpr int RC = 4;
        const bool many = nE > WAVE;
        int rows_c[RC], off_c[RC];
        rows_c[0] = lane < nE ? rows_of(lane) : 0;
        off_c[0] = !single && lane < nE ? g.offsets[lane] : 0;
#pragma unroll
        for (int c = 1; c < RC; ++c) rows_c[c] = off_c[c] = 0;
        if (many) {
#pragma unroll
            for (int c = 1; c < RC; ++c) {
                const int ee = lane + WAVE * c;
                rows_c[c] = ee < nE ? rows_of(ee) : 0;
                off_c[c] = !single && ee < nE ? g.offsets[ee] : 0;
            }
        }
        auto rows_at = [&](int ee) {            // rows of expert ee = base + lane of the caller's pass (ee uniform in ee / 64), from the 65th on
            int r = 0;
#pragma unroll
            for (int c = 1; c < RC; ++c)
                if ((ee >> 6) == c) r = rows_c[c];
            return (ee >> 6) < RC ? r : (ee < nE ? rows_of(ee) : 0);
        };
        // An expert's m-tiles are heavy (more than half a tile of rows) or light: the full tiles and, of the
        // remainder scheme, a remainder above half a tile; with the even split all tiles of an expert alike.
        // Heavy tiles are numbered before light ones, each class in expert order and each XCD taking a contiguous
        // range of either: an XCD hands out its blocks in order, so the long tiles start first and the short
        // ones fill in behind them (otherwise a long tile that starts late ends the launch late).
        // That order runs an expert's light tile long after its heavy ones, whose weight panels have left the L2 by
        // then; with many rounds of tiles the order matters little and the re-read does, so beyond 16 rounds
        // all tiles count as one class, in expert order.
        auto tiles_of = [&](int r) { return (r + Q_BM - 1) / Q_BM; };     // m-tiles of an expert with r rows
        bool split = true;
        auto heavy_of = [&](int r) {
            const int cnt = tiles_of(r);
            if (cnt == 0 || !split) return cnt;
            if (TMB == 10) return cnt > 1 || r > Q_BM / 2 ? cnt : 0;      // (two or more of equal height are above half a tile each)
            return cnt - 1 + ((r - (cnt - 1) * Q_BM) > Q_BM / 2 ? 1 : 0);
        };
        const int hv_0 = heavy_of(rows_c[0]), lt_0 = tiles_of(rows_c[0]) - hv_0;
        int incl_h = wave_scan(hv_0), incl_l = wave_scan(lt_0);
        int n_h = wave_total(incl_h), n_l = wave_total(incl_l);
        if (many) {
            int more_h = 0, more_l = 0;
            for (int ee = lane + WAVE; ee < nE; ee += WAVE) {
                const int r = rows_at(ee);
                const int hv = heavy_of(r);
                more_h += hv;
                more_l += tiles_of(r) - hv;
            }
            n_h += wave_total(wave_scan(more_h));
            n_l += wave_total(wave_scan(more_l));
        }
        if ((n_h + n_l) * n_units > 16 * 256) { split = false; n_h += n_l; n_l = 0; }
        const int total_h = n_h * n_units, total_l = n_l * n_units;
        const int per_h = (total_h + 7) >> 3, per_l = (total_l + 7) >> 3;
        const int slot = block >> 3, xcd = block & 7;
        const bool heavy = slot < per_h;
        const int t = heavy ? xcd * per_h + slot : xcd * per_l + (slot - per_h);
        if (heavy ? t >= total_h : (slot - per_h >= per_l || t >= total_l)) return;
        // Order of an XCD's tiles.  n-tile first: tile t = (m-tile t / n_tiles, n-tile t % n_tiles); the blocks that
        // run side by side on an XCD are then a few m-tiles times all n-tiles, i.e. they stream the expert's whole
        // weight matrix through the L2 once per group of m-tiles.  m-tile first (m_fastest): an expert's tiles are
        // numbered n-tile by n-tile, all its m-tiles of the class inside; the blocks side by side are then all
        // m-tiles of the expert times a few n-tiles, and every weight panel is fetched once.  In between (m_fastest =
        // G > 1): groups of G n-tiles with the expert's m-tiles inside, so that the 32 blocks of an XCD are about
        // 32 / G m-tiles times G n-tiles and fetch 32 / G + G panels between them instead of 1 + 32.  The two products
        // with a contraction over M and wide results (h = xd.w1^T + b1, t = (go.w2^T) gelu'(h)) use G = 8 for experts
        // of at least m_fastest_from = 8 m-tiles (8192 tokens, 64 experts of 2048 -> 8192, top-2, skewed loads: 798 ->
        // 766 and 777 -> 752 us); for experts of four or five m-tiles it is the slower order (16 experts of about 1024
        // rows, 1024 -> 4096: +6 and +3 us), so those keep n-tile first.
        const bool mf = g.m_fastest != 0;
        const int unit = mf ? n_tiles : 1;       // tiles per counted m-tile
        const int target = mf ? t : t / n_units;
        nt = t - target * n_units;               // (m-tile first: found below)
        // the expert whose running count (of the class) passes `target`
        int run = 0, base = 0;
        int cnt = heavy ? (split ? hv_0 : hv_0 + lt_0) : lt_0, incl = heavy ? (split ? incl_h : incl_h + incl_l) : incl_l;
        unsigned long long hit = __ballot(incl * unit > target);
        if (many) {
            while (!hit) {
                run += wave_total(incl);
                base += WAVE;
                if (base >= nE) break;
                const int r = rows_at(base + lane);
                const int hv = heavy_of(r);
                cnt = heavy ? hv : tiles_of(r) - hv;
                incl = wave_scan(cnt);
                hit = __ballot((run + incl) * unit > target);
            }
        }
        if (!hit) return;
        const int src = __ffsll(hit) - 1;
        e = base + src;
        const int c_e = __builtin_amdgcn_readlane(cnt, src);      // the expert's m-tiles of this class
        int mt_class = target - (run + __builtin_amdgcn_readlane(incl - cnt, src)) * unit;
        m_ext = __builtin_amdgcn_readlane(rows_c[0], src);
        int first_row = __builtin_amdgcn_readlane(off_c[0], src);
        if (many && base > 0) {
#pragma unroll
            for (int c = 1; c < RC; ++c)
                if (base == WAVE * c) { m_ext = __builtin_amdgcn_readlane(rows_c[c], src); first_row = __builtin_amdgcn_readlane(off_c[c], src); }
            if (base >= WAVE * RC) { m_ext = rows_of(e); first_row = g.offsets[e]; }
        }
        row0 = first_row;
        if (mf && c_e < g.m_fastest_from) {
            // an expert with few m-tiles keeps the n-tile-first order (its tiles are counted one by one here)
            const int m = mt_class / n_tiles;
            nt = mt_class - m * n_tiles;
            mt_class = m;
        } else if (mf) {
            // groups of G n-tiles, an expert's m-tiles of the class inside a group, the group's n-tiles innermost
            // (G = 1: m-tile first; the last group may be short)
            const int G = g.m_fastest;
            const int n_groups = (n_tiles + G - 1) / G;
            const int grp = min(mt_class / (c_e * G), n_groups - 1);
            const int j = mt_class - grp * c_e * G;
            const int gsz = min(G, n_tiles - grp * G);
            nt = grp * G + j % gsz;
            mt_class = j / gsz;
        }
        mt = mt_class + (heavy ? 0 : heavy_of(m_ext));   // an expert's light tiles follow its heavy ones
        const int t_e = (m_ext + Q_BM - 1) / Q_BM;
        tile_h = TMB == 10 ? ((((m_ext + t_e - 1) / t_e) + 31) & ~31) : Q_BM;
        k_ext = g.K;
        if constexpr (EPI == EPI_PART) {
            split_k = nt / n_tiles;
            nt %= n_tiles;
        }
    } else {
        // The contraction length differs from expert to expert, so experts are not handed to XCDs in
        // contiguous ranges: the (expert, m-tile) units are dealt round-robin over the 8 XCDs, which gives
        // every XCD the same share of every expert; the n-tiles of a unit stay together (they share the
        // m-side operand in that XCD's L2).
        // With hundreds of experts of many rows that spread costs more traffic than it is worth: the m-tiles of an expert
        // on different XCDs each fetch the expert's rows of the n-side operand into their own L2.  Then (wg_expert_major)
        // the experts are dealt round-robin instead, all blocks of one expert on one XCD.
        const int m_tiles = (g.M + Q_BM - 1) / Q_BM;
        const int slot = block >> 3;
        if (g.wg_expert_major) {
            const int u = slot / n_tiles;
            e = (u / m_tiles) * 8 + (block & 7);
            mt = u % m_tiles;
            if (e >= g.E) return;
        } else {
            const int unit = (slot / n_tiles) * 8 + (block & 7);
            if (unit >= g.E * m_tiles) return;
            e = unit / m_tiles;
            mt = unit % m_tiles;
        }
        nt = slot % n_tiles;
        // Blocks that also sum an operand run an eighth longer.  Consecutive slots of an XCD go to its four
        // shader engines in turn and are handed out in order, so an engine that always gets the long blocks
        // holds up the other three: the summing n-tile moves on from unit to unit, which gives every engine the
        // same number of long blocks in every round; the summing m-tile moves on from expert to expert, which
        // spreads those blocks over the XCDs.
        sum_nt = (slot / n_tiles) % n_tiles;
        sum_mt = e % m_tiles;
        m_ext = g.M;
        k_ext = g.kept ? g.kept[e] : g.single_rows;
        row0 = g.offsets ? g.offsets[e] : 0;
    }
    // the tile's coordinates are the same in every lane: say so, so that everything derived from them
    // (operand bases, LDS destinations, loop bounds) lives in scalar registers
    e = __builtin_amdgcn_readfirstlane(e);
    mt = __builtin_amdgcn_readfirstlane(mt);
    tile_h = __builtin_amdgcn_readfirstlane(tile_h);
    nt = __builtin_amdgcn_readfirstlane(nt);
    sum_nt = __builtin_amdgcn_readfirstlane(sum_nt);
    sum_mt = __builtin_amdgcn_readfirstlane(sum_mt);
    m_ext = __builtin_amdgcn_readfirstlane(m_ext);
    k_ext = __builtin_amdgcn_readfirstlane(k_ext);
    row0 = ((long)__builtin_amdgcn_readfirstlane((int)(row0 >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)row0);
    const int m0 = mt * tile_h, n0 = nt * Q_BN;
    if constexpr (WG && EPI == EPI_WGRAD) {
        if (k_ext == 0) {
            // An expert without rows: its gradient tile is zero (and adds nothing when sums are being built up).  The
            // zeros leave straight from registers - no operand ring, no LDS slab, no barrier (with skewed loads most experts of a
            // launch are such: 28 of 64 at 8192 tokens, top-2, Zipf(1.2)).  The m-tile's rows are one stretch of memory, of which
            // the blocks take equal pieces: tiles of a matrix whose rows are not whole lines share every line at their edges
            // (105 experts of 840 x 2520, 10 rows, the training pass: by tiles 386, this way 257 us).
            if (g.accumulate) return;
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            bf16_t *Cz = (bf16_t *)g.C + (long)e * g.strideC + (long)m0 * g.ldc;
            const long pieces = (long)min(Q_BM, m_ext - m0) * (g.N >> 3), lo = pieces * nt / n_tiles, hi = pieces * (nt + 1) / n_tiles;
            for (long u = lo + threadIdx.x; u < hi; u += TL::THREADS) __builtin_nontemporal_store(u32x4{0u, 0u, 0u, 0u}, reinterpret_cast<u32x4 *>(Cz) + u);
            if (g.colsum != nullptr) {
                bf16_t *out = (bf16_t *)g.colsum;
                const bf16_t z = (bf16_t)0.0f;
                if (g.colsum_side == 1 && nt == sum_nt) {
                    for (int r = threadIdx.x; r < Q_BM; r += TL::THREADS)
                        if (m0 + r < m_ext) out[(long)e * g.M + m0 + r] = z;
                } else if (g.colsum_side == 2 && mt == sum_mt) {
                    for (int c = threadIdx.x; c < Q_BN; c += TL::THREADS)
                        if (n0 + c < g.N) out[(long)e * g.N + n0 + c] = z;
                }
            }
            return;
        }
    }
    // h = xd.w1^T + b1 may read its rows where the tokens lie (a forward pass that nobody asks for xd)
    constexpr bool MAY_GATHER = EPI == EPI_BIAS_GELU;
    const int32_t *src = nullptr;
    if constexpr (MAY_GATHER) { if (g.token_of != nullptr) src = g.token_of + row0 + m0; }
    const bf16_t *Mp = (const bf16_t *)g.A + (src != nullptr ? 0 : row0 * g.lda);
    if constexpr (WG && EPI == EPI_WGRAD) {
        // Up to FEW_ROWS rows: every wave by itself, 128 columns by 64 rows of the tile (128-wide tiles: by 32); see wgrad_few.h.
        if (k_ext <= FEW_ROWS) {
            constexpr int COLS = Q_BN / 128, VM = Q_BM / 16 / (TL::NW / COLS);     // the block's waves along n; columns of a lane on the m-side
            const int w = __builtin_amdgcn_readfirstlane(wave), m_few = m0 + w / COLS * (16 * VM), n_few = n0 + w % COLS * 128;
            const bf16_t *Bp = (const bf16_t *)g.B + row0 * g.ldb;
            bf16_t *Cb = (bf16_t *)g.C + (long)e * g.strideC, *sums = nullptr;
            int side = 0;
            if (g.colsum != nullptr && g.colsum_side == 1 && nt == sum_nt && w % COLS == 0) { side = 1; sums = (bf16_t *)g.colsum + (long)e * g.M; }
            if (g.colsum != nullptr && g.colsum_side == 2 && mt == sum_mt && w / COLS == 0) { side = 2; sums = (bf16_t *)g.colsum + (long)e * g.N; }
            if (k_ext <= 32) {
                if (g.accumulate) few_rows_tile<VM, 8, 1, true>(g, Mp, Bp, Cb, sums, side, m_few, n_few, k_ext);
                else few_rows_tile<VM, 8, 1, false>(g, Mp, Bp, Cb, sums, side, m_few, n_few, k_ext);
            } else {
                if (g.accumulate) few_rows_tile<VM, 8, 2, true>(g, Mp, Bp, Cb, sums, side, m_few, n_few, k_ext);
                else few_rows_tile<VM, 8, 2, false>(g, Mp, Bp, Cb, sums, side, m_few, n_few, k_ext);
            }
            return;
        }
    }
    const bf16_t *Np = WG ? (const bf16_t *)g.B + row0 * g.ldb : (const bf16_t *)g.B + (long)e * g.strideB;
    if constexpr (EPI == EPI_PART) {           // this block's whole stages of the contraction (the last plane has the ragged end)
        split_k = __builtin_amdgcn_readfirstlane(split_k);
        const int stages = (k_ext + Q_BK - 1) / Q_BK;
        const int k_lo = split_k * stages / g.ksplit * Q_BK, k_hi = min((split_k + 1) * stages / g.ksplit * Q_BK, k_ext);
        Mp += k_lo;
        Np += N_KS ? (long)k_lo * g.ldb : (long)k_lo;
        k_ext = k_hi - k_lo;
    }

    f32x4 acc[2 * TMW][4];
    const int live = min(tile_h, m_ext - m0);
    const int tmc = (live + 31) >> 5;
    const int wu = __builtin_amdgcn_readfirstlane(wave);
    const int wm = wu / WN, wn = wu % WN;     // wave row / wave column
    uint2 bias_raw[4];
    load_bias<EPI>(g, e, n0, lane, wn, bias_raw);
    // Operand sums ride along in the weight-gradient blocks that see the whole operand once: one n-tile
    // of every m-tile for the m-side, one m-tile of every n-tile for the n-side.  These blocks run the
    // full tile shape (blocks past the operand's end repeat its last row and are not stored).
    int sum_side = 0;
    if constexpr (WG && WM == 2 && TMW <= WN) {
        if (g.colsum != nullptr && ((g.colsum_side == 1 && nt == sum_nt) || (g.colsum_side == 2 && mt == sum_mt))) sum_side = g.colsum_side;
    }
    // The live blocks are dealt evenly to the wave rows: c to each (the last row may find fewer live).
    const int c = sum_side ? TMW : (tmc + WM - 1) / WM;
    const int m0w = m0 + wm * c * 32, live_w = max(0, min(live - wm * c * 32, c * 32));
    // K loop and epilogue with C blocks per wave row
    f32x4 sums[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#define MOLE_RUN_TILE_AS(C, SUM, ONCE)                                                                                         \
    {                                                                                                                     \
        main_loop<TMB, WM, WN, NS, M_KS, N_KS, KT, WM *(C), (C), SUM, ONCE, (EPI > EPI_NONE ? EPI - EPI_NONE : 0), (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU)>(Mp, g.lda, m0, m_ext, Np, g.ldb, n0, g.N, k_ext, smem, wu, wm, wn, acc, sums, bias_raw, src, g.tokens); \
        if constexpr (SUM != 0) store_sums<SUM, (C)>(g, sums, e, m0, n0, m_ext, wm, wn, lane);                            \
        epilogue<TMB, WM, WN, WG, EPI, (C), KT && !WG>(g, acc, smem, lane, wu, wn, e, row0, m0w, n0, m_ext, live_w, split_k);      \
    }
#define MOLE_RUN_TILE_SUM(C, SUM) MOLE_RUN_TILE_AS(C, SUM, false)
#define MOLE_RUN_TILE(C) MOLE_RUN_TILE_AS(C, 0, false)
    if constexpr (WG && WM == 2 && TMW <= WN) {
        if (sum_side == 1) { MOLE_RUN_TILE_SUM(TMW, 1) return; }
        if (sum_side == 2) { MOLE_RUN_TILE_SUM(TMW, 2) return; }
    }
    if constexpr (N_KS && !WG && TMB >= 8) {
        // The only m-tile of an expert with few rows: its weights pass by once, and the launch is their stream.  (256 experts
        // of 1024 -> 2048 with 8 rows each, 1.07 GB: 197 -> 180 us; 149 of 1536 -> 1536, 17 rows: 143 -> 133.)
        if (g.once && m_ext <= 64) { MOLE_RUN_TILE_AS(1, 0, true) return; }
        if (g.once && m_ext <= 128) { MOLE_RUN_TILE_AS(2, 0, true) return; }
    }
    if (c >= TMW) MOLE_RUN_TILE(TMW)
    else if (TMW > 4 && c == 4) MOLE_RUN_TILE(TMW > 4 ? 4 : 1)
    else if (TMW > 3 && c == 3) MOLE_RUN_TILE(TMW > 3 ? 3 : 1)
    else if (TMW > 2 && c == 2) MOLE_RUN_TILE(TMW > 2 ? 2 : 1)
    else MOLE_RUN_TILE(1)
#undef MOLE_RUN_TILE
#undef MOLE_RUN_TILE_SUM
#undef MOLE_RUN_TILE_AS
}

template <int TMB, int WM, int WN, bool N_KS, bool WG, bool KT, int EPI>
__global__ __launch_bounds__((Tile<TMB, WM, WN>::THREADS), (Tile<TMB, WM, WN>::WAVES_PER_SIMD)) void gemm256_kernel(const GemmArgs g) {
    extern __shared__ __align__(16) char smem[];
    gemm256_block<TMB, WM, WN, N_KS, WG, KT, EPI>(g, blockIdx.x, smem);
}

// Two products of the backward pass that do not need each other in one launch, on 128 x 128 tiles: the first `first` blocks a row-ragged
// one (t = (go.w2^T) gelu'(h), or gx = t.w1), the others a weight gradient (g_w2 beside the former, g_w1 beside the latter).  On
// their own the row-ragged product of a small layer is a round of tiles that leaves half of the block slots empty and lasts as long as
// one block's chain of waits, and the weight gradient many short blocks that fill just such holes.  The long blocks start first.
// Bound by latency.  Training passes, apart / together: 2 x 513 tokens, 16 experts top-4, 520 -> 1416, 366 / 322 us; 2 x 130, 6 of 824 -> 824,
// top-6, skewed, 300 / 255; 2048 tokens, 16 of 512 -> 1024, top-2, 119 / 113.5.
// NS: stages of the ring, five in two blocks to a CU or three in three.
template <bool N_KS, bool KT, int EPI, int NS>
__global__ __launch_bounds__((Tile<4, 2, 2>::THREADS), (NS == 3 ? 3 : Tile<4, 2, 2>::WAVES_PER_SIMD)) void gemm256_pair_kernel(const GemmArgs g, const GemmArgs w, int first) {
    extern __shared__ __align__(16) char smem[];
    if ((int)blockIdx.x < first) gemm256_block<4, 2, 2, N_KS, false, KT, EPI, NS>(g, blockIdx.x, smem);
    else gemm256_block<4, 2, 2, true, true, true, EPI_WGRAD, NS>(w, (int)blockIdx.x - first, smem);
}

template <int TMB, int WM, int WN, bool N_KS, bool WG, bool KT, int EPI>
static int launch256_kt(GemmArgs g, int tiles, hipStream_t st, int kid) {
    typedef Tile<TMB, WM, WN> TL;
    if (tiles <= 0) return 0;
    g.n_blocks = tiles;
    const int grid = (tiles + 7) & ~7;
    auto kern = gemm256_kernel<TMB, WM, WN, N_KS, WG, KT, EPI>;
    static bool attr_done = false;
    if (!attr_done) {
        MOLE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, TL::LDS_BYTES));
        attr_done = true;
    }
    timed_launch(kid, kern, dim3(grid), dim3(TL::THREADS), TL::LDS_BYTES, st, g);
    MOLE_LAUNCH_CHECK();
    return 0;
}

// (the weight gradients' contraction is always ragged; the others have a kernel of their own for a K that is not whole
// stages, so that whole-stage ones carry no clamped offsets)
template <int TMB, int WM, int WN, bool N_KS, bool WG, int EPI>
static int launch256(const GemmArgs &g, int tiles, hipStream_t st, int kid) {
    if constexpr (WG) return launch256_kt<TMB, WM, WN, N_KS, WG, true, EPI>(g, tiles, st, kid);
    else if constexpr (EPI >= EPI_NONE) return launch256_kt<TMB, WM, WN, N_KS, WG, false, EPI>(g, tiles, st, kid);
    else return g.K % Q_BK ? launch256_kt<TMB, WM, WN, N_KS, WG, true, EPI>(g, tiles, st, kid) : launch256_kt<TMB, WM, WN, N_KS, WG, false, EPI>(g, tiles, st, kid);
}

// Launch options and their defaults; a -DMOLE_TUNING build reads them from the environment
// (MOLE_MFAST: bit mask of the products that number an expert's tiles m-tile first within groups of MOLE_MFAST_G
// n-tiles, MOLE_MFAST_FROM: m-tiles an expert needs for that order,
// MOLE_NO_SUMS: bias gradients from their own kernel).
#ifdef MOLE_TUNING
static int env_int(const char *name, int dflt) { const char *v = getenv(name); return v ? atoi(v) : dflt; }
static int m_fastest_mask() { static const int v = env_int("MOLE_MFAST", 9); return v; }
static int m_fastest_group() { static const int v = env_int("MOLE_MFAST_G", 8); return v > 0 ? v : 1; }
static int m_fastest_from() { static const int v = env_int("MOLE_MFAST_FROM", 8); return v; }
static bool sums_off() { static const bool v = getenv("MOLE_NO_SUMS") != nullptr; return v; }
#else
static int m_fastest_mask() { return 9; }        // h = xd.w1^T + b1 and t = (go.w2^T) gelu'(h)
static int m_fastest_group() { return 8; }
static int m_fastest_from() { return 8; }
static bool sums_off() { return false; }
#endif

// Blocks of a row-ragged launch: the worst-case number of m-tiles (an expert with r rows has ceil(r / BM) of them); + 16, as the heavy
// and the light tiles of an XCD are rounded up to whole slots separately.  A multiple of 8.
static int ragged_blocks(const GemmArgs &g, int epi, int rows_bound, int BM, int n_tiles) {
    const int m_bound = rows_bound / BM + (g.offsets ? min(g.E, rows_bound) : 1);
    return ((m_bound * n_tiles * (epi == EPI_PART ? g.ksplit : 1) + 7) & ~7) + 16;
}
// ... of a weight gradient by whole (expert, m-tile) units per XCD
static int wgrad_blocks(const GemmArgs &g, int BM, int n_tiles) { return 8 * ceil_div(g.E * ceil_div(g.M, BM), 8) * n_tiles; }

template <int TMB, int WM, int WN>
static int dispatch256(const GemmArgs &g, bool b_ks, bool wg, int epi, int max_rows, hipStream_t st, int kid) {
    constexpr int BM = Tile<TMB, WM, WN>::BM;
    const int n_tiles = ceil_div(g.N, (Tile<TMB, WM, WN>::BN));
    if constexpr (TMB == 8 || TMB == 4) {
        if (wg) {
            // All blocks of an expert on one XCD from 128 experts of 768 rows on: 256 experts of 2048 x 1024, 1024 rows each,
            // the training step 8624 against 8788 us.  With fewer rows it gains nothing (256 rows each: 482 against 486 us a
            // product) and loses under skewed loads, where a few XCDs get the large experts (Zipf(1.2): 755 against 516 us).
            GemmArgs gw = g;
            gw.wg_expert_major = g.E >= 128 && g.est_rows / g.E >= 768;
            // whole (expert, m-tile) units per XCD, or whole experts
            const int tiles = gw.wg_expert_major ? 8 * ceil_div(g.E, 8) * ceil_div(g.M, BM) * n_tiles : wgrad_blocks(g, BM, n_tiles);
            if (epi == EPI_WGRAD) return launch256<TMB, WM, WN, true, true, EPI_WGRAD>(gw, tiles, st, kid);
            return -100;
        }
    }
    const int rows_bound = g.offsets ? max_rows : g.single_rows;
    GemmArgs gg = g;
    gg.m_fastest = ((m_fastest_mask() >> kid) & 1) ? m_fastest_group() : 0;
    gg.m_fastest_from = m_fastest_from();
    const int tiles = ragged_blocks(g, epi, rows_bound, BM, n_tiles);
    if (wg) return -100;
    if (!b_ks) {
        if constexpr (TMB != 10) {
            if (epi == EPI_DGELU) return launch256<TMB, WM, WN, false, false, EPI_DGELU>(gg, tiles, st, kid);
            if (epi == EPI_BIAS_GELU) return launch256<TMB, WM, WN, false, false, EPI_BIAS_GELU>(gg, tiles, st, kid);
            if constexpr (TMB == 8) if (epi == EPI_F32) return launch256<TMB, WM, WN, false, false, EPI_F32>(gg, tiles, st, kid);
            if constexpr (TMB == 8) if (epi == EPI_NONE) return launch256<TMB, WM, WN, false, false, EPI_NONE>(gg, tiles, st, kid);
#ifdef MOLE_TUNING
            if constexpr (TMB == 8 && WM == 2 && WN == 4) {     // the loop's parts are probed at the default tile shape only
                if (epi == EPI_NONE + 1) return launch256<TMB, WM, WN, false, false, EPI_NONE + 1>(gg, tiles, st, kid);
                if (epi == EPI_NONE + 2) return launch256<TMB, WM, WN, false, false, EPI_NONE + 2>(gg, tiles, st, kid);
                if (epi == EPI_NONE + 3) return launch256<TMB, WM, WN, false, false, EPI_NONE + 3>(gg, tiles, st, kid);
                if (epi == EPI_NONE + 4) return launch256<TMB, WM, WN, false, false, EPI_NONE + 4>(gg, tiles, st, kid);
            }
#endif
        }
    } else {
        if (epi == EPI_BIAS) return launch256<TMB, WM, WN, true, false, EPI_BIAS>(gg, tiles, st, kid);
        if (epi == EPI_STORE) return launch256<TMB, WM, WN, true, false, EPI_STORE>(gg, tiles, st, kid);
        if (epi == EPI_PART) return launch256<TMB, WM, WN, true, false, EPI_PART>(gg, tiles, st, kid);
    }
    return -100;
}

// Tile configuration.  Eight waves (two per SIMD hide each other's waits; one fetch of the n-side tile
// serves all rows of the tile) for every product of some size.  256-row tiles by default; tiles of up to 320 rows, an
// expert's rows split evenly over them, for the two K = F products (out = a.w2 + b2 and gx = t.w1) where they need fewer
// rounds of tiles: with about 1024 rows an expert and a capacity factor of 1.25 they are one round where 256-row tiles
// are two (16 experts, 1024 -> 4096: 126 against 163 us).  Where the rounds are the same the smaller tile is the faster
// (6 experts of 1333 rows, 1088 -> 4352: 86 against 108 us).  The K = M products run several rounds anyway; their short
// remainder tiles, numbered last, fill the final round, which measured better than the even split
// (t = (go.w2^T) gelu'(h): 213 against 219 us) - and h = xd.w1^T + b1 with the GELU epilogue would spill at
// the 160 accumulators of the larger tile.
//
// Launches whose large tiles do not fill the chip once:
//   * K = F products with a long contraction split it over blocks (planes of fp32 partial results in the caller's workspace,
//     added by plane_reduce_kernel) as often as the tiles fit the chip, four times at most: every further plane costs its
//     write and its read.  out, reduction included: 16 experts of 375 rows, 1024 -> 4096: 81 -> 68 us in two planes; of 125
//     rows: 79 -> 46 in four; 8 experts of 250 rows, 2048 -> 8192: 184 -> 103 in four.
//   * the others run 128 x 128 tiles of four waves, two blocks to a CU, up to 112 large tiles (16 experts of 256 rows,
//     512 -> 1024: h 20.9 -> 14.7 us, out 26 -> 14); with more, their operand bytes per flop cost more than the idle CUs
//     (16 experts of 375 rows, 1024 -> 4096: h 109 against 83 us).  Their K = F products are split as well while the tiles
//     leave CUs idle (8 experts of 194 rows, 512 -> 2048: out 25 -> 16 us).
enum { TILE_256, TILE_320, TILE_128 };
struct TilePlan { int tile, ksplit; };
static TilePlan tile_plan(int E, int est_rows, int N, int K, bool tall) {
    TilePlan p{TILE_256, 1};
    const int active = E < est_rows ? E : est_rows;
    if (active <= 0) return p;
    // rows of an expert if they spread evenly, and of a fuller one (two standard deviations of a random routing)
    const int avg = ceil_div(est_rows, active);
    int full = avg;
    while ((full - avg) * (full - avg) < 4 * avg) ++full;
    const int n_tiles = ceil_div(N, 256), c256 = ceil_div(full, 256), c320 = ceil_div(full, 320);
    const long t256 = (long)active * c256 * n_tiles, t320 = (long)active * c320 * n_tiles;
    const bool few = (long)active * ceil_div(avg, 256) * n_tiles < 112;
    if (!tall) {
        if (few) p.tile = TILE_128;
        return p;
    }
    p.tile = (t256 + 255) / 256 > (t320 + 255) / 256 ? TILE_320 : TILE_256;
    if (K >= 3072 || (K >= 2048 && full <= 192)) {
        const long fit = 256 / t320;
        if (fit >= 2) {
            p.ksplit = fit < 4 ? (int)fit : 4;
            p.tile = c256 > c320 ? TILE_320 : TILE_256;
        }
    } else if (few) {
        p.tile = TILE_128;
        const long t128 = (long)active * ceil_div(full, 128) * ceil_div(N, 128);
        const long fit = 256 / t128, most = K / 512;
        p.ksplit = (int)(fit < most ? fit : most);
        p.ksplit = p.ksplit < 1 ? 1 : (p.ksplit > 4 ? 4 : p.ksplit);
    }
    return p;
}
// Weight gradients.  A CU pair of 128 x 128 blocks does 0.6-0.65 of the work of a 256 x 256 block in half the time of one
// (its operands cross LDS once per 128 rows instead of 256: 16 experts of 1024 x 4096, 512 rows each, 109 against 88 us),
// but wastes less where the large tiles do not fit the matrix or the last round of them is nearly empty: a round of
// 256 large tiles costs what 768 small ones do.  128 x 128 against 256 x 256: 16 experts of 520 x 1416, 128 rows, 17 / 22 us;
// 512 x 512, 1000 rows, 20 / 30; 4 of 512 x 2048, 500 rows, 13 / 19; 63 of 384 x 1536, 344 rows, 55 / 58; on the other
// side of the line 8 experts of 1024 x 3072, 500 rows, 44 / 41; 123 of 256 x 512, 325 rows, 29 / 27.
// Launches of experts with up to 24 rows are a stream of results (see wgrad_few.h), which two 128 x 128 blocks to a CU keep up where
// one of twice the waves leaves it between blocks: 128 x 128 / 256 x 256, 1 to 24 rows an expert, 200 of 384 x 768, 22 / 24 us; 64 of 1024 x
// 2048, 58 / 60 and 91 / 98 where the results are added to; 12 of 1344 x 2688, 16 / 19; 16 of 1024 x 4096, 27 / 28.  With more rows skewed
// loads leave enough to the experts above FEW_ROWS for the large tiles (64 of 1024 x 2048, 32 rows, Zipf(1.2): 71 / 67), and more than
// 2^15 blocks are slower to hand out (64 of 2048 x 8192: 405 / 385).
static int wgrad_tile(int E, int est_rows, int M, int N) {
    const long t256 = (long)E * ceil_div(M, 256) * ceil_div(N, 256), t128 = (long)E * ceil_div(M, 128) * ceil_div(N, 128);
    const int active = E < est_rows ? E : est_rows;
    if (active > 0 && est_rows <= 24l * active && t128 <= 32768) return TILE_128;
    return t128 < 768 * ((t256 + 255) / 256) ? TILE_128 : TILE_256;
}
int gemm256_ksplit(int E, int est_rows, int N, int K) { return tile_plan(E, est_rows, N, K, true).ksplit; }

// Whether the weight-gradient launch for g will also produce the operand sums asked for in g.colsum.
bool gemm256_sums_operand(const GemmArgs &g) {
    if (g.lda % 8 || g.ldb % 8 || g.ldc != g.N || g.N % 8 || g.M % 8) return false;
    return !sums_off();
}

// alignment the direct-to-LDS path relies on: 16-byte rows and pieces of K; weight gradients whose rows follow one another
static bool aligned256(const GemmArgs &g, bool a_ks, bool b_ks, bool wg) {
    if (g.lda % 8 || g.ldb % 8 || g.ldc % 8 || g.N % 8) return false;
    return wg ? a_ks && b_ks && g.M % 8 == 0 && g.ldc == g.N : !a_ks && g.K % 8 == 0;
}
// the tile of a row-ragged product; where its contraction is split, gp and epi become those of the planes
static int plan256(GemmArgs &gp, bool b_ks, int &epi, int max_rows, void *ws, size_t ws_bytes) {
    TilePlan p{TILE_256, 1};
    if (gp.offsets != nullptr && epi < EPI_NONE) p = tile_plan(gp.E, gp.est_rows, gp.N, gp.K, b_ks);
    p.ksplit = planes_allowed(p.ksplit, max_rows, gp.est_rows, gp.N);
    gp.ksplit = 1;
    if (p.ksplit > 1 && b_ks && ws != nullptr && ws_bytes >= (size_t)p.ksplit * max_rows * gp.N * sizeof(float)) {
        gp.ksplit = p.ksplit;
        gp.part = (float *)ws;
        gp.part_rows = max_rows;
        epi = EPI_PART;
    }
    return p.tile;
}

template <bool N_KS, bool KT, int EPI, int NS = Tile<4, 2, 2>::NSTAGE> static int launch_pair_kt(const GemmArgs &g, const GemmArgs &w, int max_rows, hipStream_t st, int kid) {
    typedef Tile<4, 2, 2> TL;
    const int first = ragged_blocks(g, EPI, max_rows, TL::BM, ceil_div(g.N, TL::BN)), rest = wgrad_blocks(w, TL::BM, ceil_div(w.N, TL::BN));
    auto kern = gemm256_pair_kernel<N_KS, KT, EPI, NS>;
    constexpr int lds = NS * TL::STAGE > TL::SLABS ? NS * TL::STAGE : TL::SLABS;
    static bool attr_done = false;
    if (!attr_done) {
        MOLE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        attr_done = true;
    }
    timed_launch(kid, kern, dim3(first + rest), dim3(TL::THREADS), lds, st, g, w, first);
    MOLE_LAUNCH_CHECK();
    return 0;
}
// Whether t and g_w2 take three blocks to a CU, with rings of three stages: t walks over K = M, few stages beside gx's K = F, and a third block can
// count for more than stages in flight.  It does where t's tiles are more than the CUs (256) and all of them at least two and a half a CU (640).
// M of whole stages: of 51 such training passes of random sizes 36 were 0.2 to 4 % faster with it and seven up to 0.7 % slower, 1 % in the mean.  us, two blocks / three, t's
// tiles and all: 2048 tokens of the padded layout, 16 experts of 512 -> 1024 (320, 832) 102.6 / 101.4; 429, top-4 of 4, 640 -> 2560 (308, 708) 120.0 / 117.2; 2 x 3923,
// top-2 of 14, 1024 -> 512 (273, 721) 339.1 / 329.5; 1361, top-4 of 12, 320 -> 960 (388, 676) 105.9 / 103.7; near the first bound 571, top-8 of 22, 384 -> 768 (280, 676)
// 99.1 / 99.8, 2333, 12 of 448 -> 1344 (266, 794) 109.5 / 108.7.  Not with fewer tiles of t (eight passes up to 2 % faster or slower, as often) or fewer than 540 in all (ten
// passes, 2.8 % slower in the mean: 12871, top-2 of 8, 512 -> 256 (410, 474) 193.3 / 200.1).
// M that ends inside a stage, whose stages take a third longer: where the weight gradient is added to what is there, for its blocks wait for the old values as well (27 passes of two micro-
// batches, 256 to 394 tiles of t: 23 are 0.3 to 5 % faster, four up to 1.5 % slower, 0.9 % in the mean; 2 x 490, 513 and 540 tokens, top-4 of 16, 520 -> 1416 (280, 288, 298) 286.5 / 285.6,
// 296.1 / 294.1, 304.6 / 297.3), and without that from 370 tiles of t on: 26 of 26 passes up to 487 are 0.3 to 5 % faster, 1.6 % in the mean (1522, top-8 of 16, 408 -> 408 (413, 669) 143.1 /
// 136.6; 404, 1052 in all, M = 328 144.5 / 141.0; 372, 980, M = 440 142.9 / 142.4).  From 300 to 370 eight of 25 are faster (345, 778, M = 712 166.2 / 163.8; 349, 1629, M = 904 188.3 / 191.9),
// below 300 three of 44 (261, 1661, M = 1264 187.1 / 191.9).  gx, whose walk is longer: 31.4 / 37.2 the launch of 2 x 513.
static bool three_blocks(int E, int est_rows, int F, int M, bool accumulate) {
    const int active = E < est_rows ? E : est_rows, n_tiles = ceil_div(F, 128);
    const double tiles = (est_rows / 128.0 + 0.5 * active) * n_tiles;      // (an expert's last one is half full in the mean)
    return tiles > 256.0 && (M % Q_BK == 0 || accumulate || tiles >= 370.0) && tiles + (double)E * n_tiles * ceil_div(M, 128) >= 640.0;
}
template <bool N_KS, int EPI> static int launch_pair(const GemmArgs &g, const GemmArgs &w, int max_rows, hipStream_t st, int kid) {
    if constexpr (EPI == EPI_DGELU) {
        if (three_blocks(g.E, g.est_rows, g.N, g.K, w.accumulate != 0))
            return g.K % Q_BK ? launch_pair_kt<N_KS, true, EPI, 3>(g, w, max_rows, st, kid) : launch_pair_kt<N_KS, false, EPI, 3>(g, w, max_rows, st, kid);
    }
    return g.K % Q_BK ? launch_pair_kt<N_KS, true, EPI>(g, w, max_rows, st, kid) : launch_pair_kt<N_KS, false, EPI>(g, w, max_rows, st, kid);
}
// The row-ragged product g (EPI_DGELU, or EPI_STORE with K-strided weights) and the weight gradient w together where both take 128 x 128
// tiles; -100 otherwise, and nothing is launched.
int launch_gemm256_pair(const GemmArgs &g, const GemmArgs &w, bool b_ks, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid) {
    if (!aligned256(g, false, b_ks, false) || !aligned256(w, true, true, true) || g.offsets == nullptr) return -100;
    GemmArgs gp = g;
    if (wgrad_tile(w.E, w.est_rows, w.M, w.N) != TILE_128 || plan256(gp, b_ks, epi, max_rows, ws, ws_bytes) != TILE_128) return -100;
    int rc;
    if (epi == EPI_DGELU) rc = launch_pair<false, EPI_DGELU>(gp, w, max_rows, st, kid);
    else if (epi == EPI_STORE) rc = launch_pair<true, EPI_STORE>(gp, w, max_rows, st, kid);
    else rc = launch_pair<true, EPI_PART>(gp, w, max_rows, st, kid);
    return rc != 0 || gp.ksplit == 1 ? rc : launch_plane_reduce(gp, MOLE_BF16, max_rows, st);
}

int launch_gemm256(const GemmArgs &g, bool a_ks, bool b_ks, bool wg, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid) {
    if (!aligned256(g, a_ks, b_ks, wg)) return -100;
    GemmArgs gp = g;
    TilePlan p{TILE_256, 1};
    if (!wg) p.tile = plan256(gp, b_ks, epi, max_rows, ws, ws_bytes);
    else {
        gp.ksplit = 1;
        if (epi == EPI_WGRAD) p.tile = wgrad_tile(g.E, g.est_rows, g.M, g.N);
    }
    int rc;
    if (p.tile == TILE_128) rc = dispatch256<4, 2, 2>(gp, b_ks, wg, epi, max_rows, st, kid);
    else if (p.tile == TILE_320) rc = dispatch256<10, 2, 4>(gp, b_ks, wg, epi, max_rows, st, kid);
    else rc = dispatch256<8, 2, 4>(gp, b_ks, wg, epi, max_rows, st, kid);
    return rc != 0 || gp.ksplit == 1 ? rc : launch_plane_reduce(gp, MOLE_BF16, max_rows, st);
}

}  // namespace mole

extern "C" int mole_probe_wgrad_tile(int E, int est_rows, int M, int N) { return mole::wgrad_tile(E, est_rows, M, N) == mole::TILE_128 ? 128 : 256; }

extern "C" int mole_probe_pair_stages(int E, int est_rows, int M, int F, int accumulate) {
    if (mole::wgrad_tile(E, est_rows, F, M) != mole::TILE_128 || mole::tile_plan(E, est_rows, F, M, false).tile != mole::TILE_128) return 0;
    return mole::three_blocks(E, est_rows, F, M, accumulate != 0) ? 3 : mole::Tile<4, 2, 2>::NSTAGE;
}
