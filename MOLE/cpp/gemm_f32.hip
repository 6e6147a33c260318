// fp32 grouped GEMM for gfx950: the fast path of the six expert-FFN products in the reference's own dtype
// (MOLE/cpp/define.hpp:152-155 - fp32 is the only type its kernels are instantiated for; the products are
// _BatchRecord::bffn_fwd / bffn_bwd, MOLE/cpp/core.cpp:344-356, 381-414).
//
// The products run on the bf16 matrix cores.  An fp32 number of 2^-110 or more is the sum of three bf16 numbers (8 + 8 + 8
// significand bits; bf16 ends at 2^-133), so a product is nine products of parts, of which the three smallest, together 2^-24
// of it at most and 2^-27 in the root mean square, are left out: six of v_mfma_f32_32x32x16_bf16, which takes 32 cycles for 16 of k, replace eight of
// v_mfma_f32_32x32x2_f32 of 64 each.
// Accuracy.  The matrix cores round to nearest, eight of k at a time in bf16 and one at a time in fp32, and cut off what lies far
// below the accumulator: 0.004 units of its last place an instruction, always downwards.  The products hi hi have an accumulator of
// their own, in which they are near its size; the five smaller ones go into a second, whose last place is 2^-8 of the first's, and
// the two are added once.  That leaves two roundings for 16 of k where fp32 operands take sixteen and no drift that the
// roundings do not cover, in one result or in a sum over many.  2-norm errors against 64 bits with fp32 operands / here, in 2^-24:
// 8 experts of 1000 rows, 512 -> 2048: h 6.8 / 2.2, out 7.9 / 2.8, weight gradients 9.6 and 11.8 / 3.4 and 3.8, bias gradient of
// b1 7.8 / 4.2; all operands positive: h 5.3 / 2.0, out 3.6 / 1.5, weight gradients 7.8 / 2.9; 2048 -> 4096, 300 rows, positive: h
// 10.3 / 3.7, mean error 0.04 / 0.03.  Only a sum of a single product would be no closer, 0.424 / 0.435: weight gradients of one row
// keep fp32 operands.  (One accumulator for all six: 0.75-0.9 of fp32 operands' error, but a drift of 0.02 units a stage.)
// A tile whose operands include a number below 2^-110 that is not zero, or whose results are not all finite, is computed again
// from fp32 operands.  All rows of a tile take the same steps, so equal rows give equal results.
// Time of launches one by one, fp32 operands / parts that every wave makes / parts that a block shares, on one box, us: 8 experts of 1000 rows, 512 -> 2048: h 154 / 128 / 128,
// out 135 / 115 / 106, t 154 / 125 / 127, gx 133 / 112 / 104, the weight gradients 136 / 108 each; 8 of 2000, 1024 -> 4096: 1036, 1004,
// 1047, 993, 1010 / 838, 756, 833, 750, 788.
//
// Three kinds of tile, chosen at the launch (f32_tile, f32_shares):
//   shared parts (shared_parts_loop): 128 x 128 by eight waves (2 x 4), a block to a CU.  What bounds the products by parts is that taking the operands
//     apart costs the VALU as long as the products take the matrix cores, and every number was taken apart by two or four waves; here by one.
//     The parts go through LDS, and the waves' reads of them take it as long again: the three overlap to 0.8 of the rate at which bf16
//     products run into the power limit (K = 4096: 1.72 us for 32 of k, of 1.4).  (Two blocks of four waves, each 64 x 64, with the parts
//     of one stage: no gain; 32 x 32 x 16 products, whose results a lane holds as 16 rows of a column: 5 % slower in all six products.)
//   own parts (f32_loop): 128 x 128 by four waves (2 x 2) or 64 x 128 (1 x 4), two or three blocks to a CU, which hide each other's ends: weight gradients,
//     whose contractions are short and whose outputs are long (by shared parts 1000 rows 8 % slower, 125 rows 48 %), and where the rule says.
//   fp32 operands (f32_loop): 64 x 128 where CUs have one block each.
// For the latter two, operand stages of 16 of K come as fp32 from HBM/L2 straight into a ring of four LDS stages (global_load_lds_dwordx4, one
// barrier per stage); the fragments of stage s + 1 are read and split while the MFMAs of stage s run.
//
// LDS images (the 16-byte piece a lane's load fills is fixed by the hardware; which global address it fetches
// is ours to choose, so any permutation of pieces is free):
//   * K-contiguous operand -> [row][4 x 16 B], piece index XORed with swz4(row); a ds_read_b128 gives a lane four
//     consecutive k of its row: k = 8 kk + j (lanes 0-31) and 8 kk + 4 + j (lanes 32-63) for piece kk, j < 4 - any order
//     of k is as good as any other as long as both operands use the same.
//   * K-strided operand    -> [k][rows x 4 B] as it lies in HBM, the 16-byte piece index XORed with 8 on k-rows with
//     bit 2 set (the two k-rows one MFMA step reads then fall into different banks).  A wave's two 32-row blocks are
//     the even and the odd rows of its 64: one ds_read_b64 per step serves both.
// Own parts: 32 x 32 blocks; the m-side operand feeds the MFMA's first slot and the n-side the second, so the 32 lanes of a half wave hold 32
// consecutive (or, K-strided, 64 consecutive in pairs) columns of one result row: stores are whole 128- or 256-byte
// row segments straight from the accumulators.  The others: 16 x 16 blocks, the n-side in the first slot, so a lane holds four columns
// of a row and bias, GELU and stores go by 16 bytes (fp32 operands, one 64-row tile to a CU, against 32 x 32 x 2 with the slots the other way:
// h of 64 rows x 8, 512 -> 2048 27.0 -> 24.1 us, 256 x 1, 256 -> 1024 17.6 -> 14.3, 128 x 16, 1024 -> 1024 47.2 -> 43.2, 27 x 6, 4096 -> 1216 129 -> 130).
#include "gemm.h"
#include "lds_dma.h"

#include <algorithm>
#include <cmath>
#include <type_traits>

namespace mole {
namespace {

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));       // a bias may lie anywhere

constexpr int F_BK = 16;          // k per stage: 64 bytes of a K-contiguous row
constexpr int P_BK = 32;          // k per stage of parts that the block shares

// How a tile's products are made: from fp32 operands; from parts that every wave makes of its own fragments; from parts that the
// block makes once and shares
enum How { OPERANDS, OWN_PARTS, SHARED_PARTS };

// NW waves; the MFMA blocks have EDGE rows and columns
template <int BM, int BN, int NSTAGE, int NW, How HOW> struct FTile {
    static constexpr int THREADS = 64 * NW, EDGE = HOW == OWN_PARTS ? 32 : 16;
    static constexpr int WM = BM / 64, WN = NW / WM;                        // waves along m and n
    static constexpr int TMW = 64 / EDGE, TNW = BN / WN / EDGE;             // blocks per wave on either side
    static constexpr int Q = EDGE * EDGE / 64;                              // results a lane holds of a block
    typedef float Acc __attribute__((ext_vector_type(Q)));
    static constexpr int M_BYTES = BM * F_BK * 4, N_BYTES = BN * F_BK * 4, STAGE = M_BYTES + N_BYTES;
    static constexpr int LM = BM / 16 / NW, LN = BN / 16 / NW, L = LM + LN;   // 1-KiB loads per wave and stage
    static constexpr int RING_BYTES = NSTAGE * STAGE;
};

// Per-lane byte offsets of the loads a wave issues for one stage of an operand tile, relative to the tile's first
// element at the stage's first k.  Wave w's load i fills LDS bytes [(NW i + w) 1024, +1024) of the tile.  Rows
// (k-rows) past the operand's end are clamped to the last valid one: what lands for them is finite data that only
// reaches results which are not stored - except along a ragged contraction, whose tail is zeroed in LDS.
// src: the operand's rows are those of a matrix of n_src rows that src names, and the base is that matrix (null: they lie there in order).
template <int ROWS, bool KS, int NW> struct FOff {
    static constexpr int NL = ROWS / 16 / NW;
    uint32_t off[NL];
    __device__ __forceinline__ void init(long ld, int r_left, int k_left, const int32_t *src = nullptr, int n_src = 0) {
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        uint32_t at[NL];
        if constexpr (!KS) {
#pragma unroll
            for (int i = 0; i < NL; ++i) {
                at[i] = (uint32_t)min((NW * i + w) * 16 + (lane >> 2), r_left - 1);
                if (src != nullptr) at[i] = min((uint32_t)src[at[i]], (uint32_t)n_src - 1u);
            }
        }
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            if constexpr (!KS) {
                const int row = (NW * i + w) * 16 + (lane >> 2);
                const int c = (lane & 3) ^ swz4(row);
                off[i] = (uint32_t)(at[i] * ld * 4 + c * 16);
            } else {
                constexpr int SPR = ROWS / 4, KPL = 64 / SPR;      // 16-byte pieces per k-row, k-rows per load
                const int kr = (NW * i + w) * KPL + lane / SPR;
                const int c = (lane % SPR) ^ (((kr >> 2) & 1) << 3);
                off[i] = (uint32_t)(min(kr, k_left - 1) * ld * 4 + min(c * 4, r_left - 4) * 4);
            }
        }
    }
};

// The fragments of one stage for the NB 32-row blocks of a wave on one side.  get(b, kk, j): the lane's operand
// register for block b in MFMA step (kk, j).
template <int ROWS, bool KS, int NB> struct FFrag {
    float v[8 * NB];
    __device__ __forceinline__ void read(const char *tile, uint32_t off0, uint32_t off1) {
        if constexpr (!KS) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int kk = 0; kk < 2; ++kk) {
                    const float4 t = *reinterpret_cast<const float4 *>(tile + (kk ? off1 : off0) + b * 2048);
                    v[(b * 2 + kk) * 4 + 0] = t.x; v[(b * 2 + kk) * 4 + 1] = t.y;
                    v[(b * 2 + kk) * 4 + 2] = t.z; v[(b * 2 + kk) * 4 + 3] = t.w;
                }
        } else {
#pragma unroll
            for (int kk = 0; kk < 2; ++kk)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const char *p = tile + off0 + (8 * kk + j) * (ROWS * 4);
                    if constexpr (NB == 2) {
                        const float2 t = *reinterpret_cast<const float2 *>(p);
                        v[(kk * 4 + j) * 2] = t.x; v[(kk * 4 + j) * 2 + 1] = t.y;
                    } else {
                        v[kk * 4 + j] = *reinterpret_cast<const float *>(p);
                    }
                }
        }
    }
    __device__ __forceinline__ float get(int b, int kk, int j) const {
        if constexpr (!KS) return v[(b * 2 + kk) * 4 + j]; else return v[(kk * 4 + j) * NB + b];
    }
    // per-lane LDS byte offsets inside the operand tile; blk0: the wave's first 32-row block
    static __device__ __forceinline__ void offsets(int blk0, uint32_t &off0, uint32_t &off1) {
        const int lane = threadIdx.x & 63, lr = lane & 31, h = lane >> 5;
        if constexpr (!KS) {
            const int row = blk0 * 32 + lr;
            const int c0 = h ^ swz4(row);          // swz4 does not depend on the block (bits 1-3 of the row)
            off0 = (uint32_t)(row * 64 + c0 * 16);
            off1 = (uint32_t)(row * 64 + (c0 ^ 2) * 16);
        } else {
            const int lb = (blk0 * 32 + NB * lr) * 4;                     // logical byte inside the k-row
            off0 = (uint32_t)(4 * h * (ROWS * 4) + ((((lb >> 4) ^ (h << 3)) << 4) | (lb & 15)));
            off1 = 0;
        }
    }
};

// The same for blocks of 16 rows: lane l holds row l % 16 and k-rows 4 (l / 16) + j of each.
template <int ROWS, bool KS, int NB> struct FFrag16 {
    float v[4 * NB];
    __device__ __forceinline__ void read(const char *tile, uint32_t off, uint32_t) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            if constexpr (!KS) {
                const float4 t = *reinterpret_cast<const float4 *>(tile + off + b * 1024);
                v[4 * b] = t.x; v[4 * b + 1] = t.y; v[4 * b + 2] = t.z; v[4 * b + 3] = t.w;
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j) v[4 * b + j] = *reinterpret_cast<const float *>(tile + off + b * 64 + j * (ROWS * 4));
            }
        }
    }
    __device__ __forceinline__ float get(int b, int, int j) const { return v[4 * b + j]; }
    static __device__ __forceinline__ void offsets(int blk0, uint32_t &off, uint32_t &) {
        const int lane = threadIdx.x & 63, i = lane & 15, kg = lane >> 4;
        static_assert(!KS || NB == 2, "a pair of blocks keeps its order where pieces are XORed with 8");
        if constexpr (!KS) off = (uint32_t)((blk0 * 16 + i) * 64 + ((kg ^ swz4(i)) << 4));
        else off = (uint32_t)(4 * kg * (ROWS * 4) + (blk0 ^ ((kg & 1) << 1)) * 64 + i * 4);
    }
};

// A fragment block (8 k of one row per lane) as three bf16 numbers a value: x = hi + mid + lo, each the rounding of what the ones
// before leave (8 + 8 + 8 significand bits are the 24 of fp32; exact from 2^-110 on).  A remainder is taken with
// plain additions on the unpacked parts, five instructions for a pair of values and a part: v_dot2_f32_bf16 would take three,
// but it runs on the matrix pipe (5 of them behind each of 24 MFMAs of 32 x 32 x 16: 357 -> 669 us; additions, shifts, masks
// and conversions: 331-379).
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
// least: the smallest of the numbers met so far, as the bits of its magnitude doubled, less one (zero: the largest)
__device__ __forceinline__ void split_pair(float r0, float r1, uint32_t (&part)[3], uint32_t &least) {
    const uint32_t u0 = (__float_as_uint(r0) << 1) - 1u, u1 = (__float_as_uint(r1) << 1) - 1u;
    asm("v_min3_u32 %0, %0, %1, %2" : "+v"(least) : "v"(u0), "v"(u1));
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(part[q]) : "v"(r0), "v"(r1));
        if (q < 2) {
            r0 -= __uint_as_float(part[q] << 16);
            r1 -= __uint_as_float(part[q] & 0xffff0000u);
        }
    }
}
struct Planes {
    u32x4 p[3];
    __device__ __forceinline__ void split(const float (&x)[8], uint32_t &least) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            uint32_t part[3];
            split_pair(x[2 * i], x[2 * i + 1], part, least);
#pragma unroll
            for (int q = 0; q < 3; ++q) p[q][i] = part[q];
        }
    }
    __device__ __forceinline__ bf16x8 part(int q) const { return __builtin_bit_cast(bf16x8, p[q]); }
};
// The smallest number whose three parts are sure to be exact: bf16 ends at 2^-133, 23 bits below it.
constexpr float PARTS_MIN = 0x1p-110f;
// the six of the nine products of two triples that fp32 accuracy needs, those of the last parts first
__device__ constexpr int SPLIT_M[6] = {0, 2, 1, 0, 1, 0}, SPLIT_N[6] = {2, 0, 1, 1, 0, 0};

// The K loop of one tile: acc += the products of its nk stages.  SPLIT: by the parts of the operands; returns whether this lane
// met an operand that has no exact parts.
template <int BM, int BN, int NSTAGE, int NW, How HOW, bool M_KS, bool N_KS, bool WG, bool SPLIT>
__device__ __forceinline__ bool f32_loop(const GemmArgs &g, const float *Mp, const float *Np, int m0, int n0, int m_ext, int k_ext, char *smem,
                                         int wave, int wm, int wn, typename FTile<BM, BN, NSTAGE, NW, HOW>::Acc (&acc)[FTile<BM, BN, NSTAGE, NW, HOW>::TMW][FTile<BM, BN, NSTAGE, NW, HOW>::TNW],
                                         int sum_side, float (&psum)[4][2], const int32_t *src) {
    typedef FTile<BM, BN, NSTAGE, NW, HOW> TL;
    static_assert(TL::EDGE == 32 || !(SPLIT || WG), "");
    constexpr int F_NSTAGE = NSTAGE;
    constexpr int TMW = TL::TMW, TNW = TL::TNW, L = TL::L;
    const int nk = (k_ext + F_BK - 1) / F_BK;
    if (nk <= 0) return false;
    const int kl = k_ext - (nk - 1) * F_BK;     // k-rows of the last stage (a row-ragged product's K is whole stages)
    FOff<BM, M_KS, NW> om, cm;
    FOff<BN, N_KS, NW> on, cn;
    om.init(g.lda, m_ext - m0, F_BK, src, g.tokens);
    on.init(g.ldb, g.N - n0, F_BK);
    if constexpr (WG) { cm.init(g.lda, m_ext - m0, kl); cn.init(g.ldb, g.N - n0, kl); }
    const char *bm = uniform_ptr(src != nullptr ? Mp : M_KS ? Mp + m0 : Mp + (long)m0 * g.lda);
    const char *bn = uniform_ptr(N_KS ? Np + n0 : Np + (long)n0 * g.ldb);
    const long step_m = M_KS ? g.lda * (F_BK * 4) : F_BK * 4;
    const long step_n = N_KS ? g.ldb * (F_BK * 4) : F_BK * 4;
    const uint32_t lds_w = lds_offset_of(smem) + wave * 1024;
    // load j of stage s (the m-side tile's loads come first) into ring buffer s mod NSTAGE; stages are issued in
    // order, the bases advance after a stage's last load
    auto issue_one = [&](int s, int j) __attribute__((always_inline)) {
        const uint32_t dst = lds_w + (s % F_NSTAGE) * TL::STAGE;
        const bool last = WG && s == nk - 1;
        if (j < TL::LM) {
            uint32_t o = om.off[j];
            if constexpr (WG) o = last ? cm.off[j] : o;
            dma16s(bm, o, dst + j * (NW * 1024));
        } else {
            uint32_t o = on.off[j - TL::LM];
            if constexpr (WG) o = last ? cn.off[j - TL::LM] : o;
            dma16s(bn, o, dst + TL::M_BYTES + (j - TL::LM) * (NW * 1024));
        }
        if (j == L - 1) { bm += step_m; bn += step_n; }
    };
    auto issue = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < L; ++j) issue_one(s, j);
    };
    // ragged contraction: zero the k-rows past its end in the last stage (both tiles are [k][rows] there)
    auto zero_tail = [&](int buf) __attribute__((always_inline)) {
        char *b = smem + buf * TL::STAGE;
        for (int idx = threadIdx.x; idx < (F_BK - kl) * (BM / 4); idx += TL::THREADS)
            *reinterpret_cast<float4 *>(b + kl * (BM * 4) + idx * 16) = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int idx = threadIdx.x; idx < (F_BK - kl) * (BN / 4); idx += TL::THREADS)
            *reinterpret_cast<float4 *>(b + TL::M_BYTES + kl * (BN * 4) + idx * 16) = make_float4(0.f, 0.f, 0.f, 0.f);
        __syncthreads();
    };
    uint32_t fm0, fm1, fn0, fn1;
    typedef std::conditional_t<TL::EDGE == 32, FFrag<BM, M_KS, TMW>, FFrag16<BM, M_KS, TMW>> MFrag;
    typedef std::conditional_t<TL::EDGE == 32, FFrag<BN, N_KS, TNW>, FFrag16<BN, N_KS, TNW>> NFrag;
    MFrag::offsets(wm * TMW, fm0, fm1);
    NFrag::offsets(wn * TNW, fn0, fn1);
    MFrag ma;
    NFrag na;

#pragma unroll
    for (int s = 0; s < F_NSTAGE - 1; ++s)
        if (s < nk) issue(s);
    if (F_NSTAGE == 4 && nk >= 3) __builtin_amdgcn_s_waitcnt(waitcnt_vm(2 * L));
    else if (nk >= 2) __builtin_amdgcn_s_waitcnt(waitcnt_vm(L));
    else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));
    __builtin_amdgcn_s_barrier();
    if (WG && nk == 1 && kl < F_BK) zero_tail(0);
    auto add_sums = [&]() __attribute__((always_inline)) {
        if constexpr (WG) {
            if (sum_side == 1) {
#pragma unroll
                for (int b = 0; b < TMW; ++b)
#pragma unroll
                    for (int i = 0; i < 8; ++i) psum[i & 3][b] += ma.get(b, i >> 2, i & 3);
            } else if (sum_side == 2) {
#pragma unroll
                for (int b = 0; b < TNW; ++b)
#pragma unroll
                    for (int i = 0; i < 8; ++i) psum[i & 3][b] += na.get(b, i >> 2, i & 3);
            }
        }
    };
    if constexpr (SPLIT) {
        Planes pa[TMW + TNW], pb[TMW + TNW];
        f32x16 low[TMW][TNW];           // the products below hi hi
#pragma unroll
        for (int i = 0; i < TMW; ++i)
#pragma unroll
            for (int j = 0; j < TNW; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) low[i][j][q] = 0.f;
        uint32_t least = 0xffffffffu;
        auto split_block = [&](Planes (&p)[TMW + TNW], int b) __attribute__((always_inline)) {      // m-blocks first
            float x[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) x[i] = b < TMW ? ma.get(b, i >> 2, i & 3) : na.get(b - TMW, i >> 2, i & 3);
            p[b].split(x, least);
            // (kept where it stands, among the MFMAs: left alone the compiler moves it to the use, a stage later)
            asm volatile("" : "+v"(p[b].p[0]), "+v"(p[b].p[1]), "+v"(p[b].p[2]));
        };
        ma.read(smem, fm0, fm1);
        na.read(smem + TL::M_BYTES, fn0, fn1);
        add_sums();
#pragma unroll
        for (int b = 0; b < TMW + TNW; ++b) split_block(pa, b);
#define MOLE_SPLIT_STAGE(S, PC, PN, NEXT)                                                                   \
        {                                                                                                   \
            const int s_ = (S);                                                                             \
            bool refill_ = false;                                                                           \
            const int nb_ = (s_ + 1) % F_NSTAGE;                                                            \
            if constexpr (NEXT) {                                                                           \
                if (F_NSTAGE == 4 && s_ + 2 < nk) __builtin_amdgcn_s_waitcnt(waitcnt_vm(L));                \
                else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));                                             \
                __builtin_amdgcn_s_barrier();                                                               \
                refill_ = s_ + F_NSTAGE - 1 < nk;                                                           \
                if (WG && s_ + 1 == nk - 1 && kl < F_BK) zero_tail(nb_);                                    \
                ma.read(smem + nb_ * TL::STAGE, fm0, fm1);                                                  \
                na.read(smem + nb_ * TL::STAGE + TL::M_BYTES, fn0, fn1);                                    \
            }                                                                                               \
            constexpr int CELLS_ = TMW * TNW;                                                               \
            _Pragma("unroll") for (int grp = 0; grp < 2; ++grp) {                                           \
                MOLE_SPLIT_MFMAS(PC, grp)                                                                   \
                if constexpr (NEXT) {                                                                       \
                    if (refill_) {                                                                          \
                        _Pragma("unroll") for (int j = grp * L / 2; j < (grp + 1) * L / 2; ++j) issue_one(s_ + F_NSTAGE - 1, j); \
                    }                                                                                       \
                }                                                                                           \
            }                                                                                               \
            __builtin_amdgcn_sched_barrier(0);                                                              \
            if constexpr (NEXT) {                                                                           \
                add_sums();                                                                                 \
                _Pragma("unroll") for (int b = 0; b < TMW + TNW; ++b) split_block(PN, b);                   \
            }                                                                                               \
            _Pragma("unroll") for (int grp = 2; grp < 6; ++grp) { MOLE_SPLIT_MFMAS(PC, grp) }               \
            if constexpr (NEXT) {                                                                           \
                _Pragma("unroll") for (int u = 0; u < 4 * CELLS_; ++u) {                                    \
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);                                        \
                    __builtin_amdgcn_sched_group_barrier(0x2, (56 * (TMW + TNW)) / (4 * CELLS_), 0);        \
                }                                                                                           \
            }                                                                                               \
            __builtin_amdgcn_sched_barrier(0);                                                              \
        }
#define MOLE_SPLIT_MFMAS(PC, grp)                                                                           \
        _Pragma("unroll") for (int cell_ = 0; cell_ < CELLS_; ++cell_) {                                    \
            const int tm = cell_ / TNW, tn = cell_ % TNW;                                                   \
            f32x16 &to_ = SPLIT_M[grp] + SPLIT_N[grp] == 0 ? acc[tm][tn] : low[tm][tn];                     \
            to_ = __builtin_amdgcn_mfma_f32_32x32x16_bf16(PC[tm].part(SPLIT_M[grp]), PC[TMW + tn].part(SPLIT_N[grp]), to_, 0, 0, 0); \
        }
        // The loop does two stages, the last one no other follows.  (Peeled at the end, for even and odd numbers, the stages cost the
        // 128 x 128 tiles 80 spilled registers; a reload waits for the operand loads in flight: 1140 us for 735, the training pass of
        // 8 experts, 512 -> 2048, 4096 tokens top-2.)
        int s = 0;
        if ((nk & 1) == 0) {
            MOLE_SPLIT_STAGE(0, pa, pb, true)
#pragma unroll
            for (int b = 0; b < TMW + TNW; ++b) pa[b] = pb[b];
            s = 1;
        }
        for (; s + 1 < nk; s += 2) {
            MOLE_SPLIT_STAGE(s, pa, pb, true)
            MOLE_SPLIT_STAGE(s + 1, pb, pa, true)
        }
        MOLE_SPLIT_STAGE(s, pa, pb, false)
#undef MOLE_SPLIT_STAGE
#undef MOLE_SPLIT_MFMAS
#pragma unroll
        for (int i = 0; i < TMW; ++i)
#pragma unroll
            for (int j = 0; j < TNW; ++j)
#pragma unroll
                for (int q = 0; q < 16; ++q) acc[i][j][q] += low[i][j][q];
        return least < (__float_as_uint(PARTS_MIN) << 1) - 1u;
    }
    MFrag mb;
    NFrag nb;
    ma.read(smem, fm0, fm1);
    na.read(smem + TL::M_BYTES, fn0, fn1);
    add_sums();         // (of the first stage: only contractions of one row ask for sums here)

    // One stage: the MFMAs of stage S on the fragments MC / NC.  With NEXT, behind the first of them the hand-over to stage S + 1: wait
    // until this wave's share of it has landed, barrier; then, dealt out between the MFMAs so that the matrix pipe
    // always has the next one waiting, the fragment reads of stage S + 1 into MN / NN, which are waited for first, and the loads that refill the
    // buffer stage S - 1 has left.  (A wave issues in order: eight loads and reads in a row right after the barrier
    // left the pipe idle for a tenth of a 64 x 128 tile's stage; loads before reads: 2 % at K = 2496.)  NEXT is a compile-time choice: were the fragment
    // reads under a run-time condition, the compiler could not tell how many LDS reads are outstanding at the first
    // MFMA and would wait for all of them, the ones just issued included.
    // Order of a stage's MFMAs: two waves on a SIMD that each alternate between two accumulators run at 0.85 of the
    // MFMA rate on this chip (measured with operands held in registers: one, three or four accumulators in turn, or
    // one wave per SIMD, all reach the full rate), so a wave with two cells runs its eight steps on one cell, then
    // on the other; with four or eight cells they take turns.
#define MOLE_F32_STAGE(S, MC, NC, MN, NN, NEXT)                                                             \
    {                                                                                                   \
        const int s_ = (S);                                                                             \
        bool refill_ = false;                                                                           \
        const int nb_ = (s_ + 1) % F_NSTAGE;                                                            \
        constexpr int CELLS_ = TMW * TNW, STEPS_ = TL::EDGE == 32 ? 8 : 4, G_ = STEPS_ * CELLS_ / 8;      \
        _Pragma("unroll") for (int grp = 0; grp < 8; ++grp) {                                           \
            _Pragma("unroll") for (int u = 0; u < G_; ++u) {                                            \
                const int n_ = grp * G_ + u;                                                            \
                const int cell_ = CELLS_ == 2 ? n_ / 8 : n_ % CELLS_, step_ = CELLS_ == 2 ? n_ % 8 : n_ / CELLS_; \
                const int tm = cell_ / TNW, tn = cell_ % TNW, kk = step_ / 4, j = step_ % 4;            \
                if constexpr (TL::EDGE == 32) acc[tm][tn] = __builtin_amdgcn_mfma_f32_32x32x2f32(MC.get(tm, kk, j), NC.get(tn, kk, j), acc[tm][tn], 0, 0, 0); \
                else acc[tm][tn] = __builtin_amdgcn_mfma_f32_16x16x4f32(NC.get(tn, kk, j), MC.get(tm, kk, j), acc[tm][tn], 0, 0, 0); \
            }                                                                                           \
            if constexpr (NEXT) {                                                                       \
                if (grp == 0) {                                                                         \
                    __builtin_amdgcn_sched_barrier(0);                                                  \
                    if (F_NSTAGE == 4 && s_ + 2 < nk) __builtin_amdgcn_s_waitcnt(waitcnt_vm(L));        \
                    else __builtin_amdgcn_s_waitcnt(waitcnt_vm(0));                                     \
                    __builtin_amdgcn_s_barrier();                                                       \
                    refill_ = s_ + F_NSTAGE - 1 < nk;                                                   \
                    if (WG && s_ + 1 == nk - 1 && kl < F_BK) zero_tail(nb_);                            \
                }                                                                                       \
                if (grp >= 2 && grp < L + 2 && refill_) issue_one(s_ + F_NSTAGE - 1, grp - 2);                           \
                if (grp == 0) MN.read(smem + nb_ * TL::STAGE, fm0, fm1);                                \
                if (grp == 1) NN.read(smem + nb_ * TL::STAGE + TL::M_BYTES, fn0, fn1);                  \
            }                                                                                           \
            __builtin_amdgcn_sched_barrier(0);                                                          \
        }                                                                                               \
    }
    int s = 0;
    for (; s + 2 < nk; s += 2) {
        MOLE_F32_STAGE(s, ma, na, mb, nb, true)
        MOLE_F32_STAGE(s + 1, mb, nb, ma, na, true)
    }
    if (nk - s == 2) {
        MOLE_F32_STAGE(s, ma, na, mb, nb, true)
        MOLE_F32_STAGE(s + 1, mb, nb, ma, na, false)
    } else {
        MOLE_F32_STAGE(s, ma, na, mb, nb, false)
    }
#undef MOLE_F32_STAGE
    return false;
}

// A stage of 32 of k of an operand tile of ROWS rows, as parts in LDS: the 16 bytes at ((4 part + h) ROWS + (row ^ X(h))) 16 hold the eight k
// of eighth h of a row.  A fragment read (lane l: row l % 16, eighth l / 16) is four stretches of 256 bytes; X, 12 for odd h, keeps what a
// pass of it takes of two stretches on different banks (X = 4 h, which the writes would like better: 6 % slower in all).
template <int ROWS> struct Parts {
    static constexpr int PLANE = 4 * ROWS * 16, BYTES = 3 * PLANE;
    static __device__ __forceinline__ uint32_t at(int h, int row) { return (uint32_t)((h * ROWS + (row ^ ((h & 1) * 12))) * 16); }
};

// Two stages of an operand tile on their way from memory to Parts, through the registers of the NW waves of a block.  Every value is
// taken apart once for the whole block.
//   K-contiguous: a load brings a lane four k of a row (8 rows of 128 bytes to the wave); the wave's load i is rows 8 (NW i + w) on.
//   K-strided:    a lane's task is one row and an eighth of the k, eight loads of 256 bytes to the wave; the wave's task is the 64 rows
//                 w % (ROWS / 64) and eighth w / (ROWS / 64).
template <int ROWS, bool KS, int NW> struct Raw {
    static constexpr int NV = ROWS * P_BK / (64 * NW);      // values a lane
    static constexpr int NP = NV / 2;                       // pairs of them
    static constexpr int NT = NV / 4, RG = ROWS / 64;
    static_assert(NV == 8 && RG * 4 == NW, "a task a wave");
    float v[2][NV];
    uint32_t part[4][3];
    uint32_t off[KS ? 1 : NT];      // byte offset of the lane's row (K-contiguous: and of its four k) from the base
    uint32_t lds;                   // where the lane's first values go in Parts
    const char *base[KS ? 8 : 1];   // of the stage to fetch next, wave-uniform
    long step;
    __device__ __forceinline__ void init(const float *p, long ld, int r0, int r_left, int k_ext, int wave, const int32_t *src, int n_src) {
        const int lane = threadIdx.x & 63;
        if constexpr (!KS) {
            const int q = lane & 7;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                uint32_t at = (uint32_t)min((NW * i + wave) * 8 + (lane >> 3), r_left - 1);
                if (src != nullptr) at = min((uint32_t)src[at], (uint32_t)n_src - 1u);
                off[i] = (uint32_t)(at * ld * 4 + min(q * 16, k_ext * 4 - 16));
            }
            base[0] = uniform_ptr(src != nullptr ? p : p + (long)r0 * ld);
            step = P_BK * 4;
            lds = Parts<ROWS>::at(q >> 1, wave * 8 + (lane >> 3)) + (q & 1) * 8;
        } else {
            off[0] = (uint32_t)min((wave % RG) * 64 + lane, r_left - 1) * 4;
            step = ld * (P_BK * 4);
            rows_from(p + r0, ld, min(k_ext, P_BK), wave);
            lds = Parts<ROWS>::at(wave / RG, (wave % RG) * 64 + lane);
        }
    }
    // K-strided: the k-rows of a stage that begins at p and has k_left of them
    __device__ __forceinline__ void rows_from(const float *p, long ld, int k_left, int wave) {
#pragma unroll
        for (int j = 0; j < 8; ++j) base[KS ? j : 0] = uniform_ptr(p + (long)min(8 * (wave / RG) + j, k_left - 1) * ld);
    }
    __device__ __forceinline__ void advance() {
#pragma unroll
        for (int j = 0; j < (KS ? 8 : 1); ++j) base[j] += step;
    }
    // to the last stage, which has k_left of k and begins at p (K-strided)
    __device__ __forceinline__ void advance_to_tail(const float *p, long ld, int k_left, int wave) {
        if constexpr (KS) {
            rows_from(p, ld, k_left, wave);
        } else {
            const uint32_t q = threadIdx.x & 7, past = max((int)q * 16 - (k_left * 4 - 16), 0);
#pragma unroll
            for (int i = 0; i < NT; ++i) off[i] -= past;
            advance();
        }
    }
    // the loads that bring pair u (K-contiguous: a load brings two, which the first one asks for)
    template <int D> __device__ __forceinline__ void fetch_pair(int u) {
        typedef __attribute__((address_space(1))) const char gchar;
        typedef float f4 __attribute__((ext_vector_type(4)));
        if constexpr (!KS) {
            if (u % 2 == 0) {
                const f4 t = *reinterpret_cast<const __attribute__((address_space(1))) f4 *>((gchar *)base[0] + off[u / 2]);
#pragma unroll
                for (int c = 0; c < 4; ++c) v[D][2 * u + c] = t[c];
            }
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) v[D][2 * u + c] = *reinterpret_cast<const __attribute__((address_space(1))) float *>((gchar *)base[KS ? 2 * u + c : 0] + off[0]);
        }
    }
    template <int D> __device__ __forceinline__ void fetch() {
#pragma unroll
        for (int u = 0; u < NP; ++u) fetch_pair<D>(u);
    }
    // takes pair u apart, stores what it completes and asks for the pair's successor
    template <int D> __device__ __forceinline__ void convert(char *stage, int u, uint32_t &least) {
        split_pair(v[D][2 * u], v[D][2 * u + 1], part[u], least);
        if constexpr (!KS) {
            if (u % 2 == 1) {
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x2 *>(stage + lds + (u / 2) * (NW * 8 * 16) + q * Parts<ROWS>::PLANE) = u32x2{part[u - 1][q], part[u][q]};
            }
        } else if (u == 3) {
#pragma unroll
            for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x4 *>(stage + lds + q * Parts<ROWS>::PLANE) = u32x4{part[0][q], part[1][q], part[2][q], part[3][q]};
        }
    }
    template <int D> __device__ __forceinline__ void refetch(int u) {
        if constexpr (KS) fetch_pair<D>(u);
        else if (u % 2 == 1) fetch_pair<D>(u - 1);
    }
    // the k of the last stage from k_valid on count nothing
    template <int D> __device__ __forceinline__ void clear_from(int k_valid, int wave) {
#pragma unroll
        for (int i = 0; i < NV; ++i)
            if ((KS ? 8 * (wave / RG) + i : (int)(threadIdx.x & 7) * 4 + i % 4) >= k_valid) v[D][i] = 0.f;
    }
};

// The K loop of one tile by the parts of its operands: acc += the products of its nk stages.  Returns whether this lane met an operand
// that has no exact parts.
//
// The parts of two stages stand in LDS.  Stage s:
//   the products of its first 16 of k, whose fragments are there; meanwhile the fragments of the others are read, and the m-side of stage
//   s + 1 is taken apart and stored, each load of stage s + 3 issued when its registers are free
//   barrier: stage s + 1 is whole, and nobody reads stage s any more
//   the products of the other 16 of k; meanwhile the fragments of the first 16 of stage s + 1 and the n-side of stage s + 2
template <int BM, int BN, int NW, bool N_KS>
__device__ __forceinline__ bool shared_parts_loop(const GemmArgs &g, const float *Mp, const float *Np, int m0, int n0, int m_ext, int k_ext, char *smem,
                                           int wave, int wm, int wn, f32x4 (&acc)[4][2], const int32_t *src) {
    constexpr int STAGE = Parts<BM>::BYTES + Parts<BN>::BYTES;
    const int nk = (k_ext + P_BK - 1) / P_BK;
    if (nk <= 0) return false;
    const int kl = k_ext - (nk - 1) * P_BK;     // k of the last stage
    const bool ragged = kl < P_BK;
    Raw<BM, false, NW> rm;
    Raw<BN, N_KS, NW> rn;
    rm.init(Mp, g.lda, m0, m_ext - m0, k_ext, wave, src, g.tokens);
    rn.init(Np, g.ldb, n0, g.N - n0, k_ext, wave, nullptr, 0);
    // bases of stage s; past the end they stay at the last stage, which is fetched and taken apart again for nobody
    auto to_m = [&](int s) __attribute__((always_inline)) {
        if (s >= nk) return;
        if (ragged && s == nk - 1) rm.advance_to_tail(nullptr, 0, kl, wave);
        else rm.advance();
    };
    auto to_n = [&](int s) __attribute__((always_inline)) {
        if (s >= nk) return;
        if (ragged && s == nk - 1) rn.advance_to_tail(Np + n0 + (long)s * P_BK * g.ldb, g.ldb, kl, wave);
        else rn.advance();
    };
    // what the values of stage s still need when they have come
    auto came_m = [&](auto d, int s) __attribute__((always_inline)) {
        if (s >= nk - 1 && (ragged || s >= nk)) rm.template clear_from<d>(s >= nk ? 0 : kl, wave);
    };
    auto came_n = [&](auto d, int s) __attribute__((always_inline)) {
        if (ragged && s == nk - 1) rn.template clear_from<d>(kl, wave);
    };
    constexpr std::integral_constant<int, 0> EVEN{};
    constexpr std::integral_constant<int, 1> ODD{};
    uint32_t least = 0xffffffffu;
    const int lane = threadIdx.x & 63;
    const uint32_t fm = Parts<BM>::at(lane >> 4, wm * 64 + (lane & 15)), fn = Parts<BM>::BYTES + Parts<BN>::at(lane >> 4, wn * 32 + (lane & 15));
    u32x4 pm[2][3][2], pn[2][3][2];        // fragments: of either half of the m-side; of the n-side of two stages
    auto read_m = [&](auto h, const char *stage, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 2; ++b) pm[h][q][b] = *reinterpret_cast<const u32x4 *>(stage + fm + q * Parts<BM>::PLANE + (2 * h + b) * 256);
    };
    auto read_n = [&](auto d, const char *stage, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int b = 0; b < 2; ++b) pn[d][q][b] = *reinterpret_cast<const u32x4 *>(stage + fn + q * Parts<BN>::PLANE + b * 256);
    };
    f32x4 low[4][2];              // the products below hi hi
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) low[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    // stage 0 whole, the n-side of stage 1; on their way the m-side of stages 1 and 2, the n-side of 2 and 3
    rm.template fetch<0>();
    rn.template fetch<0>();
    to_m(1);
    rm.template fetch<1>();
    to_n(1);
    rn.template fetch<1>();
    to_m(2);
    came_m(EVEN, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) { rm.template convert<0>(smem, u, least); rm.template refetch<0>(u); }
    to_n(2);
    came_n(EVEN, 0);
#pragma unroll
    for (int u = 0; u < 4; ++u) { rn.template convert<0>(smem + Parts<BM>::BYTES, u, least); rn.template refetch<0>(u); }
    to_n(3);
    came_n(ODD, 1);
#pragma unroll
    for (int u = 0; u < 4; ++u) { rn.template convert<1>(smem + STAGE + Parts<BM>::BYTES, u, least); rn.template refetch<1>(u); }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 3; ++q) { read_m(EVEN, smem, q); read_n(EVEN, smem, q); }

    // Six MFMAs of half H (product I / 4, m-block and n-block I % 4) of a stage of parity D, and a pair of an operand among them
#define MOLE_CELL(H, D, I)                                                                                       \
        {                                                                                                        \
            constexpr int i_ = 2 * (H) + (((I) >> 1) & 1), j_ = (I) & 1;                                         \
            f32x4 &to_ = (I) / 4 == 5 ? acc[i_][j_] : low[i_][j_];                                               \
            to_ = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, pn[D][SPLIT_N[(I) / 4]][j_]), __builtin_bit_cast(bf16x8, pm[H][SPLIT_M[(I) / 4]][i_ & 1]), to_, 0, 0, 0); \
        }
#define MOLE_SPREAD()                                                                                            \
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);                                                         \
        __builtin_amdgcn_sched_group_barrier(0x2, 5, 0);
#define MOLE_QUARTER(H, D, Q, R, RD, STAGE_PTR)                                                                  \
        {                                                                                                        \
            MOLE_CELL(H, D, 6 * (Q)) MOLE_CELL(H, D, 6 * (Q) + 1) MOLE_CELL(H, D, 6 * (Q) + 2)                   \
            MOLE_CELL(H, D, 6 * (Q) + 3) MOLE_CELL(H, D, 6 * (Q) + 4) MOLE_CELL(H, D, 6 * (Q) + 5)               \
            R.template convert<RD>(STAGE_PTR, Q, least);                                                         \
            R.template refetch<RD>(Q);                                                                           \
            MOLE_SPREAD() MOLE_SPREAD() MOLE_SPREAD()                                                            \
            __builtin_amdgcn_sched_barrier(0);                                                                   \
        }
    // Stage S, of parity D.  (lgkmcnt(0): the parts this wave has stored have landed; loads from memory may be in flight.)
#define MOLE_STAGE(S, D)                                                                                         \
        {                                                                                                        \
            char *const cur = smem + (D) * STAGE, *const nxt = smem + (1 - (D)) * STAGE;                         \
            to_m((S) + 3);                                                                                       \
            came_m(std::integral_constant<int, 1 - (D)>{}, (S) + 1);                                             \
            read_m(ODD, cur, 0);                                                                                 \
            read_m(ODD, cur, 1);                                                                                 \
            read_m(ODD, cur, 2);                                                                                 \
            __builtin_amdgcn_sched_barrier(0);                                                                   \
            MOLE_QUARTER(0, D, 0, rm, 1 - (D), nxt)                                                              \
            MOLE_QUARTER(0, D, 1, rm, 1 - (D), nxt)                                                              \
            MOLE_QUARTER(0, D, 2, rm, 1 - (D), nxt)                                                              \
            MOLE_QUARTER(0, D, 3, rm, 1 - (D), nxt)                                                              \
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");                                                   \
            __builtin_amdgcn_s_barrier();                                                                        \
            asm volatile("" ::: "memory");                                                                       \
            to_n((S) + 4);                                                                                       \
            came_n(std::integral_constant<int, D>{}, (S) + 2);                                                   \
            read_m(EVEN, nxt, 0);                                                                                \
            read_m(EVEN, nxt, 1);                                                                                \
            read_m(EVEN, nxt, 2);                                                                                \
            read_n(std::integral_constant<int, 1 - (D)>{}, nxt, 0);                                              \
            read_n(std::integral_constant<int, 1 - (D)>{}, nxt, 1);                                              \
            read_n(std::integral_constant<int, 1 - (D)>{}, nxt, 2);                                              \
            __builtin_amdgcn_sched_barrier(0);                                                                   \
            MOLE_QUARTER(1, D, 0, rn, D, cur + Parts<BM>::BYTES)                                                 \
            MOLE_QUARTER(1, D, 1, rn, D, cur + Parts<BM>::BYTES)                                                 \
            MOLE_QUARTER(1, D, 2, rn, D, cur + Parts<BM>::BYTES)                                                 \
            MOLE_QUARTER(1, D, 3, rn, D, cur + Parts<BM>::BYTES)                                                 \
        }
    // Two stages at a time; of an odd number the last one meets an m-side of zeros.
    for (int s = 0; s < nk; s += 2) {
        MOLE_STAGE(s, 0)
        MOLE_STAGE(s + 1, 1)
    }
#undef MOLE_STAGE
#undef MOLE_QUARTER
#undef MOLE_SPREAD
#undef MOLE_CELL
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] += low[i][j];
    return least < (__float_as_uint(PARTS_MIN) << 1) - 1u;
}

template <int BM, int BN, int NSTAGE, int NW, int BPC, How HOW, bool M_KS, bool N_KS, bool WG, int EPI>
__global__ __launch_bounds__(64 * NW, BPC * NW / 4) void gemm_f32_kernel(const GemmArgs g) {
    typedef FTile<BM, BN, NSTAGE, NW, HOW> TL;
    constexpr int TMW = TL::TMW, TNW = TL::TNW;
    constexpr bool PARTS = HOW != OPERANDS;
    extern __shared__ __align__(16) char smem[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    // ---- which tile am I?  Blocks are dealt round-robin to the 8 XCDs (block b runs on XCD b mod 8): every XCD
    //      takes a contiguous range of the real tiles, so that neighbours share operands in its L2.  For row-ragged
    //      products the number of real tiles is only known here (the grid is sized for the worst case).
    const int n_tiles = (g.N + BN - 1) / BN;
    // a contraction split over blocks: the planes of an m-tile's n-tiles are numbered like more n-tiles
    const int n_units = EPI == EPI_PART ? n_tiles * g.ksplit : n_tiles;
    int e, mt, nt, m_ext, k_ext, split_k = 0;
    long row0;
    if constexpr (!WG) {
        // (Nothing runs beside this search on a CU with one block: 777 tokens, top-2 of 8, 79.6 -> 78 us for it and its loads in one.  Lane l holds the rows and the first row of expert l, of later 64 if
        // those do not reach this tile.)
        const bool single = g.offsets == nullptr;
        const int nE = single ? 1 : g.E;
        auto fetch = [&](int ee, int &rows, int &first) {
            rows = ee < nE ? (single ? g.single_rows : g.kept[ee]) : 0;
            first = !single && ee < nE ? g.offsets[ee] : 0;
        };
        int rows, first, base = 0, run = 0;
        fetch(lane, rows, first);
        int cnt = (rows + BM - 1) / BM, incl = wave_scan(cnt), total = wave_total(incl);
        if (nE > WAVE) {
            int more = 0;
            for (int ee = lane + WAVE; ee < nE; ee += WAVE) more += (g.kept[ee] + BM - 1) / BM;
            total += wave_total(wave_scan(more));
        }
        total *= n_units;
        const int per_xcd = (total + 7) >> 3;
        const int slot = blockIdx.x >> 3;
        const int t = (blockIdx.x & 7) * per_xcd + slot;
        if (slot >= per_xcd || t >= total) return;
        const int mtg = t / n_units;
        nt = t - mtg * n_units;
        unsigned long long hit = __ballot(incl > mtg);
        while (!hit) {
            run += wave_total(incl);
            base += WAVE;
            if (base >= nE) return;
            fetch(base + lane, rows, first);
            cnt = (rows + BM - 1) / BM;
            incl = wave_scan(cnt);
            hit = __ballot(run + incl > mtg);
        }
        const int at = __ffsll(hit) - 1;
        e = base + at;
        mt = mtg - (run + __builtin_amdgcn_readlane(incl - cnt, at));
        m_ext = __builtin_amdgcn_readlane(rows, at);
        row0 = __builtin_amdgcn_readlane(first, at);
        k_ext = g.K;
        if constexpr (EPI == EPI_PART) {
            split_k = nt / n_tiles;
            nt %= n_tiles;
        }
    } else {
        const int t = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
        if (t >= g.n_blocks) return;
        const int m_tiles = (g.M + BM - 1) / BM;
        e = t / (m_tiles * n_tiles);
        const int rem = t % (m_tiles * n_tiles);
        mt = rem / n_tiles;
        nt = rem % n_tiles;
        m_ext = g.M;
        k_ext = g.kept ? g.kept[e] : g.single_rows;
        row0 = g.offsets ? g.offsets[e] : 0;
    }
    e = __builtin_amdgcn_readfirstlane(e);
    mt = __builtin_amdgcn_readfirstlane(mt);
    nt = __builtin_amdgcn_readfirstlane(nt);
    m_ext = __builtin_amdgcn_readfirstlane(m_ext);
    k_ext = __builtin_amdgcn_readfirstlane(k_ext);
    row0 = ((long)__builtin_amdgcn_readfirstlane((int)(row0 >> 32)) << 32) | (unsigned)__builtin_amdgcn_readfirstlane((int)row0);
    const int m0 = mt * BM, n0 = nt * BN;
    // h = xd.w1^T + b1 may read its rows where the tokens lie (a forward pass that nobody asks for xd)
    const int32_t *src = nullptr;
    if constexpr (EPI == EPI_BIAS_GELU) { if (g.token_of != nullptr) src = g.token_of + row0 + m0; }
    const float *Mp = (const float *)g.A + (src != nullptr ? 0 : row0 * g.lda);
    const float *Np = WG ? (const float *)g.B + row0 * g.ldb : (const float *)g.B + (long)e * g.strideB;
    if constexpr (EPI == EPI_PART) {           // this block's stages of the contraction (which is whole stages)
        split_k = __builtin_amdgcn_readfirstlane(split_k);
        constexpr int STEP = HOW == SHARED_PARTS ? P_BK : F_BK;
        const int stages = (k_ext + STEP - 1) / STEP;
        const int k_lo = split_k * stages / g.ksplit * STEP;
        k_ext = min((split_k + 1) * stages / g.ksplit * STEP, k_ext) - k_lo;
        Mp += k_lo;
        Np += N_KS ? (long)k_lo * g.ldb : (long)k_lo;
    }
    const int wm = wave / TL::WN, wn = wave % TL::WN;

    typename TL::Acc acc[TMW][TNW];
#pragma unroll
    for (int i = 0; i < TMW; ++i)
#pragma unroll
        for (int j = 0; j < TNW; ++j)
#pragma unroll
            for (int q = 0; q < TL::Q; ++q) acc[i][j][q] = 0.f;

    // Operand sums over the contraction (the bias gradients: sums of go and of t over an expert's rows, torch::sum_out
    // in MOLE/cpp/core.cpp:399, 408) ride along in the weight-gradient blocks that see the whole operand once: the
    // first n-tile of every m-tile for the m-side, the first m-tile of every n-tile for the n-side.  The wave row or
    // column that holds the operand's fragments adds them up as they pass, four partial sums per column.
    int sum_side = 0;
    if constexpr (WG) {
        if (g.colsum != nullptr) {
            if (g.colsum_side == 1 && nt == 0 && wn == 0) sum_side = 1;
            if (g.colsum_side == 2 && mt == 0 && wm == 0) sum_side = 2;
        }
    }
    constexpr int SB = 2;
    float psum[4][SB];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < SB; ++b) psum[j][b] = 0.f;

    // A weight gradient of one row is products without a sum: exact but for their rounding from fp32 operands, where the products that the
    // parts leave out add to it (2-norm error in 2^-24: 0.424, by parts 0.435; two rows 0.518 and 0.440).  Its only stage also gives the sums.
    const bool one_row = PARTS && WG && k_ext <= 1;
    bool redo = one_row;
    f32x4 old_h[TL::EDGE == 16 ? TMW : 1][TL::EDGE == 16 ? TNW : 1];
    if (!one_row) {
        bool inexact;
        if constexpr (HOW == SHARED_PARTS) inexact = shared_parts_loop<BM, BN, NW, N_KS>(g, Mp, Np, m0, n0, m_ext, k_ext, smem, wave, wm, wn, acc, src);
        else inexact = f32_loop<BM, BN, NSTAGE, NW, HOW, M_KS, N_KS, WG, PARTS>(g, Mp, Np, m0, n0, m_ext, k_ext, smem, wave, wm, wn, acc, sum_side, psum, src);
        if constexpr (TL::EDGE == 16 && EPI == EPI_DGELU) {     // h, on its way while the tile is tested
#pragma unroll
            for (int tm = 0; tm < TMW; ++tm) {
                const long r = row0 + min(m0 + wm * 64 + 16 * tm + (lane & 15), m_ext - 1);
#pragma unroll
                for (int tn = 0; tn < TNW; ++tn)
                    old_h[tm][tn] = *reinterpret_cast<const f32x4 *>((const float *)g.H + r * g.ldc + min(n0 + wn * 32 + 16 * tn + 4 * (lane >> 4), g.N - 4));
            }
        }
        if constexpr (PARTS) {
            // An infinity, a NaN or a value within half a unit of bf16 of the overflow limit has no finite parts: its products with
            // a part that is zero are NaN.  A tile with any result that is not finite is computed again with fp32 operands.
            float poison = 0.f;
#pragma unroll
            for (int i = 0; i < TMW; ++i)
#pragma unroll
                for (int j = 0; j < TNW; ++j)
#pragma unroll
                    for (int q = 0; q < TL::Q; ++q) poison = fmaf(acc[i][j][q], 0.f, poison);
            int *flag = reinterpret_cast<int *>(smem);
            __syncthreads();
            const bool bad = __ballot(poison != 0.f || inexact) != 0;      // (NaN compares unequal)
            if (lane == 0) flag[wave] = bad;
            __syncthreads();
#pragma unroll
            for (int i = 0; i < NW; ++i) redo |= flag[i] != 0;
        }
    }
    if constexpr (PARTS) {
        if (__builtin_amdgcn_readfirstlane(redo)) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < TMW; ++i)
#pragma unroll
                for (int j = 0; j < TNW; ++j)
#pragma unroll
                    for (int q = 0; q < TL::Q; ++q) acc[i][j][q] = 0.f;
            f32_loop<BM, BN, NSTAGE, NW, HOW, M_KS, N_KS, WG, false>(g, Mp, Np, m0, n0, m_ext, k_ext, smem, wave, wm, wn, acc, one_row ? sum_side : 0, psum, src);
        }
    }

    if constexpr (WG) {
        if (sum_side != 0) {
            // a lane's fragments cover k-rows 8 kk + 4 (lane / 32) + j: the two half waves hold the two halves of the sum
            const int nbk = sum_side == 1 ? TMW : TNW;
            const int first = sum_side == 1 ? m0 + wm * 32 * TMW : n0 + wn * 32 * TNW;
            const int ext = sum_side == 1 ? m_ext : g.N;
            float *out = (float *)g.colsum + (long)e * ext;
#pragma unroll
            for (int b = 0; b < SB; ++b) {
                float v = (psum[0][b] + psum[1][b]) + (psum[2][b] + psum[3][b]);
                v += __shfl_xor(v, 32, WAVE);
                const int c = first + nbk * (lane & 31) + b;
                if (b < nbk && lane < 32 && c < ext) {
                    if (g.accumulate) v += out[c];
                    out[c] = v;
                }
            }
        }
    }

    // ---- epilogue
    float *Cb = EPI == EPI_PART ? g.part : (float *)g.C;
    const long ldc = EPI == EPI_PART ? (long)g.N : g.ldc;
    long crow0 = EPI == EPI_PART ? split_k * g.part_rows + row0 : row0;
    if constexpr (WG) { crow0 = 0; Cb += (long)e * g.strideC; }
    const bool store = EPI != EPI_BIAS_GELU || g.C != nullptr;      // h is left out where no backward pass will ask for it
    if constexpr (TL::EDGE == 16) {
        // acc[tm][tn][q] = C[m, n] with m = lane % 16 in the m-block and n = 4 (lane / 16) + q in the n-block: the four columns go as one
        // access (N is a multiple of 4), 64 bytes of 16 rows to the wave
        int ncol[TNW];
        f32x4 bias[TNW];
#pragma unroll
        for (int tn = 0; tn < TNW; ++tn) {
            ncol[tn] = n0 + wn * 32 + 16 * tn + 4 * (lane >> 4);
            bias[tn] = f32x4{0.f, 0.f, 0.f, 0.f};
            if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU)
                if (ncol[tn] < g.N) bias[tn] = *reinterpret_cast<const f32x4_any *>((const float *)g.bias + (long)e * g.N + ncol[tn]);
        }
#pragma unroll
        for (int tm = 0; tm < TMW; ++tm) {
            const int m = m0 + wm * 64 + 16 * tm + (lane & 15);
            if (m >= m_ext) continue;
            float *dst = Cb + (crow0 + m) * ldc;
#pragma unroll
            for (int tn = 0; tn < TNW; ++tn) {
                if (ncol[tn] >= g.N) continue;
                f32x4 v = acc[tm][tn], v2 = v;
                if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU) v += bias[tn];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    if constexpr (EPI == EPI_BIAS_GELU) {
                        v2[q] = gelu_erf(v[q]);
                    } else if constexpr (EPI == EPI_DGELU) {
                        const float hv = old_h[tm][tn][q];
                        v[q] *= g.gelu_bwd == MOLE_GELU_BWD_TANH ? d_gelu_tanh(hv) : d_gelu_exact(hv);
                    }
                }
                if (store) *reinterpret_cast<f32x4 *>(dst + ncol[tn]) = v;
                if constexpr (EPI == EPI_BIAS_GELU) *reinterpret_cast<f32x4 *>((float *)g.C2 + (crow0 + m) * ldc + ncol[tn]) = v2;
            }
        }
    } else {
        // acc[tm][tn][q] = C[m, n] with i = 8 (q / 4) + 4 (lane / 32) + q % 4 the row inside the m-block and
        // lane % 32 the column inside the n-block; a K-strided side interleaves the wave's blocks (row 2 i + tm).
        const int lr = lane & 31, h = lane >> 5;
        constexpr bool PAIR = N_KS && TNW == 2;         // a lane holds two adjacent columns: 8-byte accesses
        int ncol[TNW];
        float bias[TNW];
#pragma unroll
        for (int tn = 0; tn < TNW; ++tn) {
            ncol[tn] = N_KS ? n0 + wn * 32 * TNW + TNW * lr + tn : n0 + (wn * TNW + tn) * 32 + lr;
            bias[tn] = 0.f;
            if constexpr (EPI == EPI_BIAS || EPI == EPI_BIAS_GELU)
                if (ncol[tn] < g.N) bias[tn] = ((const float *)g.bias)[(long)e * g.N + ncol[tn]];
        }
        auto row_of = [&](int tm, int q) {
            const int i = 8 * (q >> 2) + 4 * h + (q & 3);
            return M_KS ? m0 + wm * 32 * TMW + TMW * i + tm : m0 + (wm * TMW + tm) * 32 + i;
        };
#pragma unroll
        for (int tm = 0; tm < TMW; ++tm) {
            // GELU', accumulation: the old values of this block's 16 rows are fetched first, unconditionally (rows and
            // columns past the end read a clamped address and are not used), so that they are in flight together
            float old[16][TNW];
            if constexpr (EPI == EPI_DGELU || EPI == EPI_WGRAD) {
                if (EPI == EPI_DGELU || g.accumulate) {
                    const float *src = EPI == EPI_DGELU ? (const float *)g.H : Cb;
#pragma unroll
                    for (int q = 0; q < 16; ++q) {
                        const long r = crow0 + min(row_of(tm, q), m_ext - 1);
                        if constexpr (PAIR) {
                            const float2 t = *reinterpret_cast<const float2 *>(src + r * ldc + min(ncol[0], g.N - 2));
                            old[q][0] = t.x; old[q][1] = t.y;
                        } else {
#pragma unroll
                            for (int tn = 0; tn < TNW; ++tn) old[q][tn] = src[r * ldc + min(ncol[tn], g.N - 1)];
                        }
                    }
                }
            }
#pragma unroll
            for (int q = 0; q < 16; ++q) {
                const int m = row_of(tm, q);
                if (m >= m_ext) continue;
                float v[TNW], v2[TNW];
#pragma unroll
                for (int tn = 0; tn < TNW; ++tn) {
                    v[tn] = acc[tm][tn][q];
                    v2[tn] = 0.f;
                    if constexpr (EPI == EPI_BIAS) {
                        v[tn] += bias[tn];
                    } else if constexpr (EPI == EPI_BIAS_GELU) {
                        v[tn] += bias[tn];
                        v2[tn] = gelu_erf(v[tn]);
                    } else if constexpr (EPI == EPI_DGELU) {
                        const float hv = old[q][tn];
                        v[tn] *= g.gelu_bwd == MOLE_GELU_BWD_TANH ? d_gelu_tanh(hv) : d_gelu_exact(hv);
                    } else if constexpr (EPI == EPI_WGRAD) {
                        if (g.accumulate) v[tn] += old[q][tn];
                    }
                }
                float *dst = Cb + (crow0 + m) * ldc;
                // The weight gradients (which nothing reads before the optimizer) leave with non-temporal stores: -2 us on
                // 8 x 2048 x 512.  For h, a and t it measured neutral to worse: the launches that follow read them.
                constexpr bool STREAM = EPI == EPI_WGRAD;
                auto put = [&](float *p, float x) __attribute__((always_inline)) {
                    if constexpr (STREAM) __builtin_nontemporal_store(x, p); else *p = x;
                };
                auto put2 = [&](float *p, float x, float y) __attribute__((always_inline)) {
                    typedef float f32x2 __attribute__((ext_vector_type(2)));
                    if constexpr (STREAM) __builtin_nontemporal_store(f32x2{x, y}, reinterpret_cast<f32x2 *>(p));
                    else *reinterpret_cast<float2 *>(p) = make_float2(x, y);
                };
                if constexpr (PAIR) {
                    if (ncol[0] < g.N) {
                        if (store) put2(dst + ncol[0], v[0], v[1]);
                        if constexpr (EPI == EPI_BIAS_GELU) put2((float *)g.C2 + (crow0 + m) * ldc + ncol[0], v2[0], v2[1]);
                    }
                } else {
#pragma unroll
                    for (int tn = 0; tn < TNW; ++tn) {
                        if (ncol[tn] >= g.N) continue;
                        if (store) put(dst + ncol[tn], v[tn]);
                        if constexpr (EPI == EPI_BIAS_GELU) put((float *)g.C2 + (crow0 + m) * ldc + ncol[tn], v2[tn]);
                    }
                }
            }
        }
    }
}

template <int BM, int BN, int NSTAGE, int NW, int BPC, How HOW, bool M_KS, bool N_KS, bool WG, int EPI>
int launch_f32(GemmArgs g, int tiles, hipStream_t st, int kid) {
    if (tiles <= 0) return 0;
    g.n_blocks = tiles;
    const int grid = (tiles + 7) & ~7;
    auto kern = gemm_f32_kernel<BM, BN, NSTAGE, NW, BPC, HOW, M_KS, N_KS, WG, EPI>;
    // the LDS request also caps the blocks a CU takes: with room for more than BPC, the dispatcher fills some CUs
    // and leaves others short, and the launch lasts as long as the fullest
    constexpr int lds_min = 160 * 1024 / (BPC + 1) + 1024;
    constexpr int ring = FTile<BM, BN, NSTAGE, NW, HOW>::RING_BYTES, shared = HOW == SHARED_PARTS ? 2 * (Parts<BM>::BYTES + Parts<BN>::BYTES) : 0;
    constexpr int need = shared > ring ? shared : ring, lds = need > lds_min ? need : lds_min;
    static bool attr_done = false;
    if (!attr_done) {
        MOLE_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        attr_done = true;
    }
    timed_launch(kid, kern, dim3(grid), dim3(64 * NW), lds, st, g);
    MOLE_LAUNCH_CHECK();
    return 0;
}

template <int BM, int BN, int NSTAGE, int NW, int BPC, How HOW>
int dispatch_f32(const GemmArgs &g, bool b_ks, bool wg, int epi, int max_rows, hipStream_t st, int kid) {
    const int n_tiles = ceil_div(g.N, BN);
    if (wg) {
        const int tiles = g.E * ceil_div(g.M, BM) * n_tiles;
        if constexpr (BM == 128 && HOW == OWN_PARTS)
            if (epi == EPI_WGRAD) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, true, true, true, EPI_WGRAD>(g, tiles, st, kid);
        return -100;
    }
    const int rows_bound = g.offsets ? max_rows : g.single_rows;
    const int tiles = (rows_bound / BM + (g.offsets ? g.E : 1)) * n_tiles;     // every expert may end in a partial tile
    if (!b_ks) {
        if (epi == EPI_BIAS_GELU) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, false, false, false, EPI_BIAS_GELU>(g, tiles, st, kid);
        if (epi == EPI_DGELU) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, false, false, false, EPI_DGELU>(g, tiles, st, kid);
    } else {
        if (epi == EPI_BIAS) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, false, true, false, EPI_BIAS>(g, tiles, st, kid);
        if (epi == EPI_STORE) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, false, true, false, EPI_STORE>(g, tiles, st, kid);
        if (epi == EPI_PART) return launch_f32<BM, BN, NSTAGE, NW, BPC, HOW, false, true, false, EPI_PART>(g, tiles * g.ksplit, st, kid);
    }
    return -100;
}

}  // namespace

// Whether the weight-gradient launch for g also produces the operand sums asked for in g.colsum.
bool gemm_f32_sums_operand(const GemmArgs &g) {
    return !(g.lda % 4 || g.ldb % 4 || g.ldc % 4 || g.N % 4 || g.N < 4 || g.M % 4 || g.M < 4);
}

// How a launch's tiles are made, and its number of planes.  A CU works off its tiles one after the other (those that share it share the
// pipes), so a launch takes ceil(tiles / 256) walks over K.  us, each way forced on experts of equal rows (rows x experts, widths: h = xd.w1^T
// + b1 with GELU | out = a.w2 + b2 without planes; 64-row tiles of fp32 operands / of own parts / 128-row tiles of shared parts):
//   128 x 8, 512 -> 2048      27.5 | 70.1 /  31.2 | 70.4 /  31.0 | 82.6     64 x 64, 256 -> 512      19.5 | 23.8 /  23.2 | 26.7 /  23.6 | 29.4
//   128 x 16, 1024 -> 1024    41.8 | 39.5 /  45.8 | 43.3 /  48.0 | 47.3    128 x 32, 1024 -> 1024    76.5 | 71.4 /  72.7 | 68.2 /  55.2 | 54.0
//   192 x 8, 512 -> 2048      43.2 | 71.6 /  42.6 | 73.5 /  34.5 | 83.8    192 x 20, 832 -> 1664      112 |  106 /   107 |  108 /   123 |  145
//   512 x 8, 512 -> 2048      83.3 | 80.5 /  84.7 | 93.5 /  68.3 | 93.6   1024 x 8, 512 -> 2048       161 |  149 /   153 |  145 /   129 |  106
//   1024 x 4, 1024 -> 4096     280 |  272 /   271 |  280 /   234 |  208   2048 x 8, 1024 -> 4096     1061 | 1006 /  1016 |  968 /   870 |  779
// (128-row tiles of own parts, which the last were: 1024 x 8 129 | 119, 128 x 32 72.3 | 63.9, 2048 x 8 881 | 779.)
// So: a stage of 16 of K takes 0.58 us on 64-row tiles, several blocks of which share a CU's pipes, and on 128-row tiles of shared parts 0.7
// us and, as the chip fills, 0.75.  A CU that has one of these left over makes the others wait.
// Experts do not share the rows evenly; one whose rows go past a tile's end, where the capacity lets it, is a tile more (their spread is taken as
// twice that of random picks; of 64 experts of 94 rows, 256 -> 512, one with more than 128 made h 31 -> 39 us by 128-row tiles).
// The constants are those that choose best for 111 products of 4 to 64 experts, 48 of them with rows that random gates give: 2 % above the
// fastest way and plane count measured, 6 % below what the choice between own parts of either height took.
// The K = F products are narrow and long and may also be split over blocks into p planes of partial results, which costs the
// planes' way through memory at 5 TB/s and the reduction's launch.
static double f32_tiles(int bm, int p, int E, Rows rows, int N) {
    const int active = E < rows.est ? E : rows.est;
    const double mean = (double)rows.est / active, whole = std::ceil(mean / bm) * bm, spread = 2.0 * std::sqrt(mean);
    const double past = bm == 128 && whole < rows.most ? std::floor(active * 0.5 * std::erfc((whole - mean) / (std::sqrt(2.0) * spread))) : 0.0;
    return (double)p * ceil_div(N, 128) * (active * (whole / bm) + past);
}
// Whether 128-row tiles are of shared parts.  Their blocks have a CU to themselves, and their loop takes two stages of 32 at a time.  Blocks of
// own parts, two to a CU, hide each other's ends, and that counts where a CU walks more than once over a short K (shared / own, us, out:
// 1636 rows x 23, 576 -> 576 193 / 172; 528 x 64, 320 -> 320 85 / 73; 1238 x 20, 768 -> 320 128 / 120; 1570 x 20, 512 -> 832 238 / 227; K = 1664,
// 1160 x 8 241 / 240, K = 2880, 391 x 20 620 / 634), over a K in planes (two, of the same: 337 / 291, 248 / 230, 688 / 639) and where an eighth of h's walk over K would be padding (7911 x 7, 336 -> 1008 347 / 320).
// h and t of many walks take the same time either way when launches are timed one by one (1024 x 8, 512 -> 2048: 265 / 266 for both, and shared ones read 151
// and 217 MB instead of 130 and 198); passes that follow each other run into the power limit, and there shared ones are ahead, shared / own, us: 4096 tokens, 8 experts top-2,
// 512 -> 2048 704 / 714, 16384 2660 / 2680, 16 of 768 -> 2048 1048 / 1067, 8 of 1024 -> 2048 1269 / 1301; 8192, 8 of 1024 -> 4096 4855 / 4977; 7548, 46 of 1600 -> 1600 3693 /
// 3764; 10617, 14 of 544 -> 1088 1375 / 1376.  Of 19 passes with 4 to 33 walks 13 were 0.4 to 2.7 % faster, six within 0.3 % of even.
static double f32_pairs(double stages) { return std::ceil(stages * F_BK / (2 * P_BK)) * (2 * P_BK / F_BK); }
static bool f32_shares(double walks, double stages, bool heavy, int p) {
    return walks <= 1.0 || (p == 1 && (heavy ? f32_pairs(stages) <= 1.1 * stages : stages > 64.0));
}
static double f32_cost(int bm, int p, int E, Rows rows, int N, int K, bool heavy) {
    const double walks = f32_tiles(bm, p, E, rows, N) / 256.0, whole = std::ceil(walks);
    const double stages = K / F_BK / (double)p, planes = p > 1 ? p * (2.0 * rows.est * N * sizeof(float) / 5.0e6) + 6.0 : 0.0;
    if (bm == 64) return std::max(1.0, (3.0 * whole + walks) / 4.0) * 0.58 * stages + (heavy ? 4.0 : 3.0) + planes;
    if (!f32_shares(walks, stages, heavy, p)) return (whole + walks) / 2.0 * (0.8 * stages + (heavy ? 6.0 : 3.0)) + planes;
    return whole * ((0.7 + 0.05 * std::min(1.0, walks)) * f32_pairs(stages) + 6.0) + planes;
}
static int f32_tile(int p, int E, Rows rows, int N, int K, bool heavy) {
    if (E <= 0 || rows.est <= 0 || N <= 64) return 64;      // (half of the columns or more are padding: 64 rows pad less)
    return f32_cost(128, p, E, rows, N, K, heavy) < f32_cost(64, p, E, rows, N, K, heavy) ? 128 : 64;
}
int gemm_f32_ksplit(int E, Rows rows, int N, int K, int room) {
    if (E <= 0 || rows.est <= 0 || K % F_BK) return 1;
    int best = 1;
    double least = 0.0;
    for (int p = 1; p <= room && (p == 1 || K / p >= 16 * F_BK); ++p) {
        const int bm = f32_tile(p, E, rows, N, K, false);
        double us = f32_cost(bm, p, E, rows, N, K, false);
        if (bm == 64 && f32_tiles(64, p, E, rows, N) <= 256.0) us += 0.1 * K / F_BK / p;      // of near equals the one with parts, whose results are closer
        if (p == 1 || us < least) { least = us; best = p; }
    }
    return best;
}

// The planes that callers laid scratch out for when a launch had tiles of own parts or fp32 operands alone, of either height, and its rows were taken to
// lie evenly: scratch of that size stays enough.  It has no say in which way a launch goes.
int gemm_f32_planes_laid_out(int E, int est_rows, int N, int K) {
    if (E <= 0 || est_rows <= 0 || K % F_BK) return 1;
    const int active = E < est_rows ? E : est_rows;
    auto us = [&](int bm, int p) {
        const long rounds = ((long)p * active * ceil_div(ceil_div(est_rows, active), bm) * ceil_div(N, 128) + 255) / 256;
        const double stages = K / F_BK / (double)p, planes = p > 1 ? p * (2.0 * est_rows * N * sizeof(float) / 5.0e6) + 6.0 : 0.0;
        return bm == 64 ? rounds * (rounds == 1 ? 0.52 : 0.47) * stages + planes : rounds * ((rounds == 1 ? 0.88 : 0.76) * stages + 3.0) + planes;
    };
    auto least = [&](int p) { return N <= 64 ? us(64, p) : std::min(us(64, p), us(128, p)); };
    int best = 1;
    for (int p = 2; p <= 4 && K / p >= 16 * F_BK; ++p)
        if (least(p) < least(best)) best = p;
    return best;
}

bool gemm_f32_takes(int N, int K) { return N >= 4 && N % 4 == 0 && K > 0 && K % F_BK == 0; }

int launch_gemm_f32(const GemmArgs &g0, bool a_ks, bool b_ks, bool wg, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid) {
    GemmArgs g = g0;
    g.ksplit = 1;
    const Rows rows{g.est_rows, g.most_rows};
    // what the direct-to-LDS path relies on: 16-byte rows, whole stages of K for row-ragged products
    if (g.lda % 4 || g.ldb % 4 || g.ldc % 4 || g.N % 4 || g.N < 4) return -100;
    if (!wg && (a_ks || !gemm_f32_takes(g.N, g.K))) return -100;
    if (wg && (!a_ks || !b_ks || g.M % 4 || g.M < 4)) return -100;
    if (wg) return dispatch_f32<128, 128, 4, 4, 2, OWN_PARTS>(g, b_ks, wg, epi, max_rows, st, kid);
    if (b_ks && g.offsets != nullptr && ws != nullptr && max_rows > 0) {
        // as many planes as the scratch has room for, at most
        const int room = planes_allowed((int)std::min<size_t>(4, ws_bytes / ((size_t)max_rows * g.N * sizeof(float))), max_rows, g.est_rows, g.N);
        const int p = gemm_f32_ksplit(g.E, rows, g.N, g.K, room);
        if (p > 1) {
            g.ksplit = p;
            g.part = (float *)ws;
            g.part_rows = max_rows;
        }
    }
    const bool heavy = epi == EPI_BIAS_GELU || epi == EPI_DGELU;
    const int e = g.ksplit > 1 ? (int)EPI_PART : epi;
    int rc;
    if (f32_tile(g.ksplit, g.E, rows, g.N, g.K, heavy) == 128) {
        if (f32_shares(f32_tiles(128, g.ksplit, g.E, rows, g.N) / 256.0, g.K / F_BK, heavy, g.ksplit)) rc = dispatch_f32<128, 128, 4, 8, 1, SHARED_PARTS>(g, b_ks, wg, e, max_rows, st, kid);
        else rc = dispatch_f32<128, 128, 4, 4, 2, OWN_PARTS>(g, b_ks, wg, e, max_rows, st, kid);
    }
    else if (g.E > 0 && g.est_rows > 0 && f32_tiles(64, g.ksplit, g.E, rows, g.N) <= 256.0) rc = dispatch_f32<64, 128, 4, 4, 3, OPERANDS>(g, b_ks, wg, e, max_rows, st, kid);
    else rc = dispatch_f32<64, 128, 4, 4, 3, OWN_PARTS>(g, b_ks, wg, e, max_rows, st, kid);
    return rc != 0 || g.ksplit == 1 ? rc : launch_plane_reduce(g, MOLE_F32, max_rows, st);
}

}  // namespace mole
