// Shared declarations of the grouped-GEMM kernels: argument block, epilogue kinds, activation math.
#pragma once
#include "common.h"

#include <math.h>

namespace mole {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------------------------
// activation math (fp32)
// ---------------------------------------------------------------------------------------------
// Phi(x) = 1/2 (1 + erf(x / sqrt 2)) and exp(-x^2 / 2), from one hardware exponential and one reciprocal: erf by the
// rational form of Abramowitz & Stegun 7.1.26 (absolute error 1.5e-7), written for the tail that is small so that
// nothing cancels: Phi(x) = q for x < 0 and 1 - q for x >= 0 with q = 1/2 t (a1 + t (a2 + ...)) exp(-x^2 / 2),
// t = 1 / (1 + p |x| / sqrt 2).  The library's erff costs about twice the instructions of everything else in an
// fp32 epilogue.
__device__ __forceinline__ float std_normal_cdf(float x, float &exp_half_sq) {
    const float y = fabsf(x) * 0.70710678118654752f;
    const float t = __builtin_amdgcn_rcpf(fmaf(0.3275911f, y, 1.0f));
    float p = 1.061405429f;
    p = fmaf(p, t, -1.453152027f);
    p = fmaf(p, t, 1.421413741f);
    p = fmaf(p, t, -0.284496736f);
    p = fmaf(p, t, 0.254829592f);
    exp_half_sq = __builtin_amdgcn_exp2f(-y * y * 1.44269504088896341f);
    const float q = 0.5f * p * t * exp_half_sq;
    return x < 0.f ? q : 1.0f - q;
}
__device__ __forceinline__ float gelu_erf(float x) {
    float e;
    return x * std_normal_cdf(x, e);
}

// derivative of the tanh-approximate GELU, term by term as MOLE/cpp/gelu.cu:3-14; tanh(u) = 1 - 2 / (1 + exp(2u)),
// which saturates correctly at both ends (exp -> inf gives 1, exp -> 0 gives -1)
__device__ __forceinline__ float d_gelu_tanh(float x) {
    const float sqrt_param = 0.79788456080286535587989211986876f;
    const float mul_param = 0.044715f;
    const float x2mul = x * x * mul_param;
    const float u = sqrt_param * (x + x * x2mul);
    // exp(2u) = 2^(hi) (1 + lo ln 2): hi + lo is the product 2u log2(e) to twice the working precision (at |u| of a few
    // units the rounding of the product alone would cost a digit of the exponential)
    const float c_hi = 2.88539008177792681f, c_lo = 2.88539008177792681 - (double)c_hi;
    const float hi = u * c_hi;
    const float lo = fmaf(u, c_hi, -hi) + u * c_lo;
    const float e2u = __builtin_amdgcn_exp2f(hi) * fmaf(lo, 0.69314718055994531f, 1.0f);
    const float tan_h = 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + e2u);
    const float dg1 = 0.5f * (1.0f + tan_h);
    const float dg2 = x * 0.5f * sqrt_param * (1.0f - tan_h * tan_h);
    const float dg3 = dg2 * 3.0f * x2mul;
    return dg1 + dg2 + dg3;
}
// derivative of the erf GELU (at::gelu_backward): Phi(x) + x*phi(x)
__device__ __forceinline__ float d_gelu_exact(float x) {
    float e;
    const float cdf = std_normal_cdf(x, e);
    return cdf + x * e * 0.39894228040143267794f;
}

// ---- activation math for a bf16 result -----------------------------------------------------------
// On this chip every VALU instruction of an epilogue takes issue time from the MFMAs of the wave that
// shares its SIMD, and exp / rcp run at a quarter of the plain rate, so the three functions are evaluated
// as clamped odd polynomials: f(x) = v q(v^2), v = clamp(x / c, -1, 1), fitted (near-minimax, Lawson
// iteration) to erf(x / sqrt 2) and to the odd parts of the two GELU derivatives.  Beyond the clamp the
// functions are constant to within the stated error.  Absolute errors in fp32 Horner evaluation:
// erf 5.8e-5, derivatives 1.8e-4 - an order of magnitude below the bf16 rounding of the result, except where the result
// itself is small (gelu(-4) = -1.3e-4).  Products whose contraction is not whole stages of 32 keep the closed forms above on
// every kernel: their loops leave the time for it, and such layers have had that accuracy from the first.
// gelu(x) = x (1/2 + 1/2 erf(x / sqrt 2)).  The fit of erf(x / sqrt 2) is v q(v^2) in v = clamp(x / 4, -1, 1); with every
// coefficient scaled by a power of two (c_k / (8 * 16^k): exact in binary floating point, the Horner steps round as
// before) the same polynomial is evaluated in v = clamp(x, -4, 4) itself and delivers 1/2 erf directly:
// clamp, square, eight FMAs, one FMA for the 1/2 and the product with x - twelve instructions, no scaling of x, no
// separate x / 2.  Beyond the clamp erf is +-1 to within the fit's error, so x (1/2 +- 1/2) is x or 0 as it should be.
__device__ __forceinline__ float fast_gelu_erf(float x) {
    constexpr float c[9] = {3.19138169f / 8.0f,
                            -8.50055408f / (8.0f * 16.0f),
                            20.229044f / (8.0f * 256.0f),
                            -37.1561737f / (8.0f * 4096.0f),
                            51.8556824f / (8.0f * 65536.0f),
                            -52.8050575f / (8.0f * 1048576.0f),
                            36.4542885f / (8.0f * 16777216.0f),
                            -15.039053f / (8.0f * 268435456.0f),
                            2.77038407f / (8.0f * 4294967296.0f)};
    const float v = __builtin_amdgcn_fmed3f(x, -4.0f, 4.0f);
    const float t = v * v;
    float q = c[8];
#pragma unroll
    for (int k = 7; k >= 0; --k) q = fmaf(q, t, c[k]);
    return x * fmaf(v, q, 0.5f);
}
// The two GELU derivatives share the clamp (4.5) and the degree, so the variant is a choice of coefficients,
// made once per tile, not a branch per element: tanh form = what the reference's backward multiplies by
// (MOLE/cpp/gelu.cu:3-14), exact form = Phi(x) + x phi(x).  d(x) = 1/2 + v q(v^2), v = clamp(x / 4.5, -1, 1); as above
// the polynomial is evaluated in v = clamp(x, -4.5, 4.5) with the coefficients divided by 4.5^(2k+1) (in double
// precision, then rounded once: 4.5 is not a power of two).
struct DGeluCoef {
    float c[10];
    __device__ __forceinline__ void select(bool tanh_form) {
        constexpr double ct[10] = {3.58895016, -24.237009, 110.279869, -345.395355, 772.538513,
                                   -1226.4845, 1338.11902, -946.521179, 388.703674, -70.0920258};
        constexpr double ce[10] = {3.58931732, -24.1413288, 108.150215, -329.418243, 711.674683,
                                   -1091.27979, 1154.8053, -796.700195, 320.776367, -56.9563408};
        double s = 1.0 / 4.5;
#pragma unroll
        for (int i = 0; i < 10; ++i) {
            c[i] = (float)((tanh_form ? ct[i] : ce[i]) * s);
            s *= 1.0 / (4.5 * 4.5);
        }
    }
    __device__ __forceinline__ float operator()(float x) const {
        const float v = __builtin_amdgcn_fmed3f(x, -4.5f, 4.5f);
        const float t = v * v;
        float q = c[9];
#pragma unroll
        for (int k = 8; k >= 0; --k) q = fmaf(q, t, c[k]);
        return fmaf(v, q, 0.5f);
    }
};

enum { EPI_STORE = 0, EPI_BIAS = 1, EPI_BIAS_GELU = 2, EPI_DGELU = 3, EPI_WGRAD = 4, EPI_F32 = 5,
       EPI_PART = 6 /* one plane of a contraction split over blocks: fp32 into GemmArgs.part */,
       EPI_NONE = 7 /* measurement only: the K loop runs, nothing is stored; EPI_NONE + 1..4: the K loop without
                       its operand loads / its fragment reads / its barriers / all three */ };

// The combine behind out = a.w2 + b2, y[i] = sum over the k choices of gates[j][i] out[row[j][i]], for the reduction of a split
// contraction to do on its way (layer.hip).  done: it has.
struct CombineTail {
    const int32_t *row, *idx;   // [k][S] row of a pair (-1: dropped), its expert
    const float *gates;         // [k][S]
    void *y;                    // [S][N]
    int S, k;
    bool keep_out;              // out is read after the pass (by a backward pass or the caller)
    bool done;
};

// The dispatch in front of h = xd.w1^T + b1, xd[row[j][i]] = x[i], for the product to do as it reads its rows (layer.hip): the few-row
// kernel turns row round by itself, the tiles take the routing's list.
struct DispatchHead {
    const int32_t *row;     // [k][S] row of a pair (-1: dropped)
    const int32_t *token_of;    // token of a row (tiles; null: few-row kernel)
    int S, k;
};
constexpr int HEAD_PAIRS = 512;     // most pairs, one per thread of a block

struct GemmArgs {
    const void *A, *B;      // operands (see A_KS / B_KS for their layout)
    void *C, *C2;           // outputs; C2 = gelu(h) for EPI_BIAS_GELU, whose C may be null (h is then not stored)
    const void *bias;       // [E][N] for EPI_BIAS*, else unused
    const void *H;          // [rows][N] pre-activation for EPI_DGELU
    const int32_t *offsets; // [E] first row of every expert (NULL: one group starting at row 0)
    const int32_t *kept;    // [E] rows of every expert (NULL: single_rows)
    int single_rows;
    int E;
    int M;                  // output rows per expert for weight gradients (F), unused for row-ragged
    int N, K;               // N output columns; K contraction length (row-ragged products)
    long lda, ldb, ldc;
    long strideB;           // elements between experts in B (row-ragged) -- weights
    long strideC;           // elements between experts in C (weight gradients)
    int m_tiles_bound;      // upper bound of the number of m-tiles over all experts (row-ragged)
    int accumulate;         // EPI_WGRAD: add into C
    int gelu_bwd;           // EPI_DGELU: MOLE_GELU_BWD_*
    int n_blocks;           // real number of tiles in the launch (grid is rounded up to 8)
    void *colsum;           // weight gradients, direct-to-LDS kernels: [E][M] (side 1) or [E][N] (side 2) sums of an operand
    int colsum_side;        //   over the expert's rows: 1 = the m-side operand (A), 2 = the n-side operand (B)
    int wg_expert_major;    // weight gradients, 256-wide kernel: all (m-tile, n-tile) blocks of an expert on one XCD
    int m_fastest_from;     //   ... for experts with at least this many m-tiles (of the class); the others n-tile first
    float *part;            // fp32 partial results [ksplit][part_rows][N] of a contraction split over blocks
    long part_rows;
    int ksplit;
    int once;               // row-ragged products with K-strided weights: see weights_pass_by()
    int est_rows;           // host's estimate of the rows of all experts together (no more than the launch's bound)
    int most_rows;          // the most rows that one expert can have
    CombineTail *tail;      // host side only: see CombineTail (null: none)
    const int32_t *pair_row;    // A is the tokens and not their dispatched rows: [pairs], pair p is token p % tokens (null: it is the rows)
    int pairs, tokens;
    const int32_t *token_of;    // A is the tokens and its row r token token_of[r] (null: A is the rows); EPI_BIAS_GELU by tiles
    int m_fastest;          // row-ragged products, 256-wide kernel: number an expert's tiles m-tile first (see gemm256.hip)
};


// 256x256 bf16 tiles with direct-to-LDS loads (gemm256.hip).  Returns -100 when the shape does not
// meet its alignment requirements; the caller then uses the generic kernel.
int launch_gemm256(const GemmArgs &g, bool a_ks, bool b_ks, bool wg, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid);
// ... a row-ragged product of the backward pass and a weight gradient in one launch; -100 where they have no kernel in common.
int launch_gemm256_pair(const GemmArgs &g, const GemmArgs &w, bool b_ks, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid);
// planes a K = F product of est_rows rows over E experts would be split into, given the workspace (1: none)
int gemm256_ksplit(int E, int est_rows, int N, int K);
// out = sum of the planes (+ bias), for the rows of g's experts (gemm_skinny.hip)
int launch_plane_reduce(const GemmArgs &g, int dtype, int max_rows, hipStream_t st);
bool gemm256_sums_operand(const GemmArgs &g);
// Planes of a split that asks for ks.  A plane has a row for every row of the launch's buffers, also where few of them are
// used: the padded layout holds E C rows however few are routed (1 token, top-2 of 256 experts, capacity factor 2,
// 2048 -> 4096: 1024 rows for 2, 67 MB in eight planes).  Beyond four times the rows that can be used, 32 MB in all.
inline int planes_allowed(int ks, int max_rows, int est_rows, int N) {
    if (max_rows <= 4ll * est_rows) return ks;
    const long long fit = (32ll << 20) / ((long long)max_rows * N * (long long)sizeof(float));
    return fit < 2 ? 1 : (ks < fit ? ks : (int)fit);
}
// Few rows per expert (gemm_skinny.hip): weights streamed straight into fragments; -100 when the shape is not its.
int launch_gemm_skinny(const GemmArgs &g, int dtype, bool b_ks, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid);
bool gemm_skinny_takes(const GemmArgs &g, int dtype, bool b_ks, int max_rows, void *ws, size_t ws_bytes);
bool gemm_skinny_takes_tokens(int E, int max_rows, int est_rows, int N, int K, int dtype);    // as dispatched by a DispatchHead
int gemm_skinny_ksplit(int E, int max_rows, int est_rows, int N, int K, int dtype);    // 0: not its shape
// fp32 tiles with direct-to-LDS loads (gemm_f32.hip); -100 as above.
int launch_gemm_f32(const GemmArgs &g, bool a_ks, bool b_ks, bool wg, int epi, int max_rows, void *ws, size_t ws_bytes, hipStream_t st, int kid);
int gemm_f32_ksplit(int E, Rows rows, int N, int K, int room);      // of at most `room` planes
int gemm_f32_planes_laid_out(int E, int est_rows, int N, int K);
bool gemm_f32_takes(int N, int K);      // the widths of a row-ragged product
bool gemm_f32_sums_operand(const GemmArgs &g);

}  // namespace mole
