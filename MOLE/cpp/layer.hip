// The layer's forward and backward as one call each: gate, routing, dispatch, grouped FFN and combine (and their
// gradients) enqueued back to back from native code on buffers the caller laid out.
//
// Replaces the sequence of MOLEModule.forward (MOLE/moe/layer.py:440-462) and its autograd.  The kernels are those of
// the separate entry points, which these two call; what goes away is the host's work between them - a tensor
// allocation per intermediate, a foreign call with its argument conversion per step - which for short batches took
// longer than the kernels (61 tokens, 16 experts of 1024 -> 4096: 95 us of host time for 75 us of kernels).
#include "gemm.h"

#include <algorithm>
#include <cmath>

namespace mole {

// rows the experts hold in all likelihood: every pair, or the capacity's bound where that is less (the padded layout's
// buffers have a row for every slot)
static int est_rows(const mole_layer &L) { return L.rows < L.S * L.k ? L.rows : L.S * L.k; }
static Rows rows_of(const mole_layer &L) {
    // an expert takes a token once, and of those no more than the capacity
    const double capacity = L.capacity_factor > 0. ? (double)L.k * std::floor(L.capacity_factor * ((L.S + L.E - 1) / L.E)) : (double)L.S;
    return Rows{est_rows(L), capacity < L.S ? (int)capacity : L.S};
}
static size_t planes_bytes(const mole_layer &L, bool least) { return ffn_workspace_bytes(L.dtype, L.E, L.rows, est_rows(L), L.M, L.F, least); }

// Whether the first product reads the tokens through the list although their rows are written for later: where the rows of several choices are
// more than the last-level cache holds and the tokens are well below it, so that the tokens come from the cache and the rows do not.  Training
// passes and their first product, from the rows / from the tokens, us (two runs of one side differ by 0.4 % at most): rows of whole lines, 20000
// tokens, 32 experts top-4, 2048 -> 1024, 2474 / 2442 and 384 / 352; 32768, 64 top-8, 1024 -> 512, 2611 / 2587 and 394 / 359; 32768, 16 top-8, 1024 -> 512,
// skewed, 3058 / 3035 and 348 / 315; rows that share theirs with others, 30000, 64 top-8, 1000 -> 1000, 4702 / 4568 and 949 / 794; 32768, 16 top-4,
// 1400 -> 704, 2955 / 2873 and 481 / 386; fp32 16384, 32 top-8, 1008 -> 1008, 10650 / 10619 and 1759 / 1749.  On the other side of the line, tokens of
// 134 and 268 MB, passes of 32768, 256 top-8, 2048 -> 1024, 8292 / 8315; 32768, 8 top-2, 4096 -> 2048, 6434 / 6479.
static bool tokens_beside_rows(const mole_layer &L) {
    const size_t width = (size_t)L.M * (L.dtype == MOLE_BF16 ? 2 : 4);
    return L.k >= 2 && est_rows(L) * width >= (size_t)256 << 20 && L.S * width <= (size_t)96 << 20;
}

static size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

// out [ro][co] in T = in [r][c] fp32, zeros beyond, for two matrices in one launch: `first` blocks for the first.  Bound by the launch: training
// passes, a launch each / one for both, 300 tokens, 100 experts of 512 133.3 / 130.9 us; 3000, 128 of 1024 487.6 / 483.6.
struct PadConvert {
    const float *in;
    void *out;
    int r, c, ro, co;
    unsigned blocks() const { return (unsigned)(((size_t)ro * co + 255) / 256); }
};
template <typename T>
__global__ __launch_bounds__(256) void pad_convert_kernel(const PadConvert a, const PadConvert b, unsigned first) {
    const bool second = blockIdx.x >= first;
    const PadConvert &p = second ? b : a;
    const size_t i = (size_t)(blockIdx.x - (second ? first : 0)) * 256 + threadIdx.x;
    if (i >= (size_t)p.ro * p.co) return;
    const int y = (int)(i / p.co), x = (int)(i % p.co);
    ((T *)p.out)[i] = y < p.r && x < p.c ? from_f32<T>(p.in[(size_t)y * p.c + x]) : from_f32<T>(0.f);
}
template <typename T>
__global__ __launch_bounds__(256) void to_f32_kernel(const T *__restrict__ in, float *__restrict__ out, size_t n) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) out[i] = to_f32(in[i]);
}
static int pad_convert(const PadConvert &a, const PadConvert &b, int dtype, hipStream_t st) {
    const dim3 grid(a.blocks() + b.blocks());
    if (dtype == MOLE_BF16) hipLaunchKernelGGL(pad_convert_kernel<bf16_t>, grid, dim3(256), 0, st, a, b, a.blocks());
    else hipLaunchKernelGGL(pad_convert_kernel<float>, grid, dim3(256), 0, st, a, b, a.blocks());
    MOLE_LAUNCH_CHECK();
    return 0;
}

// Whether dlogits^T . x of a gate that the matrix-core kernel does not take goes by the grouped-GEMM tiles, with the result in the tokens'
// type, and not by gate_wgrad's VALU kernel, whose work grows with E M where a tile's walk over the tokens does not.  Training passes, tiles / VALU
// kernel, us: bf16, 16384 tokens, 256 experts of 1800 871 / 802, 600 of 1024 875 / 855, 1024 of 1024 1172 / 1247, 256 of 4088 1354 / 1449; 2000
// tokens of the last 533 / 533, 1000 464 / 450; fp32, 8192 tokens, 512 of 4096 2541 / 2436, 700 of 4096 3172 / 3280.
static bool gate_wgrad_may_go_by_tiles(const mole_layer &L) { return L.E > 32 && !(L.dtype == MOLE_BF16 && L.E <= 256 && L.M % 64 == 0); }
static bool gate_wgrad_by_tiles(const mole_layer &L) {
    const size_t em = (size_t)L.E * L.M;
    return gate_wgrad_may_go_by_tiles(L) && (L.dtype == MOLE_BF16 ? em > 5 << 17 && L.S > 1024 : em > 1 << 21);
}

// Scratch of the backward's gate part, and which way its two products go.
struct GateBwdPlan {
    bool fold, fold_wide;    // dlogits . Wg inside mole_dispatch_bwd (up to 32 experts) / inside dispatch_bwd_fold
    bool wgrad_tiles;        // dlogits^T . x on the grouped-GEMM tiles
    int e_pad;           // experts rounded up to the tiles' granule
    size_t dgates, dl_t, wg_t, dx_add, wgrad, total;     // bytes
};
static GateBwdPlan gate_bwd_plan(const mole_layer &L, bool wgrad_tiles) {
    GateBwdPlan p{};
    const size_t es = L.dtype == MOLE_BF16 ? 2 : 4;
    const int epc = L.dtype == MOLE_BF16 ? 8 : 4;
    p.fold = L.E <= 32;
    p.fold_wide = !p.fold && dispatch_bwd_folds(L.dtype, L.E);
    const bool product = !p.fold && !p.fold_wide;
    p.e_pad = (L.E + epc - 1) / epc * epc;
    p.dgates = L.E > 256 ? up256((size_t)L.k * L.S * 4) : 0;
    p.wgrad_tiles = wgrad_tiles;
    p.dl_t = !product && !p.wgrad_tiles ? 0 : up256((size_t)L.S * p.e_pad * es);
    p.wg_t = !product ? 0 : up256((size_t)p.e_pad * L.M * es);
    p.dx_add = !product ? 0 : up256((size_t)L.S * L.M * es);
    p.wgrad = up256(p.wgrad_tiles ? (size_t)p.e_pad * L.M * es : gate_wgrad_bytes(L.dtype, L.S, L.E, L.M));
    p.total = p.dgates + p.dl_t + p.wg_t + p.dx_add + p.wgrad;
    return p;
}

}  // namespace mole

using namespace mole;

extern "C" size_t mole_layer_workspace_bytes(const mole_layer *L, int backward) {
    if (L == nullptr || L->S <= 0 || L->E <= 0) return 0;
    const size_t ffn = planes_bytes(*L, false);
    size_t other = backward ? gate_bwd_plan(*L, gate_wgrad_by_tiles(*L)).total : mole_gate_route_shape_workspace_bytes(L->dtype, L->S, L->E, L->M, L->k);
    if (!backward && tokens_beside_rows(*L)) other = up256(other) + (size_t)L->rows * 4;
    return ffn > other ? ffn : other;        // the two are never in use at the same time
}

static int check_layer(const char *fn, const mole_layer *L, mole_stream_t) {
    MOLE_REQUIRE(L != nullptr, "%s: null argument block", fn);
    MOLE_REQUIRE(L->S >= 1 && L->rows >= 1 && L->E >= 1 && L->F >= 1, "%s: bad sizes S=%d rows=%d E=%d F=%d", fn, L->S, L->rows, L->E, L->F);
    MOLE_REQUIRE(L->x && L->wg && L->scores && L->gates && L->idx && L->row && L->counts && L->kept_rows && L->offsets && L->xd &&
                     (L->h || L->forward_only) && L->a && L->out && L->workspace, "%s: null pointer", fn);
    return 0;
}

extern "C" int mole_layer_fwd(const mole_layer *L, void *y, mole_stream_t stream) {
    if (int rc = check_layer("mole_layer_fwd", L, stream)) return rc;
    const size_t route_bytes = mole_gate_route_shape_workspace_bytes(L->dtype, L->S, L->E, L->M, L->k);
    const size_t need = std::max(route_bytes, planes_bytes(*L, false));
    if (L->workspace_bytes < std::max(gate_route_least_bytes(L->dtype, L->S, L->E, L->M, L->k), planes_bytes(*L, true))) {
        set_error("mole_layer_fwd: workspace of %zu bytes, need %zu", L->workspace_bytes, need);
        return MOLE_E_WORKSPACE;
    }
    const bool scratch = L->forward_only == 2;       // xd and out are read by nobody after this pass
    // Where nobody wants xd the first product reads the tokens where they lie: the few-row kernel, which turns the pairs' rows round by
    // itself, up to HEAD_PAIRS; the tiles from a list that the routing leaves in xd's place.  A tile's start then waits for memory once
    // more, about 0.5 us; a dispatch is a launch, writes R M elements and has them read from memory instead of the tokens from the
    // caches.  Forward passes, dispatched / from the list, us: 61 tokens, 16 experts top-1, 1024 -> 4096, 63.5 / 61.8; 3001, 16 top-2,
    // 1024 -> 4096, 169.5 / 166.5; 4000, 8 top-2, 4096 -> 2048, 341 / 328; 32768, 64 top-8, 2048 -> 1024, 2640 / 2382; 30000, 64 top-8,
    // 1000 -> 1000, whose rows share their 128-byte lines, 1712 / 1446; fp32 10000, 16 top-2, 1024 -> 1024, 661 / 641.
    // Where tokens_beside_rows, they are read so beside a dispatch, from a list in the workspace.
    // Up to HEAD_PAIRS pairs of tokens narrower than 256 keep their dispatch, which test_tokens_in_place_of_dispatched_rows counts, and not for
    // speed: dispatched / from the list, us, 400 tokens, 64 experts, 136 -> 520, 33.7 / 31.8; 512, 16, 136 -> 544, 30.7 / 28.7; fp32 512, 4, 128 -> 512,
    // 44.3 / 42.5.
    // What the dispatch would refuse, and tokens that 32-bit offsets do not reach, are left to it.
    FwdTokens takes = TOKENS_NO;
    const bool beside = !scratch && tokens_beside_rows(*L) && L->workspace_bytes >= up256(route_bytes) + (size_t)L->rows * 4;
    if ((scratch || beside) && L->k >= 1 && L->k <= 16 && ((uintptr_t)L->x & 15) == 0)
        takes = ffn_fwd_takes_tokens(L->dtype, L->E, L->rows, rows_of(*L), L->M, L->F);
    if (takes == TOKENS_PAIRS && (beside || (long)L->S * L->k > HEAD_PAIRS)) takes = TOKENS_NO;
    if (takes == TOKENS_LIST && ((size_t)L->S * L->M * (L->dtype == MOLE_BF16 ? 2 : 4) >= (size_t)1 << 31 ||
                                 (L->M < 256 && (long)L->S * L->k <= HEAD_PAIRS))) takes = TOKENS_NO;
    if (takes == TOKENS_LIST && !beside && ((uintptr_t)L->xd & 15) != 0) takes = TOKENS_NO;
    int32_t *const token_of = takes != TOKENS_LIST ? nullptr : beside ? (int32_t *)((char *)L->workspace + up256(route_bytes)) : (int32_t *)L->xd;
    if (int rc = gate_route(L->x, L->dtype, L->wg, L->logit_bias, L->S, L->E, L->M, L->k, L->capacity_factor, L->normalize_gate, 1,
                            L->layout, L->scores, L->idx, L->loc, L->gates, L->row, L->counts, L->kept_rows, L->offsets,
                            L->capacity, L->l_aux, token_of, L->workspace, L->workspace_bytes, stream)) return rc;
    const DispatchHead head{L->row, token_of, L->S, L->k};
    const bool head_ok = takes != TOKENS_NO;
    if (!head_ok || beside)
        if (int rc = mole_dispatch_fwd(L->x, L->dtype, L->row, L->S, L->M, L->k, L->xd, stream)) return rc;
    // (what the combine would refuse is left to it)
    CombineTail tail{L->row, L->idx, L->gates, y, L->S, L->k, !scratch, false};
    const bool tail_ok = y != nullptr && ((uintptr_t)y & 15) == 0 && L->k >= 1 && L->k <= 16;
    if (int rc = ffn_fwd(head_ok ? L->x : L->xd, L->dtype, L->offsets, L->kept_rows, L->E, L->rows, rows_of(*L), L->M, L->F, L->w1, L->b1, L->w2,
                         L->b2, L->h, L->a, L->out, L->workspace, L->workspace_bytes, L->forward_only, head_ok ? &head : nullptr,
                         tail_ok ? &tail : nullptr, (hipStream_t)stream)) return rc;
    if (tail.done) return 0;
    return mole_combine_fwd(L->out, L->dtype, L->row, L->gates, L->S, L->M, L->k, y, stream);
}

extern "C" int mole_layer_bwd(const mole_layer *L, const mole_layer_grads *G, mole_stream_t stream) {
    if (int rc = check_layer("mole_layer_bwd", L, stream)) return rc;
    MOLE_REQUIRE(!L->forward_only, "mole_layer_bwd: the forward pass was a forward_only one");
    MOLE_REQUIRE(G && G->dy && G->dlogits && G->d_o && G->t && G->gxd && G->dx && G->dwg, "mole_layer_bwd: null gradient pointer");
    const size_t ffn = planes_bytes(*L, true);
    GateBwdPlan p = gate_bwd_plan(*L, gate_wgrad_by_tiles(*L));
    const size_t need = std::max(planes_bytes(*L, false), p.total);
    // (a workspace that does not hold the partial sums of a large gate has its weight gradient by the tiles)
    if (L->workspace_bytes < p.total && gate_wgrad_may_go_by_tiles(*L)) p = gate_bwd_plan(*L, true);
    if (L->workspace_bytes < std::max(ffn, p.total)) {
        set_error("mole_layer_bwd: workspace of %zu bytes, need %zu", L->workspace_bytes, need);
        return MOLE_E_WORKSPACE;
    }
    hipStream_t st = (hipStream_t)stream;
    char *ws = (char *)L->workspace;
    const int32_t *counts0 = G->d_l_aux ? L->counts : nullptr;
    if (p.dgates == 0) {
        if (int rc = mole_combine_bwd_gate(G->dy, L->out, L->dtype, L->row, L->gates, L->S, L->M, L->k, G->d_o, L->scores, L->idx, L->E,
                                           L->normalize_gate, 1, counts0, G->d_l_aux, G->dlogits, stream)) return rc;
    } else {
        float *dgates = (float *)ws;
        if (int rc = mole_combine_bwd(G->dy, L->out, L->dtype, L->row, L->gates, L->S, L->M, L->k, G->d_o, dgates, stream)) return rc;
        if (int rc = mole_gate_bwd(dgates, L->scores, L->idx, L->S, L->E, L->k, L->normalize_gate, 1, counts0, G->d_l_aux, G->dlogits,
                                   stream)) return rc;
    }
    // (the FFN's scratch takes the place of dgates and makes room for the gate's products, in stream order)
    if (int rc = ffn_bwd(G->d_o, L->xd, L->h, L->a, L->dtype, L->offsets, L->kept_rows, L->E, L->rows, rows_of(*L), L->M, L->F, L->w1, L->w2,
                                 G->t, G->g_w1, G->g_b1, G->g_w2, G->g_b2, G->gxd, G->accumulate, G->gelu_bwd, L->workspace,
                                 L->workspace_bytes, st)) return rc;
    char *dl_t = ws + p.dgates, *wg_t = dl_t + p.dl_t, *dx_add = wg_t + p.wg_t, *wgrad = dx_add + p.dx_add;
    // (not where dwg lies on what the dispatch's backward or other blocks of its own still read: the launches' order then keeps them apart)
    const size_t dwg_bytes = (size_t)L->E * L->M * 4, token_bytes = (size_t)L->M * (L->dtype == MOLE_BF16 ? 2 : 4), pairs = (size_t)L->S * L->k;
    const bool dwg_apart = !overlap(G->dwg, dwg_bytes, L->wg, dwg_bytes) && !overlap(G->dwg, dwg_bytes, G->gxd, L->rows * token_bytes) &&
                           !overlap(G->dwg, dwg_bytes, L->row, pairs * 4) && !overlap(G->dwg, dwg_bytes, G->dlogits, (size_t)L->S * L->E * 4) &&
                           !overlap(G->dwg, dwg_bytes, L->x, L->S * token_bytes);
    if (!p.wgrad_tiles && dwg_apart && gate_wgrad_beside(L->dtype, L->S, L->E, L->M))
        return dispatch_bwd_gate_wgrad(G->gxd, L->row, L->S, L->M, L->k, G->dlogits, L->wg, L->E, G->dx, L->x, G->dwg, wgrad, p.wgrad, st);
    if (p.fold) {
        if (int rc = mole_dispatch_bwd(G->gxd, L->dtype, L->row, L->S, L->M, L->k, G->dlogits, L->wg, L->E, nullptr, G->dx, stream)) return rc;
    } else if (p.fold_wide) {
        // 33 to 64 experts: operands and result in bf16 like those of the product below, bit for bit, without the result's way through
        // memory and three launches less.  Training passes, by the product / folded, us: 8 tokens, 64 experts of 1024 top-2, 123.5 / 117.8;
        // 300, 40 of 1024, 175.1 / 166.9; 3000, 64 of 1024, 319.5 / 309.8; 8192, 64 of 2048, 857 / 838; 30000, 64 of 1000 top-8, 4838 / 4813;
        // 2000, 64 of 4096, 924.8 / 916.  Beyond, a wave would hold more than 64 registers of weights or read them again for every 16 tokens.
        if (int rc = dispatch_bwd_fold(G->gxd, L->row, L->S, L->M, L->k, G->dlogits, L->wg, L->E, G->dx, st)) return rc;
    } else {
        if (int rc = pad_convert({G->dlogits, dl_t, L->S, L->E, L->S, p.e_pad}, {L->wg, wg_t, L->E, L->M, p.e_pad, L->M}, L->dtype, st)) return rc;
        if (int rc = mole_gemm_nn(dl_t, wg_t, L->dtype, L->S, L->M, p.e_pad, dx_add, stream)) return rc;
        if (int rc = mole_dispatch_bwd(G->gxd, L->dtype, L->row, L->S, L->M, L->k, nullptr, nullptr, 0, dx_add, G->dx, stream)) return rc;
    }
    if (!p.wgrad_tiles) return gate_wgrad(G->dlogits, L->x, L->dtype, L->S, L->E, L->M, G->dwg, wgrad, p.wgrad, st);
    if (p.fold_wide)
        if (int rc = pad_convert({G->dlogits, dl_t, L->S, L->E, L->S, p.e_pad}, {}, L->dtype, st)) return rc;
    if (int rc = mole_gemm_tn(dl_t, L->x, L->dtype, L->S, p.e_pad, L->M, wgrad, stream)) return rc;
    const size_t n = (size_t)L->E * L->M;
    const dim3 grid((unsigned)((n + 255) / 256));
    if (L->dtype == MOLE_BF16) hipLaunchKernelGGL(to_f32_kernel<bf16_t>, grid, dim3(256), 0, st, (const bf16_t *)wgrad, G->dwg, n);
    else hipLaunchKernelGGL(to_f32_kernel<float>, grid, dim3(256), 0, st, (const float *)wgrad, G->dwg, n);
    MOLE_LAUNCH_CHECK();
    return 0;
}
