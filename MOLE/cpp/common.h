// Shared helpers of the gfx950 kernels: error plumbing, bf16 <-> fp32, wave-level primitives.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>
#include <stdio.h>
#include <stdarg.h>

#include "mole_hip.h"

namespace mole {

void set_error(const char *fmt, ...);

#define MOLE_REQUIRE(cond, ...)                 \
    do {                                        \
        if (!(cond)) {                          \
            mole::set_error(__VA_ARGS__);       \
            return MOLE_E_INVALID;              \
        }                                       \
    } while (0)

#define MOLE_HIP(call)                                                                   \
    do {                                                                                 \
        hipError_t e_ = (call);                                                          \
        if (e_ != hipSuccess) {                                                          \
            mole::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, __LINE__); \
            return (int)e_;                                                              \
        }                                                                                \
    } while (0)

// after a kernel launch: report launch-configuration errors without synchronising
#define MOLE_LAUNCH_CHECK()                                                              \
    do {                                                                                 \
        hipError_t e_ = hipGetLastError();                                               \
        if (e_ != hipSuccess) {                                                          \
            mole::set_error("kernel launch failed: %s (%s:%d)", hipGetErrorString(e_), __FILE__, __LINE__); \
            return (int)e_;                                                              \
        }                                                                                \
    } while (0)

typedef __bf16 bf16_t;

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f32(float v);
template <> __device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return (bf16_t)v; }  // round to nearest even

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t lo16) { return __uint_as_float(lo16 << 16); }

constexpr int WAVE = 64;

__device__ __forceinline__ int lane_id() { return threadIdx.x & (WAVE - 1); }

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int m = WAVE / 2; m >= 1; m >>= 1) v += __shfl_xor(v, m, WAVE);
    return v;
}

// Sums of all lanes up to and with each lane (the whole wave has to be active).  DPP moves lanes on the vector ALU: within rows of
// 16, then lane 15 into the next row and lane 31 into the upper half.  Six steps of __shfl_up go through the LDS crossbar and
// wait for it each time.  Every block of a ragged product begins with a search for its tile among the experts: 2.0 us with
// those, 1.6 with these, most of it the loads of the experts' rows; passes of 1, 61 and 256 tokens 52.4, 74.4, 433 -> 51.4, 72.8,
// 425 us, a training pass of 16 experts of 128 rows 123 -> 119.6.
__device__ __forceinline__ int wave_scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, false);      // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);      // row_bcast 15 into rows 1 and 3
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);      // row_bcast 31 into rows 2 and 3
    return v;
}
__device__ __forceinline__ int wave_total(int scanned) { return __builtin_amdgcn_readlane(scanned, WAVE - 1); }

static inline int ceil_div(int a, int b) { return (a + b - 1) / b; }

// optional per-kernel timing (see error.cpp); ids are the MOLE_K_* of mole_hip.h
bool timing_enabled();
void timing_begin(int id, hipStream_t st);
void timing_end(hipStream_t st);
struct ScopedTiming {
    hipStream_t st;
    bool on;
    ScopedTiming(int id, hipStream_t s) : st(s), on(timing_enabled()) { if (on) timing_begin(id, st); }
    ~ScopedTiming() { if (on) timing_end(st); }
};

// One kernel under a timing id.  With timing on, the launch carries its own start/stop events, which take the
// kernel's begin and end from its dispatch packet: the measured time is the kernel's run time, as a profiler
// sees it.  (An event pair recorded around a launch adds two marker packets to the stream, about 2.4 us - a
// fifth of a 12 us kernel.)  ScopedTiming remains for entry points that launch several kernels under one id.
void timing_events(int id, hipEvent_t *start, hipEvent_t *stop);
template <typename... KArgs, typename... Args>
inline void timed_launch(int id, void (*kernel)(KArgs...), dim3 grid, dim3 block, unsigned lds, hipStream_t st,
                         Args... args) {
    if (timing_enabled()) {
        hipEvent_t a, b;
        timing_events(id, &a, &b);
        hipExtLaunchKernelGGL(kernel, grid, block, lds, st, a, b, 0, static_cast<KArgs>(args)...);
    } else {
        hipLaunchKernelGGL(kernel, grid, block, lds, st, static_cast<KArgs>(args)...);
    }
}

// dWg = dlogits^T . x of a gate of any size, with a workspace of gate_wgrad_bytes (permute.hip)
size_t gate_wgrad_bytes(int dtype, int S, int E, int M);
int gate_wgrad(const float *dlogits, const void *x, int dtype, int S, int E, int M, float *dwg, void *workspace, size_t workspace_bytes, hipStream_t st);

// the dispatch's backward with the gate's input gradient from bf16 operands, beyond the 32 experts of mole_dispatch_bwd's own (permute.hip)
bool dispatch_bwd_folds(int dtype, int E);
bool gate_wgrad_beside(int dtype, int S, int E, int M);      // dispatch_bwd_gate_wgrad takes the two in one launch
inline bool overlap(const void *p, size_t np, const void *q, size_t nq) {      // of np bytes at p and nq at q
    return p != nullptr && q != nullptr && (uintptr_t)p < (uintptr_t)q + nq && (uintptr_t)q < (uintptr_t)p + np;
}
int dispatch_bwd_gate_wgrad(const void *dxd, const int32_t *row, int S, int M, int k, const float *dlogits, const float *wg, int E, void *dx, const void *x, float *dwg, void *workspace,
                            size_t workspace_bytes, hipStream_t st);
int dispatch_bwd_fold(const void *dxd, const int32_t *row, int S, int M, int k, const float *dlogits, const float *wg, int E, void *dx, hipStream_t st);

struct CombineTail;     // gemm.h
struct DispatchHead;
// what the caller knows of the rows beside their bound: how many all experts hold in all likelihood, and the most that one can hold
struct Rows { int est, most; };
// the FFN's entry points with these (ffn_gemm.hip)
size_t ffn_workspace_bytes(int dtype, int E, int max_rows, int est_rows, int M, int F, bool least);     // least: what a call needs at least
size_t gate_route_least_bytes(int dtype, int S, int E, int M, int k);     // gate_route's without small blocks
int gate_route(const void *x, int dtype, const float *wg, const float *logit_bias, int S, int E, int M, int k, double capacity_factor,
               int normalize_gate, int alignment, int layout, float *scores, int32_t *idx, int32_t *loc, float *gates, int32_t *row, int32_t *counts,
               int32_t *kept_rows, int32_t *offsets, int32_t *capacity, float *l_aux, int32_t *token_of, void *workspace, size_t workspace_bytes,
               mole_stream_t stream);
int ffn_fwd(const void *xd, int dtype, const int32_t *offsets, const int32_t *kept_rows, int E, int max_rows, Rows rows, int M, int F,
            const void *w1, const void *b1, const void *w2, const void *b2, void *h, void *a, void *out, void *workspace,
            size_t workspace_bytes, int forward_only, const DispatchHead *head, CombineTail *tail, hipStream_t st);     // head: xd is the tokens
// Whether h = xd.w1^T + b1 can read the tokens where they lie: not at all, from the pairs' rows or from the list of the rows' tokens
enum FwdTokens { TOKENS_NO, TOKENS_PAIRS, TOKENS_LIST };
FwdTokens ffn_fwd_takes_tokens(int dtype, int E, int max_rows, Rows rows, int M, int F);
int ffn_bwd(const void *go, const void *xd, const void *h, const void *a, int dtype, const int32_t *offsets, const int32_t *kept_rows, int E,
            int max_rows, Rows rows, int M, int F, const void *w1, const void *w2, void *t, void *g_w1, void *g_b1, void *g_w2, void *g_b2,
            void *gx, int accumulate, int gelu_bwd, void *workspace, size_t workspace_bytes, hipStream_t st);

}  // namespace mole
