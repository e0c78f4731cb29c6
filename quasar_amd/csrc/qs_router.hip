// qs_router.hip - the mixture-of-experts router's expert choice on the device: per token,
// the softmax of its router logits and the n_used most probable experts, with the
// optional renormalisation of their weights (forward_cpu.c:296-304 with the softmax of
// forward_cpu.c:165-172), bit for bit.
//
// Four tokens per wavefront, one per 16-lane row: n_expert <= 256 logits, lane l of a row
// holding experts l, l+16, ... (NQ of them: 4, 8 or 16).  Maxima and arg-maxima are row
// reductions over DPP moves (quad permutes and the half-row and row mirrors: every lane of the
// row ends with the result).  The reference's sums are sequential float sums in expert (or
// slot) order, which no tree reproduces: every lane adds its row's numerators in expert order
// out of an LDS copy (broadcast reads, 32 numerators read ahead of the 32 being added); the
// slot-order sum of the chosen weights is kept by every lane as the choices are made.  The
// expf is the library's libm-equal routine.  The choice is a sequence of row arg-maxima: the
// largest probability, then the lowest index that holds it (the reference's strict `>` scan
// from index 0), and never a NaN.
//
// What bounds it: one wavefront a SIMD at 4096 tokens (2.4 MB, under a microsecond of HBM), so
// the time is one wavefront's instructions and their latencies.  4096 tokens x 128 experts,
// top 8: 10.6 us with 64-bit (probability, ~index) keys, the experts of a lane guarded one by
// one and each numerator's read waited for by its additions; 7.1 us (5.8 of kernel,
// the rest the host's launch) with 32-bit keys, the
// experts of a lane fixed by the kernel and the reads ahead.

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>

#include "../../include/quasar_sampler.h"
#include "qs_device.h"
#include "qs_internal.h"

namespace {

using namespace qs;

constexpr int RT_WAVES = 4;          // wavefronts per workgroup
constexpr int RT_TOK = 4;            // tokens per wavefront (16 lanes each)
constexpr int RT_MAX_E = 256;        // experts (forward_cpu.c:299 keeps taken[256])
constexpr int RT_MAX_U = 64;         // experts used (forward_cpu.c:298 keeps idx[64])

__constant__ uint64_t c_exp_tab_r[QS_EXPF_TAB_N] = QS_EXPF_TABLE_INIT;

// A probability's key: its bits + 1 (never negative, so the bits order them; +0 is 1); 0 is
// never chosen (NaN, and lanes past the experts).
__device__ __forceinline__ uint32_t choice_key(float p) {
    return p == p ? __float_as_uint(p) + 1u : 0u;
}

// Reductions over each 16-lane row; every lane of the row gets the row's result.
template <typename T, typename F>
__device__ __forceinline__ T row_reduce(T v, F &&op) {
    v = op(v, dpp_move<0xB1, 0xF>(v));      // quad_perm [1,0,3,2]
    v = op(v, dpp_move<0x4E, 0xF>(v));      // quad_perm [2,3,0,1]
    v = op(v, dpp_move<0x141, 0xF>(v));     // row_half_mirror
    v = op(v, dpp_move<0x140, 0xF>(v));     // row_mirror
    return v;
}

// expf of x <= 0 or NaN, as qs_expf_tab gives it.
__device__ __forceinline__ float expf_neg(float x, const uint64_t *tab) {
    const float y = qs_expf_core(x, tab);
    return x >= -0x1.9fe368p6f ? y : (x != x ? x : 0.0f);
}

// NQ: experts per lane; NS: chosen slots per lane (slot s on lane s % 16).
template <int NQ, int NS>
__global__ void __launch_bounds__(64 * RT_WAVES)
k_router(const float *logits, int64_t stride, int n_tokens, int n_expert, int n_used,
         int norm, int32_t *out_idx, float *out_wt) {
    __shared__ uint64_t tab[QS_EXPF_TAB_N];
    __shared__ __attribute__((aligned(16))) float num[RT_WAVES][RT_TOK][16 * NQ];   // numerators
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int row = lane >> 4, l16 = lane & 15;
    const int64_t t = ((int64_t)blockIdx.x * RT_WAVES + wv) * RT_TOK + row;
    const bool live = t < n_tokens;
    const float *a = logits + (live ? t * stride : 0);
    float v[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const int e = 16 * q + l16;
        v[q] = e < n_expert ? a[e] : -INFINITY;
    }
    const float a0 = a[0];
    if (threadIdx.x < QS_EXPF_TAB_N) tab[threadIdx.x] = c_exp_tab_r[threadIdx.x];
    __syncthreads();

    // forward_cpu.c:166-167: mx = a[0], then every later a[i] > mx replaces it: a NaN
    // a[0] stays, later NaNs never enter.  fmaxf drops NaNs the same way.
    float m = -INFINITY;
#pragma unroll
    for (int q = 0; q < NQ; ++q) m = fmaxf(m, v[q]);
    m = row_reduce(m, [](float x, float y) { return fmaxf(x, y); });
    const float mx = (a0 != a0) ? a0 : m;

    // forward_cpu.c:169-171: e = expf(a - mx); sum in order; inv = 1/sum; p = e * inv (the
    // copy's places past the experts hold 0: adding it changes no sum)
    float *nrow = num[wv][row];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        v[q] = expf_neg(v[q] - mx, tab);
        nrow[16 * q + l16] = 16 * q + l16 < n_expert ? v[q] : 0.0f;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float sum = 0.0f;
    {
        constexpr int AH = 8;                       // float4s read ahead
        const float4 *n4 = (const float4 *)nrow;
        float4 f[2][AH];
#pragma unroll
        for (int i = 0; i < AH; ++i) f[0][i] = n4[i];
#pragma unroll
        for (int c = 0; c < NQ * 4 / AH; ++c) {
            if (c + 1 < NQ * 4 / AH) {
#pragma unroll
                for (int i = 0; i < AH; ++i) f[(c + 1) & 1][i] = n4[AH * (c + 1) + i];
            }
#pragma unroll
            for (int i = 0; i < AH; ++i) {
                sum += f[c & 1][i].x;
                sum += f[c & 1][i].y;
                sum += f[c & 1][i].z;
                sum += f[c & 1][i].w;
            }
        }
    }
    const float inv = 1.0f / sum;
    uint32_t key[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        v[q] = v[q] * inv;
        key[q] = 16 * q + l16 < n_expert ? choice_key(v[q]) : 0u;
    }

    // forward_cpu.c:300-303: n_used arg-maxima; a slot with nothing left to take (all
    // remaining probabilities NaN) reports expert -1 with weight 0.  forward_cpu.c:304: sm
    // is the weights' sum in slot order; if sm > 0 each is divided by it.
    float wt_mine[NS];
    int idx_mine[NS];
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        wt_mine[j] = 0.0f;
        idx_mine[j] = -1;
    }
    float sm = 0.0f;
    for (int s = 0; s < n_used; ++s) {
        uint32_t k = key[0];
#pragma unroll
        for (int q = 1; q < NQ; ++q) k = max(k, key[q]);
        const uint32_t best = row_reduce(k, [](uint32_t x, uint32_t y) { return max(x, y); });
        uint32_t mine = 0xFFFFFFFFu;                // this lane's lowest expert holding it
#pragma unroll
        for (int q = NQ - 1; q >= 0; --q)
            if (key[q] == best) mine = 16u * q;
        const uint32_t at =
            row_reduce(mine == 0xFFFFFFFFu ? mine : mine + (uint32_t)l16,
                       [](uint32_t x, uint32_t y) { return min(x, y); });
        const uint32_t d = at - (uint32_t)l16;      // 16 q in the lane that holds it
#pragma unroll
        for (int q = 0; q < NQ; ++q)
            if (d == 16u * q) key[q] = 0u;          // taken
        const bool any = best != 0u;
        const float w = any ? __uint_as_float(best - 1u) : 0.0f;
        sm += w;
#pragma unroll
        for (int j = 0; j < NS; ++j)
            if (16 * j + l16 == s) {
                wt_mine[j] = w;
                idx_mine[j] = any ? (int)at : -1;
            }
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const int s = 16 * j + l16;
        if (live && s < n_used) {
            out_idx[t * n_used + s] = idx_mine[j];
            out_wt[t * n_used + s] = (norm && sm > 0.0f) ? wt_mine[j] / sm : wt_mine[j];
        }
    }
}

}  // namespace

extern "C" {

int qs_router_topk(const float *d_logits, int64_t row_stride, int n_tokens, int n_expert,
                   int n_used, int norm_topk, int32_t *d_idx, float *d_wt, void *stream) {
    if (!d_logits || !d_idx || !d_wt || n_tokens < 0 || n_expert < 1 ||
        n_expert > RT_MAX_E || n_used < 1 || n_used > RT_MAX_U || n_used > n_expert ||
        row_stride < n_expert) {
        qs_set_error("qs_router_topk: bad arguments");
        return QS_EINVAL;
    }
    if (n_tokens == 0) return 0;
    const int64_t per_block = (int64_t)RT_WAVES * RT_TOK;
    const unsigned blocks = (unsigned)(((int64_t)n_tokens + per_block - 1) / per_block);
    static_assert(RT_MAX_E == 16 * 16 && RT_MAX_U == 16 * 4, "the kernels below");
    auto *k = n_used <= 16 ? (n_expert <= 64    ? k_router<4, 1>
                              : n_expert <= 128 ? k_router<8, 1>
                                                : k_router<16, 1>)
                           : (n_expert <= 64    ? k_router<4, 4>
                              : n_expert <= 128 ? k_router<8, 4>
                                                : k_router<16, 4>);
    hipLaunchKernelGGL(k, dim3(blocks), dim3(64 * RT_WAVES), 0, (hipStream_t)stream, d_logits,
                       row_stride, n_tokens, n_expert, n_used, norm_topk ? 1 : 0, d_idx, d_wt);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        qs_set_error("k_router launch: %s", hipGetErrorString(e));
        return QS_EDEVICE;
    }
    return 0;
}

int qs_router_time(const float *d_logits, int64_t row_stride, int n_tokens, int n_expert,
                   int n_used, int norm_topk, int32_t *d_idx, float *d_wt, int iters,
                   float *ms) {
    if (iters < 1 || !ms) {
        qs_set_error("qs_router_time: bad arguments");
        return QS_EINVAL;
    }
    hipStream_t st = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    int rc = 0;
    if (hipStreamCreateWithFlags(&st, hipStreamNonBlocking) != hipSuccess ||
        hipEventCreate(&e0) != hipSuccess || hipEventCreate(&e1) != hipSuccess) {
        qs_set_error("qs_router_time: stream or event creation failed");
        rc = QS_EDEVICE;
    }
    if (!rc && hipEventRecord(e0, st) != hipSuccess) rc = QS_EDEVICE;
    for (int i = 0; !rc && i < iters; ++i)
        rc = qs_router_topk(d_logits, row_stride, n_tokens, n_expert, n_used, norm_topk, d_idx,
                            d_wt, st);
    if (!rc && (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                hipEventElapsedTime(ms, e0, e1) != hipSuccess)) {
        qs_set_error("qs_router_time: timing failed");
        rc = QS_EDEVICE;
    }
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    if (st) (void)hipStreamDestroy(st);
    return rc;
}

}  // extern "C"
