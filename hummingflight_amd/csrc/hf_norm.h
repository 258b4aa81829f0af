// hf_norm.h -- RMSNorm of one row by a 256-thread block, into LDS
// (glm_forward.cpp:185-197), for kernels that multiply a normalised row and
// would otherwise wait for a launch that writes it.
#pragma once

#include "hf_common.h"

namespace hf {

// The norm of a row a kernel normalises itself: weight (null: ones), epsilon.
struct RowNorm {
    const uint16_t* w;
    float eps;
};

constexpr int kRowNormThreads = 256;  // the block
constexpr int kNormThreads = 1024;    // rmsnorm_kernel's block, whose sums these are

// x * r * w of the K values at x (16-byte aligned, K a multiple of 4, at most
// 512 KCH) into xa / xb: chunk ch = values 8 ch .. 8 ch + 7 as halves xa[ch],
// xb[ch], zeros from K on.  Thread t stands for rmsnorm_kernel's threads
// t + 256 m, in its order: the same bits.  red: [kNormThreads / 64] LDS floats.
// The caller synchronises the block before it reads xa / xb.
template <int KCH>
__device__ __forceinline__ void stage_rmsnorm(const float* __restrict__ x, const uint16_t* __restrict__ w, float eps,
                                              int K, float4* xa, float4* xb, float* red) {
    constexpr int M = kNormThreads / kRowNormThreads, J = (KCH * 512 + 4 * kNormThreads - 1) / (4 * kNormThreads);
    const int t = threadIdx.x;
    float4 v[M][J];
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int i = 4 * (t + m * kRowNormThreads + j * kNormThreads);
            v[m][j] = i < K ? *reinterpret_cast<const float4*>(x + i) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
#pragma unroll
    for (int m = 0; m < M; ++m) {
        float sq = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            sq = fmaf(v[m][j].x, v[m][j].x, sq);
            sq = fmaf(v[m][j].y, v[m][j].y, sq);
            sq = fmaf(v[m][j].z, v[m][j].z, sq);
            sq = fmaf(v[m][j].w, v[m][j].w, sq);
        }
        sq = wave_sum(sq);
        if ((t & 63) == 0) red[(t >> 6) + m * (kRowNormThreads / 64)] = sq;
    }
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) tot += red[i];
    const float r = 1.0f / sqrtf(tot / (float)K + eps);
    auto wt = [&](int i) { return w ? __uint_as_float((uint32_t)w[i] << 16) : 1.0f; };
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int i = 4 * (t + m * kRowNormThreads + j * kNormThreads);
            if (i >= KCH * 512) continue;
            const float4 h = v[m][j];
            ((i >> 2) & 1 ? xb : xa)[i >> 3] =
                i < K ? make_float4(h.x * r * wt(i), h.y * r * wt(i + 1), h.z * r * wt(i + 2), h.w * r * wt(i + 3))
                      : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
}

}  // namespace hf
