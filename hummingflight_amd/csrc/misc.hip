// misc.hip -- RMSNorm and residual add around the MoE block
// (glm_forward.cpp:185-197 and :785-796).
#include "hf_api_internal.h"
#include "hf_norm.h"

namespace hf {

// One block of 1024 threads per token: r = 1/sqrt(sum(x^2)/n + eps);
// out = x*r*w (w BF16 or 1).  Each thread loads its (at most two) float4
// chunks once and keeps them in registers for the second pass, so a token
// costs one round trip to memory, not two.
__global__ __launch_bounds__(kNormThreads) void rmsnorm_kernel(const float* __restrict__ h,
                                                               const uint16_t* __restrict__ w,
                                                               float* __restrict__ out, int d, float eps) {
    __shared__ float red[kNormThreads / 64];
    const float* x = h + (size_t)blockIdx.x * d;
    float* y = out + (size_t)blockIdx.x * d;
    const bool vec = (d & 3) == 0;
    float4 v[2];
    float sq = 0.0f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = 4 * (threadIdx.x + j * kNormThreads);
        v[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (vec && i < d) v[j] = *reinterpret_cast<const float4*>(x + i);
        sq = fmaf(v[j].x, v[j].x, sq);
        sq = fmaf(v[j].y, v[j].y, sq);
        sq = fmaf(v[j].z, v[j].z, sq);
        sq = fmaf(v[j].w, v[j].w, sq);
    }
    if (!vec)
        for (int i = threadIdx.x; i < d; i += kNormThreads) sq = fmaf(x[i], x[i], sq);
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) tot += red[i];
    const float r = 1.0f / sqrtf(tot / (float)d + eps);
    auto wt = [&](int i) { return w ? __uint_as_float((uint32_t)w[i] << 16) : 1.0f; };
    if (vec) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int i = 4 * (threadIdx.x + j * kNormThreads);
            if (i < d)
                *reinterpret_cast<float4*>(y + i) =
                    make_float4(v[j].x * r * wt(i), v[j].y * r * wt(i + 1), v[j].z * r * wt(i + 2), v[j].w * r * wt(i + 3));
        }
    } else {
        for (int i = threadIdx.x; i < d; i += kNormThreads) y[i] = x[i] * r * wt(i);
    }
}

// The same for d a multiple of 4, straight to the BF16 hi / lo halves that the
// multi-token GEMMs read (hi = RNE(y), lo = RNE(y - hi), as split_bf16_kernel;
// *flag = 1 when any lo half is nonzero): neither the FP32 rows nor a launch
// between the norm and the GEMMs.
__global__ __launch_bounds__(kNormThreads) void rmsnorm_split_kernel(const float* __restrict__ h,
                                                                     const uint16_t* __restrict__ w,
                                                                     uint16_t* __restrict__ hi,
                                                                     uint16_t* __restrict__ lo, int d, float eps,
                                                                     unsigned* __restrict__ flag) {
#pragma clang fp contract(off)  // lo is what the rounded y leaves, not the exact product
    __shared__ float red[kNormThreads / 64];
    const size_t row = (size_t)blockIdx.x * d;
    float4 v[2];
    float sq = 0.0f;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = 4 * (threadIdx.x + j * kNormThreads);
        v[j] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (i < d) v[j] = *reinterpret_cast<const float4*>(h + row + i);
        sq = fmaf(v[j].x, v[j].x, sq);
        sq = fmaf(v[j].y, v[j].y, sq);
        sq = fmaf(v[j].z, v[j].z, sq);
        sq = fmaf(v[j].w, v[j].w, sq);
    }
    sq = wave_sum(sq);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = sq;
    __syncthreads();
    float tot = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormThreads / 64; ++i) tot += red[i];
    const float r = 1.0f / sqrtf(tot / (float)d + eps);
    auto wt = [&](int i) { return w ? __uint_as_float((uint32_t)w[i] << 16) : 1.0f; };
    bool nz = false;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int i = 4 * (threadIdx.x + j * kNormThreads);
        if (i < d) {
            const float y[4] = {v[j].x * r * wt(i), v[j].y * r * wt(i + 1), v[j].z * r * wt(i + 2), v[j].w * r * wt(i + 3)};
            uint32_t hw[4], lw[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                hw[q] = f32_to_bf16(y[q]);
                lw[q] = f32_to_bf16(y[q] - __uint_as_float(hw[q] << 16));
                nz |= (lw[q] & 0x7FFFu) != 0;
            }
            *reinterpret_cast<uint2*>(hi + row + i) = make_uint2(hw[0] | (hw[1] << 16), hw[2] | (hw[3] << 16));
            *reinterpret_cast<uint2*>(lo + row + i) = make_uint2(lw[0] | (lw[1] << 16), lw[2] | (lw[3] << 16));
        }
    }
    if (__ballot(nz) != 0ull && (threadIdx.x & 63) == 0) *flag = 1u;
}

__global__ void add_inplace_kernel(float* __restrict__ dst, const float* __restrict__ src, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] += src[i];
}

// n floats from src to dst, either of which may be mapped host memory: a
// small transfer done by the compute queue, without a DMA-engine round trip.
__global__ void copy_f32_kernel(const float* __restrict__ src, float* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy_f32(const float* src, float* dst, size_t n, hipStream_t s) {
    size_t blocks = (n + 255) / 256;
    if (blocks > 64) blocks = 64;
    return launch(copy_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
}

// BF16 bits -> FP32 (exact: a BF16 value is the top half of its FP32), eight
// values per thread and step (a 16-byte load, two 16-byte stores) when both
// buffers are 16-byte aligned, then single values for the rest.
__global__ void bf16_to_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst, size_t n) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    const bool vec = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
    const size_t n8 = vec ? n / 8 : 0;
    for (size_t i = tid; i < n8; i += stride) {
        const uint4 v = reinterpret_cast<const uint4*>(src)[i];
        float4* o = reinterpret_cast<float4*>(dst) + 2 * i;
        o[0] = make_float4(__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xFFFF0000u), __uint_as_float(v.y << 16),
                           __uint_as_float(v.y & 0xFFFF0000u));
        o[1] = make_float4(__uint_as_float(v.z << 16), __uint_as_float(v.z & 0xFFFF0000u), __uint_as_float(v.w << 16),
                           __uint_as_float(v.w & 0xFFFF0000u));
    }
    for (size_t i = n8 * 8 + tid; i < n; i += stride) dst[i] = __uint_as_float((uint32_t)src[i] << 16);
}

hipError_t launch_bf16_to_f32(const uint16_t* src, float* dst, size_t n, hipStream_t s) {
    size_t blocks = (n / 8 + 255) / 256;
    if (blocks < 1) blocks = 1;
    if (blocks > 4096) blocks = 4096;
    return launch(bf16_to_f32_kernel, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
}

// The lo half of a BF16 value held as FP32 is zero, but for an infinity or NaN,
// whose difference from its own hi half is NaN.  So x goes to the multi-token
// GEMMs as it is, and two kernels stand for the widening to FP32 and its split:
// the first reads x (2 of the 14 bytes per value that those moved; 4096 x 6144
// 66 -> 14 us) and flags such values, the second writes the lo halves, only
// where there are any.
__device__ __forceinline__ bool bf16_special(uint32_t v) { return (v & 0x7F80u) == 0x7F80u; }

__global__ void bf16_specials_kernel(const uint16_t* __restrict__ x, size_t n, unsigned* __restrict__ flag) {
    const size_t tid = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    bool any = false;
    auto test = [&](uint32_t w) { any |= bf16_special(w) || bf16_special(w >> 16); };
    for (size_t i = tid; i < n / 8; i += stride) {
        const uint4 v = reinterpret_cast<const uint4*>(x)[i];
        test(v.x);
        test(v.y);
        test(v.z);
        test(v.w);
    }
    if (tid < n % 8) any |= bf16_special(x[n - 1 - tid]);
    if (__ballot(any) != 0ull && (threadIdx.x & 63) == 0) *flag = 1u;
}

__global__ void bf16_lo_kernel(const uint16_t* __restrict__ x, uint16_t* __restrict__ lo, size_t n,
                               const unsigned* __restrict__ flag) {
    if (*flag == 0u) return;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
        const float v = __uint_as_float((uint32_t)x[i] << 16);
        lo[i] = f32_to_bf16(v - __uint_as_float((uint32_t)f32_to_bf16(v) << 16));
    }
}

hipError_t launch_bf16_lo(const uint16_t* x, uint16_t* lo, size_t n, unsigned* flag, hipStream_t s) {
    if (reinterpret_cast<uintptr_t>(x) & 15) return hipErrorInvalidValue;
    const size_t blocks = std::min<size_t>((n / 8 + 255) / 256 + 1, 2048);
    hipError_t e = launch(bf16_specials_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, n, flag);
    if (e != hipSuccess) return e;
    return launch(bf16_lo_kernel, dim3((unsigned)blocks), dim3(256), 0, s, x, lo, n, flag);
}

__global__ void copy_u32_kernel(const uint32_t* __restrict__ src, uint32_t* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy_u32(const uint32_t* src, uint32_t* dst, size_t n, hipStream_t s) {
    size_t blocks = (n + 255) / 256;
    if (blocks > 64) blocks = 64;
    return launch(copy_u32_kernel, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
}

__global__ void copy_u64_kernel(const uint64_t* __restrict__ src, uint64_t* __restrict__ dst, size_t n) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

hipError_t launch_copy_u64(const uint64_t* src, uint64_t* dst, size_t n, hipStream_t s) {
    size_t blocks = (n + 255) / 256;
    if (blocks > 64) blocks = 64;
    return launch(copy_u64_kernel, dim3((unsigned)blocks), dim3(256), 0, s, src, dst, n);
}

hipError_t launch_rmsnorm(const float* h, const uint16_t* w, float* out, int T, int d, float eps,
                          hipStream_t s) {
    if (d > 8 * kNormThreads) return hipErrorInvalidValue;
    return launch(rmsnorm_kernel, dim3(T), dim3(kNormThreads), 0, s, h, w, out, d, eps);
}

hipError_t launch_rmsnorm_split(const float* h, const uint16_t* w, uint16_t* hi, uint16_t* lo, int T, int d, float eps,
                                unsigned* flag, hipStream_t s) {
    if (d > 8 * kNormThreads || d % 4) return hipErrorInvalidValue;
    return launch(rmsnorm_split_kernel, dim3(T), dim3(kNormThreads), 0, s, h, w, hi, lo, d, eps, flag);
}

hipError_t launch_add_inplace(float* dst, const float* src, size_t n, hipStream_t s) {
    size_t blocks = (n + 255) / 256;
    if (blocks > 4096) blocks = 4096;
    return launch(add_inplace_kernel, dim3((unsigned)blocks), dim3(256), 0, s, dst, src, n);
}

}  // namespace hf
