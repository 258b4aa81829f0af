// lm_head.hip -- final RMSNorm, LM-head logits and greedy argmax
// (GLMForward::lmHeadAndSample, glm_forward.cpp:663-731).
//
// logits[v] = lm_head[v, :] . RMSNorm(h) over the whole vocabulary (154880 x
// 6144 BF16 = 1.9 GB at GLM-5.2: a bandwidth-bound GEMV), then the first
// index of the largest logit (the reference's serial scan keeps the first
// maximum; its OpenMP merge of per-thread winners is the same unless two
// threads hold exactly equal maxima).
//
// T = 1: a persistent GEMV.  Each block normalises the hidden state into LDS; each wavefront streams whole vocabulary rows, two at a time, 16-byte
//   non-temporal loads (lane l: elements 512j + 8l .. +7; the weights are read
//   once and kept out of the caches' way); lane 0 writes the logit and
//   keeps the wavefront's running winner, the block merges its four, and one
//   small launch merges the blocks' winners (lowest row on equal values).
// T > 1: a GEMM (one group, fixed B = lm_head) writes the logits, then one
//   block per token finds its argmax.
#include "hf_api_internal.h"
#include "hf_grouped.h"
#include "hf_norm.h"

#include <climits>

namespace hf {

struct ArgMax {
    float v;
    int i;
};

__device__ __forceinline__ bool better(float va, int ia, float vb, int ib) {
    return va > vb || (va == vb && ia < ib);
}

constexpr int kLmBlock = 256;

// NORM: x is the hidden state, and each block normalises it on the way into
// LDS (stage_rmsnorm: rmsnorm_kernel's bits): 36 KB from L2 beside the table's 3.7 MB a block, for a launch
// less (vocab 154880 x 6144 294 -> 288 us, 32000 x 2048 27 -> 24).
template <int KCH, int RF, bool NORM>
__global__ __launch_bounds__(kLmBlock) void lm_gemv_kernel(const uint16_t* __restrict__ W,
                                                           const float* __restrict__ x, int V, int K,
                                                           const uint16_t* __restrict__ norm, float eps,
                                                           float* __restrict__ logits,
                                                           ArgMax* __restrict__ part) {
    // x in LDS, chunk ch = x[8 ch .. 8 ch + 8) split into halves xs[0][ch],
    // xs[1][ch] so that a wavefront's 16-byte reads are consecutive: at 32-byte
    // strides they met in half the banks, and every row pair waited for its
    // reads (vocab 154880 x 6144 291 -> 283 us, 32000 x 2048 23.2 -> 20).
    __shared__ float4 xs[2][KCH * 64];
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int nwaves = gridDim.x * (kLmBlock / 64);
    const int gw = blockIdx.x * (kLmBlock / 64) + wave;
    if constexpr (NORM) {
        __shared__ float red[kNormThreads / 64];
        static_assert(kLmBlock == kRowNormThreads, "block");
        stage_rmsnorm<KCH>(x, norm, eps, K, xs[0], xs[1], red);
    } else {
        for (int i = threadIdx.x; i < KCH * 512; i += kLmBlock)  // (x may start on any 4-byte boundary)
            reinterpret_cast<float*>(xs[(i >> 2) & 1])[(i >> 3) * 4 + (i & 3)] = i < K ? x[i] : 0.0f;
    }
    __syncthreads();
    float best = -INFINITY;
    int best_i = INT_MAX;
    for (int r0 = gw * RF; r0 < V; r0 += nwaves * RF) {
        u32x4 w[RF][KCH];
#pragma unroll
        for (int u = 0; u < RF; ++u) {
            const int r = min(r0 + u, V - 1);
            const uint16_t* row = W + (size_t)r * K;
#pragma unroll
            for (int j = 0; j < KCH; ++j) {
                const int k0 = j * 512 + lane * 8;
                w[u][j] = k0 < K ? ld_stream(reinterpret_cast<const u32x4*>(row + k0)) : (u32x4){0, 0, 0, 0};
            }
        }
        float acc[RF];
#pragma unroll
        for (int u = 0; u < RF; ++u) acc[u] = 0.0f;
        // Re-read x from LDS for every row pair: an opaque offset keeps the
        // compiler from hoisting the reads (and 96 registers) out of the loop.
        int xo = lane;
        asm volatile("" : "+v"(xo));
#pragma unroll
        for (int j = 0; j < KCH; ++j) {
            const float4 xa = xs[0][j * 64 + xo], xb = xs[1][j * 64 + xo];
            const float xv[8] = {xa.x, xa.y, xa.z, xa.w, xb.x, xb.y, xb.z, xb.w};
#pragma unroll
            for (int u = 0; u < RF; ++u) {
                const u32x4 v = w[u][j];
                const uint32_t ws[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    acc[u] = fmaf(__uint_as_float(ws[q] << 16), xv[2 * q], acc[u]);
                    acc[u] = fmaf(__uint_as_float(ws[q] & 0xFFFF0000u), xv[2 * q + 1], acc[u]);
                }
            }
        }
#pragma unroll
        for (int u = 0; u < RF; ++u) {
            const float dot = wave_sum(acc[u]);
            const int r = r0 + u;
            if (r < V) {
                if (lane == 0) logits[r] = dot;
                if (better(dot, r, best, best_i)) {
                    best = dot;
                    best_i = r;
                }
            }
        }
    }
    if (!part) return;  // plain matvec: no winner wanted
    __shared__ ArgMax wbest[kLmBlock / 64];
    if (lane == 0) wbest[wave] = {best, best_i};
    __syncthreads();
    if (threadIdx.x == 0) {
        ArgMax b = wbest[0];
        for (int i = 1; i < kLmBlock / 64; ++i)
            if (better(wbest[i].v, wbest[i].i, b.v, b.i)) b = wbest[i];
        part[blockIdx.x] = b;
    }
}

// Winner of n partial winners (one block).
__global__ __launch_bounds__(256) void argmax_merge_kernel(const ArgMax* __restrict__ part, int n,
                                                           int* __restrict__ out) {
    __shared__ ArgMax s[256];
    ArgMax b{-INFINITY, INT_MAX};
    for (int i = threadIdx.x; i < n; i += 256)
        if (better(part[i].v, part[i].i, b.v, b.i)) b = part[i];
    s[threadIdx.x] = b;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w && better(s[threadIdx.x + w].v, s[threadIdx.x + w].i, s[threadIdx.x].v,
                                          s[threadIdx.x].i))
            s[threadIdx.x] = s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = s[0].i == INT_MAX ? 0 : s[0].i;
}

// One block per row of a [T, V] matrix: first index of the row's maximum.
// A row is one block's to read (620 KB at the GLM vocabulary), so what bounds
// it is how many loads that block keeps in flight: 1024 threads, each with
// four 16-byte loads out before it compares the first (a row that does not
// start on a 16-byte boundary: single loads up to the first one).  24 rows of
// 154880: 188 us with 256 threads and one 4-byte load each, 15 us now.
constexpr int kArgmaxThreads = 1024;
__global__ __launch_bounds__(kArgmaxThreads) void row_argmax_kernel(const float* __restrict__ logits, int V,
                                                                    int* __restrict__ out,
                                                                    unsigned* __restrict__ clear) {
    if (clear && blockIdx.x == 0 && threadIdx.x == 0) *clear = 0u;
    constexpr int U = 4;
    __shared__ ArgMax s[kArgmaxThreads / 64];
    const int t = threadIdx.x;
    const float* row = logits + (size_t)blockIdx.x * V;
    const int lead = min(V, (int)(((16 - (reinterpret_cast<uintptr_t>(row) & 15)) & 15) / 4));
    const int n4 = (V - lead) / 4;
    const float4* r4 = reinterpret_cast<const float4*>(row + lead);
    ArgMax b{-INFINITY, INT_MAX};
    auto take = [&](float v, int i) {
        if (better(v, i, b.v, b.i)) b = {v, i};
    };
    if (t < lead) take(row[t], t);
    for (int i = t; i < n4; i += U * kArgmaxThreads) {
        float4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = i + u * kArgmaxThreads;
            v[u] = r4[j < n4 ? j : i];  // past the end: element i again, which changes no winner
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = i + u * kArgmaxThreads;
            const int k = lead + 4 * (j < n4 ? j : i);
            take(v[u].x, k);
            take(v[u].y, k + 1);
            take(v[u].z, k + 2);
            take(v[u].w, k + 3);
        }
    }
    for (int i = lead + 4 * n4 + t; i < V; i += kArgmaxThreads) take(row[i], i);
    wave_argmax(b.v, b.i);
    if ((t & 63) == 0) s[t >> 6] = b;
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < kArgmaxThreads / 64; ++w)
            if (better(s[w].v, s[w].i, b.v, b.i)) b = s[w];
        out[blockIdx.x] = b.i == INT_MAX ? 0 : b.i;
    }
}

template <int KCH>
static hipError_t lm_gemv_inst(const uint16_t* W, const float* x, int V, int K, const RowNorm* norm, float* logits,
                               ArgMax* part, int grid, hipStream_t s) {
    constexpr int RF = KCH <= 12 ? 2 : 1;
    if (norm)
        return launch(lm_gemv_kernel<KCH, RF, true>, dim3(grid), dim3(kLmBlock), 0, s, W, x, V, K, norm->w, norm->eps,
                      logits, part);
    return launch(lm_gemv_kernel<KCH, RF, false>, dim3(grid), dim3(kLmBlock), 0, s, W, x, V, K, nullptr, 0.0f, logits,
                  part);
}

hipError_t launch_row_argmax(const float* x, int T, int n, int* out, unsigned* clear, hipStream_t s) {
    return launch(row_argmax_kernel, dim3(T), dim3(kArgmaxThreads), 0, s, x, n, out, clear);
}

static hipError_t launch_lm_gemv(const uint16_t* W, const float* x, int V, int K, const RowNorm* norm, float* logits,
                                 ArgMax* part, int grid, hipStream_t s) {
    const int kch = (K + 511) / 512;
    if (kch <= 4) return lm_gemv_inst<4>(W, x, V, K, norm, logits, part, grid, s);
    if (kch <= 8) return lm_gemv_inst<8>(W, x, V, K, norm, logits, part, grid, s);
    if (kch <= 12) return lm_gemv_inst<12>(W, x, V, K, norm, logits, part, grid, s);
    if (kch <= 16) return lm_gemv_inst<16>(W, x, V, K, norm, logits, part, grid, s);
    return hipErrorInvalidValue;
}

// Two 4-wave blocks per CU (two rows of loads in flight per wavefront take
// ~176 registers at hidden 6144; more rows or blocks measured no faster).
// y[M] = W[M, K] . x[K] (K a multiple of 8, at most 8192), no argmax.
hipError_t launch_matvec_bf16(const uint16_t* W, const float* x, int M, int K, float* y, hipStream_t s) {
    return launch_lm_gemv(W, x, M, K, nullptr, y, nullptr, g.num_cus * 2, s);
}

static int lm_grid() { return env_int("HFMOE_LM_BLOCKS", g.num_cus * 2); }
// Workgroups of a T = 1 call: HFMOE_LM_BLOCKS as read now, within the
// per-workgroup winners allocated at registration.
static int lm_call_grid() { return std::max(1, std::min(lm_grid(), g.lm.part_n)); }

void lm_head_release() {
    if (g.lm.part) hipFree(g.lm.part);
    g.lm = LmHead{};
}

#define HF_CHECK_LAUNCH(expr, what)                      \
    do {                                                 \
        hipError_t e_ = (expr);                          \
        prof_end(p, s);                                  \
        if (e_ != hipSuccess) return fail_hip(e_, what); \
    } while (0)

// The one-group tiles for T tokens, of 4 or 5 column blocks (cb), whichever the
// estimate says (at the GLM vocabulary 242 tiles of 640 rows are one round of
// 256 CUs, 303 of 512 two); cb = 0: the 128-row kernel, for a table or batch
// too small for them.  Up to 16 tokens its first wavefront alone, with one
// 16-row block, keeps up with the table's stream, on two workgroups per CU
// (154880 x 6144: T = 2 310 against 326 us, 8 326 against 331, 16 339 against
// 335-350, 24 377 against 335, 64 490 against 361, 128 690 against 430; T =
// 300 1673 on 256-row tiles against 1114).
constexpr int kLmFixedTokens = 17;
static FixedPlan lm_plan(int T, int d, int vocab, int& cb) {
    FixedPlan best;
    cb = 0;
    if (T < kLmFixedTokens || !fixed_worth(T, (size_t)vocab * d)) return best;
    // K-split partials go to the MoE path's y rows (the split sum adds four
    // logits at a time).
    const size_t one = (size_t)T * vocab, y_floats = (size_t)g.max_tokens * (g.cfg.k + g.cfg.n_shared) * g.cfg.d;
    const int splits = one % 4 ? 1 : (int)std::max((size_t)1, std::min((size_t)kFixedMaxSplits, y_floats / one));
    for (int c = 4; c <= 5; ++c) {
        if (vocab < fixed_tile_cols(c, false) || (c == 5 && T > fixed_tile_rows(5))) continue;
        const FixedPlan pl = plan_fixed_gemm(T, vocab, false, c, d / kGemmTileK, splits, g.num_cus);
        if (!cb || pl.us < best.us) {
            best = pl;
            cb = c;
        }
    }
    // A short table without room for the splits that fill the chip.
    if (T <= kGemmTileRows && 2 * best.m_tiles * best.n_tiles * best.ksplit < g.num_cus) cb = 0;
    return best;
}

static int lm_head_forward(const float* h, int T, float* logits, int* token, hipStream_t s) {
    const Cfg& c = g.cfg;
    const LmHead& L = g.lm;
    Pending p;
    const bool gemm = T > 1 && g.gws.xh && c.d % kGemmTileK == 0;
    if (!gemm) {
        const RowNorm norm{L.norm, c.eps};
        const int grid = lm_call_grid();
        for (int t = 0; t < T; ++t) {
            prof_begin(p, "lm_head_gemv", s);
            HF_CHECK_LAUNCH(launch_lm_gemv(L.w, h + (size_t)t * c.d, L.vocab, c.d, &norm, logits + (size_t)t * L.vocab,
                                           static_cast<ArgMax*>(L.part), grid, s),
                            "lm head gemv");
            if (token) {
                prof_begin(p, "lm_argmax", s);
                HF_CHECK_LAUNCH(launch(argmax_merge_kernel, dim3(1), dim3(256), 0, s,
                                       static_cast<const ArgMax*>(L.part), grid, token + t),
                                "argmax");
            }
        }
        return HFMOE_OK;
    }
    // The norm writes the halves the GEMM reads; the argmax, which follows it,
    // clears their flag.
    GroupedWorkspace& gw = g.gws;
    const int rc = lo_flag_begin(gw.one_lo_flag(), gw.one_dirty, s);
    if (rc) return rc;
    prof_begin(p, "lm_norm", s);
    HF_CHECK_LAUNCH(launch_rmsnorm_split(h, L.norm, gw.xh, gw.xl, T, c.d, c.eps, gw.one_lo_flag(), s), "final norm");
    GemmArgs a{};
    a.K = c.d;
    a.N = L.vocab;
    a.rows_total = T;
    a.a_hi = gw.xh;
    a.a_lo = gw.xl;
    a.a_lo_flag = gw.one_lo_flag();
    a.b_fixed0 = L.w;
    a.b_ld = c.d;
    a.out_f32 = logits;
    a.ksplit = 1;
    int cb = 0;
    const FixedPlan pl = lm_plan(T, c.d, L.vocab, cb);
    if (cb) {
        a.tile_rows = pl.tile_rows;
        a.m_tiles = pl.m_tiles;
        a.n_tiles = pl.n_tiles;
        a.ksplit = pl.ksplit;
        if (pl.ksplit > 1) a.out_f32 = gw.y;
        prof_begin(p, "lm_head_gemm", s);
        HF_CHECK_LAUNCH(launch_fixed_gemm(EPI_PARTIAL, false, cb, a, gemm_blocks(kPrefillTileRows), s), "lm head gemm");
        if (pl.ksplit > 1) {
            prof_begin(p, "lm_head_sum", s);
            HF_CHECK_LAUNCH(launch_sum_splits(gw.y, pl.ksplit, (size_t)T * L.vocab, logits, s), "lm head split sum");
        }
    } else {
        // Past one 128-row M tile (a table shorter than one 512-row tile), the
        // 256-row tiles (HFMOE_LM_MIN_TOKENS).
        const int TR = T >= env_int("HFMOE_LM_MIN_TOKENS", kGemmTileRows + 1) ? kDenseTileRows : kGemmTileRows;
        a.tile_rows = TR;
        a.tile_cols = gemm_tile_cols(TR, EPI_PARTIAL);
        a.n_tiles = gemm_n_tiles(EPI_PARTIAL, L.vocab, a.tile_cols);
        a.m_tiles = (T + TR - 1) / TR;
        prof_begin(p, "lm_head_gemm", s);
        HF_CHECK_LAUNCH(launch_grouped_gemm(EPI_PARTIAL, a, gemm_blocks(TR), s), "lm head gemm");
    }
    if (token) {
        prof_begin(p, "lm_argmax", s);
        HF_CHECK_LAUNCH(launch_row_argmax(logits, T, L.vocab, token, gw.one_lo_flag(), s), "argmax");
    } else {
        HF_CHECK_LAUNCH(launch_clear_u32(gw.one_lo_flag(), 1, s), "flag clear");
    }
    gw.one_dirty = false;
    return HFMOE_OK;
}

}  // namespace hf

using namespace hf;

extern "C" {

int hfmoe_register_lm_head(const uint16_t* lm_head_dev, const uint16_t* final_norm_dev, int32_t vocab) {
    int rc = require_cfg();
    if (rc) return rc;
    if (!lm_head_dev || vocab <= 0) return fail(HFMOE_ERR_INVALID_ARGUMENT, "lm head weights and vocab > 0 required");
    if ((reinterpret_cast<uintptr_t>(lm_head_dev) & 15) || g.cfg.d % 8)
        return fail(HFMOE_ERR_INVALID_ARGUMENT, "lm head must be 16-byte aligned with hidden a multiple of 8");
    if (g.cfg.d > 8192) return fail(HFMOE_ERR_UNSUPPORTED, "hidden %d > 8192", g.cfg.d);
    lm_head_release();
    const int part_n = std::max(1, lm_grid());
    hipError_t e = hipMalloc(&g.lm.part, sizeof(ArgMax) * (size_t)part_n);
    if (e != hipSuccess) return fail_hip(e, "lm head workspace");
    g.lm.part_n = part_n;
    g.lm.w = lm_head_dev;
    g.lm.norm = final_norm_dev;
    g.lm.vocab = vocab;
    return HFMOE_OK;
}

int hfmoe_lm_head(const float* h_dev, int32_t T, float* logits_dev, int32_t* token_dev, void* stream) {
    int rc = require_cfg();
    if (rc) return rc;
    if (!g.lm.w) return fail(HFMOE_ERR_NOT_REGISTERED, "no lm head registered");
    if (T < 0 || T > g.max_tokens)
        return fail(HFMOE_ERR_INVALID_ARGUMENT, "T=%d outside 0..max_tokens=%d", T, g.max_tokens);
    if (T == 0) return HFMOE_OK;
    if (!h_dev || !logits_dev) return fail(HFMOE_ERR_INVALID_ARGUMENT, "null hidden state or logits pointer");
    if ((reinterpret_cast<uintptr_t>(h_dev) | reinterpret_cast<uintptr_t>(logits_dev)) & 15)
        return fail(HFMOE_ERR_INVALID_ARGUMENT, "buffers must be 16-byte aligned");
    return lm_head_forward(h_dev, T, logits_dev, token_dev, pick_stream(stream));
}

}  // extern "C"
