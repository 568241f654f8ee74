// gemm16.hip -- launchers of the 16-bit matrix-core products (gemm16.hpp) and
// the kernels that put weights into the pair format.
#include "gemm16.hpp"

#include <algorithm>

namespace ebh {

// ---------------------------------------------------------------------------
// Weight preparation
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void to_pair_kernel(const float* __restrict__ x, uint32_t* __restrict__ y,
                                                      int64_t n8, float scale) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const float4 a = *reinterpret_cast<const float4*>(x + 8 * i), b = *reinterpret_cast<const float4*>(x + 8 * i + 4);
    uint4 h, l;
    split_f16x2(a.x * scale, a.y * scale, h.x, l.x);
    split_f16x2(a.z * scale, a.w * scale, h.y, l.y);
    split_f16x2(b.x * scale, b.y * scale, h.z, l.z);
    split_f16x2(b.z * scale, b.w * scale, h.w, l.w);
    *reinterpret_cast<uint4*>(y + 8 * i) = h;
    *reinterpret_cast<uint4*>(y + 8 * i + 4) = l;
}

hipError_t launch_to_pair(const float* x, uint32_t* y, int64_t n, float scale, hipStream_t s) {
    if (n % 8 || ((uintptr_t)x & 15) || ((uintptr_t)y & 15)) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(to_pair_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, s, x, y, n / 8, scale);
    return hipGetLastError();
}

// One wave per row.  A NaN in a row shows in norm2 (amax alone would lose it:
// fmaxf drops NaN).
__global__ __launch_bounds__(256) void row_stats_kernel(const float* __restrict__ W, int N, int K,
                                                        float* __restrict__ norm2, float* __restrict__ amax) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (row >= N) return;
    float s = 0.0f, m = 0.0f;
    for (int k = lane; k < K; k += 64) {
        const float v = W[(int64_t)row * K + k];
        s += v * v;
        m = fmaxf(m, fabsf(v));
    }
    s = wave_sum(s);
    m = wave_max(m);
    if (lane == 0) {
        norm2[row] = s;
        amax[row] = m;
    }
}

hipError_t launch_row_stats(const float* W, int N, int K, float* norm2, float* amax, hipStream_t s) {
    if (N <= 0) return hipSuccess;
    hipLaunchKernelGGL(row_stats_kernel, dim3((N + 3) / 4), dim3(256), 0, s, W, N, K, norm2, amax);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Tile choice.  Each tile's time on a shape is estimated from its work items:
// with n items on the busiest CU, wpc of them resident at a time,
//   launch + sum over rounds of (k-tiles * kt[resident] + resident * epi),
// the constants (us) fitted to a sweep on MI355X of the four products of
// MiniLM and BERT-base at 96 .. 49,152 rows and 1 .. 8 splits (rms error of a
// fit 8-13%; the tile it picks takes 1.03 times the best one's time on
// average over that sweep).  What the numbers say: a 256-wide tile runs its
// k-loop fastest but pays a long epilogue (its C is all of a CU's stores), so
// it wins on many rounds or a long K; small tiles keep a small job on all CUs.
// Each split beyond the first costs the LayerNorm that follows a read of
// M * N floats (at 4 TB/s).
// ---------------------------------------------------------------------------
struct TileCost {
    int bm, bn, wpc;
    float launch, epi, epi_gelu, kt[4];
};
static const TileCost kPairTiles[GEMM16_TILES] = {
    {256, 256, 1, 0.0f, 11.0f, 2.37f, {1.653f}},
    {256, 192, 1, 0.0f, 9.78f, 1.70f, {1.312f}},
    {128, 128, 2, 0.96f, 3.27f, 0.17f, {0.703f, 1.144f}},
    {128, 96, 2, 1.16f, 2.27f, 0.16f, {0.692f, 1.044f}},
    {64, 128, 2, 2.45f, 1.33f, 0.33f, {0.430f, 0.713f}},
    {128, 64, 3, 1.84f, 1.53f, 1.11f, {0.455f, 0.692f, 1.079f}},
    {64, 64, 4, 2.19f, 0.64f, 0.14f, {0.374f, 0.535f, 0.703f, 0.860f}},
};

Gemm16Plan gemm16_pair_plan(int M, int N, int K, bool gelu, int min_splits, int max_splits) {
    Gemm16Plan best{0, 1};
    double best_us = 1e30;
    const int cus = device_cu_count();
    for (int i = 0; i < GEMM16_TILES; ++i) {
        const TileCost& t = kPairTiles[i];
        for (int S : {1, 2, 3, 4, 6, 8}) {
            if (S < min_splits || S > std::max(max_splits, 1) || K % (64 * S)) continue;
            const int64_t items = (int64_t)((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * S;
            const int64_t per = (items + cus - 1) / cus, full = per / t.wpc, rem = per % t.wpc;
            const double nk = K / 32.0 / S, e = t.epi + (gelu ? t.epi_gelu : 0.0f);
            double us = t.launch + full * (nk * t.kt[t.wpc - 1] + e * t.wpc) + (S - 1) * ((double)M * N * 4e-6 / 4.0);
            if (rem) us += nk * t.kt[rem - 1] + e * rem;
            if (us < best_us) {
                best_us = us;
                best = Gemm16Plan{i, S};
            }
        }
    }
    return best;
}

template <int BM, int BN, int WAVES_M, int WAVES_N, int NST>
static hipError_t launch_pair_tile(const Gemm16Args& a, int epi, bool out_pair, int wpc, hipStream_t s) {
    const int64_t items = (int64_t)((a.M_max + BM - 1) / BM) * ((a.N + BN - 1) / BN) * (a.splits > 1 ? a.splits : 1);
    if (items == 0) return hipSuccess;
    const dim3 grid((unsigned)std::min<int64_t>(items, (int64_t)device_cu_count() * wpc)), block(64 * WAVES_M * WAVES_N);
    if (epi == EPI_BIAS && out_pair)
        hipLaunchKernelGGL((gemm16_kernel<true, BM, BN, WAVES_M, WAVES_N, NST, EPI_BIAS, OUT_PAIR>), grid, block, 0, s, a);
    else if (epi == EPI_NONE && !out_pair)
        hipLaunchKernelGGL((gemm16_kernel<true, BM, BN, WAVES_M, WAVES_N, NST, EPI_NONE, OUT_F32>), grid, block, 0, s, a);
    else if (epi == EPI_BIAS_GELU && out_pair)
        hipLaunchKernelGGL((gemm16_kernel<true, BM, BN, WAVES_M, WAVES_N, NST, EPI_BIAS_GELU, OUT_PAIR>), grid, block, 0, s, a);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_gemm16_pair(const Gemm16Args& a, int epi, bool out_pair, int tile, hipStream_t s) {
    auto al16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    const int S = a.splits > 1 ? a.splits : 1;
    const bool ok = a.M_max >= 0 && a.N > 0 && a.K > 0 && a.N % 8 == 0 && a.K % (64 * S) == 0 && a.lda % 8 == 0 &&
                    a.ldw % 8 == 0 && a.ldc % 8 == 0 && a.lda >= a.K && a.ldw >= a.K && a.ldc >= a.N &&
                    al16(a.A) && al16(a.W) && al16(a.C) && (S == 1 || (epi == EPI_NONE && a.split_stride % 8 == 0)) &&
                    (epi == EPI_NONE || (a.bias && al16(a.bias))) && gemm_offsets_fit32(a.lda, a.ldw, 4) &&
                    a.ldc <= gemm_stride_max(4);
    if (!ok) return hipErrorInvalidValue;
    switch (tile) {
        case 0: return launch_pair_tile<256, 256, 2, 4, 2>(a, epi, out_pair, 1, s);
        case 1: return launch_pair_tile<256, 192, 4, 2, 2>(a, epi, out_pair, 1, s);
        case 2: return launch_pair_tile<128, 128, 2, 2, 2>(a, epi, out_pair, 2, s);
        case 3: return launch_pair_tile<128, 96, 4, 1, 2>(a, epi, out_pair, 2, s);
        case 4: return launch_pair_tile<64, 128, 2, 2, 3>(a, epi, out_pair, 2, s);
        case 5: return launch_pair_tile<128, 64, 2, 2, 2>(a, epi, out_pair, 3, s);
        case 6: return launch_pair_tile<64, 64, 2, 2, 2>(a, epi, out_pair, 4, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ebh
