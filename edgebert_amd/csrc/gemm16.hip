// gemm16.hip -- launchers of the 16-bit matrix-core products (gemm16.hpp) and
// the kernels that put weights into the pair format.
#include "gemm16.hpp"

#include <algorithm>
#include <cmath>

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
// MiniLM and BERT-base at 96 .. 49,152 rows (bf16: .. 131,072) and 1 .. 8
// splits (rms error of a fit 6-14%; the tile picked takes 1.025 times the best
// one's time on average over that sweep).  What the numbers say: a 256-wide
// tile runs its k-loop fastest but pays a long epilogue (its C is all of a CU's
// stores), so it wins on many rounds or a long K; small tiles keep a small
// job on all CUs.  Each split beyond the first costs the LayerNorm that
// follows a read of M * N floats (at 4 TB/s).
//
// Device-buffer calls know only the padded rows, of which a ragged batch fills
// a part: there the estimate is summed over fills from half to all (all counts
// twice).  Over the sweep that choice takes 1.08 times the best tile's time on
// ragged batches and 1.06 on full ones, against 1.13 and 1.025 for one that
// takes every batch as full.
// ---------------------------------------------------------------------------
struct TileCost {
    int bm, bn, wpc;
    float launch, epi, epi_gelu, kt[4];
};
static const TileCost kPairTiles[GEMM16_TILES] = {
    {256, 256, 1, 0.0f, 10.41f, 1.69f, {1.673f}},
    {256, 192, 1, 0.0f, 9.06f, 1.40f, {1.330f}},
    {128, 128, 2, 2.08f, 2.35f, 0.07f, {0.719f, 1.141f}},
    {128, 96, 2, 1.85f, 1.80f, 0.30f, {0.693f, 1.001f}},
    {64, 128, 2, 2.98f, 1.00f, 0.44f, {0.429f, 0.709f}},
    {128, 64, 3, 2.45f, 0.99f, 1.22f, {0.467f, 0.705f, 1.095f}},
    {64, 64, 4, 2.48f, 0.50f, 0.18f, {0.374f, 0.536f, 0.684f, 0.840f}},
};
// bf16; the first is gemm_bf16_ring_kernel (gemm.hip).
constexpr int BF16_TILES = 6;
static const TileCost kBf16Tiles[BF16_TILES] = {
    {256, 256, 1, 0.0f, 4.98f, 2.84f, {1.268f}},
    {256, 192, 1, 0.0f, 4.94f, 1.50f, {1.050f}},
    {128, 128, 2, 2.51f, 0.40f, 0.60f, {0.604f, 0.972f}},
    {128, 96, 2, 2.46f, 0.40f, 0.55f, {0.563f, 0.829f}},
    {64, 128, 2, 2.94f, 0.20f, 0.44f, {0.396f, 0.600f}},
    {64, 64, 2, 2.81f, 0.25f, 0.19f, {0.284f, 0.399f}},
};

static double tile_us(const TileCost& t, double M, int N, int nk, bool gelu, int S) {
    const int cus = device_cu_count();
    const int64_t rows = std::max<int64_t>(1, (int64_t)std::ceil(M / t.bm));
    const int64_t items = rows * ((N + t.bn - 1) / t.bn) * S, per = (items + cus - 1) / cus;
    const int64_t full = per / t.wpc, rem = per % t.wpc;
    const double k = (double)nk / S, e = t.epi + (gelu ? t.epi_gelu : 0.0f);
    double us = t.launch + full * (k * t.kt[t.wpc - 1] + e * t.wpc) + (S - 1) * (M * N * 4e-6 / 4.0);
    if (rem) us += k * t.kt[rem - 1] + e * rem;
    return us;
}

// The estimate at M rows, or summed over the fills of M that a device-buffer
// call may meet.
template <class F>
static double over_fills(int M, bool exact, F&& us_at) {
    if (exact) return us_at((double)M);
    double us = 0.0;
    for (double fill : {0.5, 0.6, 0.7, 0.8, 0.9, 1.0, 1.0}) us += us_at(fill * M);
    return us;
}

static double tile_us_of(const TileCost& t, int M, bool exact, int N, int nk, bool gelu, int S) {
    return over_fills(M, exact, [&](double m) { return tile_us(t, m, N, nk, gelu, S); });
}

Gemm16Plan gemm16_pair_plan(int M, bool exact, int N, int K, bool gelu, int min_splits, int max_splits, double* us_out) {
    Gemm16Plan best{0, 1};
    double best_us = 1e30;
    for (int i = 0; i < GEMM16_TILES; ++i)
        for (int S : {1, 2, 3, 4, 6, 8}) {
            if (S < min_splits || S > std::max(max_splits, 1) || K % (64 * S)) continue;
            const double us = tile_us_of(kPairTiles[i], M, exact, N, K / 32, gelu, S);
            if (us < best_us) {
                best_us = us;
                best = Gemm16Plan{i, S};
            }
        }
    if (us_out) *us_out = best_us;
    return best;
}

// ffn_pair_kernel: rounds of one workgroup per CU; a chunk of 128 intermediate
// columns takes 12.6 us with up to half of the CUs at work and 16.6 us with all
// (measured at 256 .. 40,000 rows, 1 .. 12 splits; a product kernel per step takes
// as long or longer where these rounds are filled, e.g. 14,355 rows: 105 us in 2
// splits against 108).  The estimate is weighed at 0.9: the two products' own
// takes the best tile for granted, which a call that knows only the padded
// rows often misses (the same rows of 24,750 padded ones, in a forward: 138 us).
static double ffn_us(double M, int I, int S) {
    const int cus = device_cu_count();
    const int64_t items = std::max<int64_t>(1, (int64_t)std::ceil(M / 128)) * S;
    const double chunks = (double)(I / 128) / S;
    auto round = [&](int64_t n) {
        return 3.0 + chunks * 12.6 * (1.0 + 0.64 * std::max(0.0, (double)n / cus - 0.5));
    };
    double us = (double)(items / cus) * round(cus) + (S - 1) * (M * 384 * 4e-6 / 4.0);
    if (items % cus) us += round(items % cus);
    return us;
}

FfnPairPlan ffn_pair_plan(int M, bool exact, int H, int I, int min_splits, int max_splits) {
    FfnPairPlan best{};
    double up_us = 0.0, best_us = 1e30;
    best.up = gemm16_pair_plan(M, exact, I, H, true, 1, 1, &up_us);
    best.down = gemm16_pair_plan(M, exact, H, I, false, min_splits, max_splits, &best_us);
    best_us += up_us;
    best.fused = false;
    best.splits = best.down.splits;
    if (!ffn_pair_shape_ok(H, I)) return best;
    for (int S : {1, 2, 3, 4, 6}) {
        if (S < min_splits || S > std::max(max_splits, 1) || (I / 128) % S) continue;
        const double us = 0.9 * over_fills(M, exact, [&](double m) { return ffn_us(m, I, S); });
        if (us < best_us) {
            best_us = us;
            best.fused = true;
            best.splits = S;
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

template <int BM, int BN, int WAVES_M, int WAVES_N, int NST>
static hipError_t launch_bf16_tile(const Gemm16Args& a, int epi, int wpc, hipStream_t s) {
    const int64_t items = (int64_t)((a.M_max + BM - 1) / BM) * ((a.N + BN - 1) / BN);
    const dim3 grid((unsigned)std::min<int64_t>(items, (int64_t)device_cu_count() * wpc)), block(64 * WAVES_M * WAVES_N);
    switch (epi) {
        case EPI_BIAS:
            hipLaunchKernelGGL((gemm16_kernel<false, BM, BN, WAVES_M, WAVES_N, NST, EPI_BIAS, OUT_BF16>), grid, block, 0, s, a);
            break;
        case EPI_BIAS_GELU:
            hipLaunchKernelGGL((gemm16_kernel<false, BM, BN, WAVES_M, WAVES_N, NST, EPI_BIAS_GELU, OUT_BF16>), grid, block, 0, s, a);
            break;
        case EPI_NONE:
            hipLaunchKernelGGL((gemm16_kernel<false, BM, BN, WAVES_M, WAVES_N, NST, EPI_NONE, OUT_BF16>), grid, block, 0, s, a);
            break;
        default:
            return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

bool launch_gemm16_bf16(const GemmArgs& g, int epi, hipStream_t s, hipError_t* err) {
    if (g.M_max <= 0 || g.K % 128 || g.lda < g.K || g.ldw < g.K || g.ldc < g.N || g.ldc > gemm_stride_max(4)) return false;
    int best = 0;
    double best_us = 1e30;
    for (int i = 0; i < BF16_TILES; ++i) {
        const double us = tile_us_of(kBf16Tiles[i], g.M_max, g.M_dev == nullptr, g.N, g.K / 64, epi == EPI_BIAS_GELU, 1);
        if (us < best_us) {
            best_us = us;
            best = i;
        }
    }
    Gemm16Args a{};
    a.A = g.A;
    a.W = g.W;
    a.bias = g.bias;
    a.C = g.C;
    a.lda = g.lda;
    a.ldw = g.ldw;
    a.ldc = g.ldc;
    a.M_max = g.M_max;
    a.M_dev = g.M_dev;
    a.N = g.N;
    a.K = g.K;
    a.splits = 1;
    switch (best) {
        case 1: *err = launch_bf16_tile<256, 192, 4, 2, 2>(a, epi, 1, s); return true;
        case 2: *err = launch_bf16_tile<128, 128, 2, 2, 2>(a, epi, 2, s); return true;
        case 3: *err = launch_bf16_tile<128, 96, 4, 1, 2>(a, epi, 2, s); return true;
        case 4: *err = launch_bf16_tile<64, 128, 2, 2, 3>(a, epi, 2, s); return true;
        case 5: *err = launch_bf16_tile<64, 64, 2, 2, 4>(a, epi, 2, s); return true;
        default: return false;   // the ring kernel
    }
}

}  // namespace ebh
