// gemm16.hip -- launchers of the 16-bit matrix-core products (gemm16.hpp) and
// the kernels that put weights into the pair format.
#include "gemm16.hpp"

#include <algorithm>

namespace ebh {

// ---------------------------------------------------------------------------
// Weight preparation
// ---------------------------------------------------------------------------
// scale * x - h - l of two values: differences of fp32 numbers that are exact.
__device__ __forceinline__ uint32_t rest_f16x2(float a, float b, uint32_t h, uint32_t l) {
    typedef _Float16 v2h __attribute__((ext_vector_type(2)));
    const v2h hh = __builtin_bit_cast(v2h, h), ll = __builtin_bit_cast(v2h, l);
    const v2h r = {(_Float16)((a - (float)hh[0]) - (float)ll[0]), (_Float16)((b - (float)hh[1]) - (float)ll[1])};
    return __builtin_bit_cast(uint32_t, r);
}

// K8 > 0: rows of K8 groups of 8, each row's rest behind its pairs.
__global__ __launch_bounds__(256) void to_pair_kernel(const float* __restrict__ x, uint32_t* __restrict__ y,
                                                      int64_t n8, int K8, float scale) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (i >= n8) return;
    const float4 a = *reinterpret_cast<const float4*>(x + 8 * i), b = *reinterpret_cast<const float4*>(x + 8 * i + 4);
    uint4 h, l;
    split_f16x2(a.x * scale, a.y * scale, h.x, l.x);
    split_f16x2(a.z * scale, a.w * scale, h.y, l.y);
    split_f16x2(b.x * scale, b.y * scale, h.z, l.z);
    split_f16x2(b.z * scale, b.w * scale, h.w, l.w);
    const int64_t row = K8 > 0 ? i / K8 : 0;
    uint32_t* const at = y + row * 4 * K8 + 8 * i;        // 12 K8 words a row
    *reinterpret_cast<uint4*>(at) = h;
    *reinterpret_cast<uint4*>(at + 4) = l;
    if (K8 > 0)
        *reinterpret_cast<uint4*>(y + row * 12 * K8 + 8 * K8 + 4 * (i - row * K8)) =
            make_uint4(rest_f16x2(a.x * scale, a.y * scale, h.x, l.x), rest_f16x2(a.z * scale, a.w * scale, h.y, l.y),
                       rest_f16x2(b.x * scale, b.y * scale, h.z, l.z), rest_f16x2(b.z * scale, b.w * scale, h.w, l.w));
}

hipError_t launch_to_pair(const float* x, uint32_t* y, int64_t n, float scale, hipStream_t s) {
    if (n % 8 || ((uintptr_t)x & 15) || ((uintptr_t)y & 15)) return hipErrorInvalidValue;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(to_pair_kernel, dim3((unsigned)((n / 8 + 255) / 256)), dim3(256), 0, s, x, y, n / 8, 0, scale);
    return hipGetLastError();
}

hipError_t launch_to_pair_rest(const float* x, uint32_t* y, int64_t N, int K, float scale, hipStream_t s) {
    if (N < 0 || K <= 0 || K % 8 || ((uintptr_t)x & 15) || ((uintptr_t)y & 15)) return hipErrorInvalidValue;
    const int64_t n8 = N * (K / 8);
    if (n8 == 0) return hipSuccess;
    hipLaunchKernelGGL(to_pair_kernel, dim3((unsigned)((n8 + 255) / 256)), dim3(256), 0, s, x, y, n8, K / 8, scale);
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
// Family and tile choice: the cost model of gemm16.hpp with constants fitted to
// a sweep on MI355X of the four products of MiniLM and BERT-base at 96 ..
// 40,000 rows (bf16: .. 131,072) and 1 .. 6 splits (rms error of a fit 5-10%;
// least where operands come from a cache: MiniLM's two FFN products at 32,768
// rows take 205 us, 172 by the tables).
// What the numbers say: a 256-wide tile runs its k-loop fastest but pays a long
// epilogue (its C is all of a CU's stores), so it wins on many rounds or a long
// K; small tiles, two workgroups per CU, keep a small job on all CUs.  Each split
// beyond the first costs the LayerNorm that follows a read of M * N floats
// (at 4 TB/s).  A k-tile of the rest, two thirds of a pair k-tile's MFMAs on as
// many loads, takes 0.70 of one on the largest tile and as much as one on the
// smallest (the same products at 1,061 .. 32,768 rows).
//
// Device-buffer calls know only the padded rows, of which a ragged batch fills
// a part: the family is the one that is best over fills from half to all (all
// counts twice), and the kernel picks the tile by the rows it finds.  Over the
// sweep that takes 1.03 times the best tile's time on ragged batches and 1.025
// on full ones; a tile picked by the host in the same way took 1.09 and 1.02
// (3,456 of 6,144 rows of BERT-base: QKV 57, FFN up 58 and FFN down 71 us, on
// the best tiles 36, 46 and 47).
// ---------------------------------------------------------------------------
constexpr int FAMILIES = 2;
static const TileFamily kPairFamilies[FAMILIES] = {
    {{{256, 256, 1, 0.0f, 11.02f, 2.07f, {1.714f}, 0.70f},
      {256, 192, 1, 0.0f, 10.15f, 1.64f, {1.274f}, 0.78f},
      {256, 128, 1, 0.0f, 7.44f, 1.01f, {1.002f}, 0.86f},
      {128, 128, 1, 1.39f, 3.54f, 0.68f, {0.677f}, 0.92f}}},
    {{{128, 128, 2, 2.21f, 2.96f, 0.29f, {0.636f, 1.152f}, 0.95f},
      {128, 96, 2, 2.30f, 2.12f, 0.38f, {0.556f, 0.968f}, 0.95f},
      {64, 128, 2, 2.61f, 1.35f, 0.38f, {0.465f, 0.739f}, 0.93f},
      {64, 64, 2, 2.83f, 0.66f, 0.31f, {0.326f, 0.489f}, 1.10f}}},
};
static const TileFamily kBf16Families[FAMILIES] = {
    {{{256, 256, 1, 0.0f, 6.71f, 2.50f, {1.127f}},
      {256, 192, 1, 0.0f, 5.30f, 1.54f, {1.059f}},
      {256, 128, 1, 0.63f, 3.91f, 1.14f, {0.799f}},
      {128, 128, 1, 2.26f, 1.51f, 0.80f, {0.580f}}}},
    {{{128, 128, 2, 2.58f, 1.08f, 0.55f, {0.548f, 0.897f}},
      {128, 96, 2, 2.49f, 0.72f, 0.50f, {0.489f, 0.759f}},
      {64, 128, 2, 2.70f, 0.51f, 0.39f, {0.411f, 0.621f}},
      {64, 64, 2, 2.67f, 0.42f, 0.24f, {0.307f, 0.421f}}}},
};
// gemm_bf16_ring_kernel (gemm.hip)
static const TileFamily kBf16Ring = {{{256, 256, 1, 0.0f, 5.04f, 3.33f, {1.265f}}, {}, {}, {}}};

// The estimate at M rows, or summed over the fills of M that a device-buffer
// call may meet.
template <class F>
static double over_fills(int M, bool exact, F&& us_at) {
    if (exact) return us_at(M);
    double us = 0.0;
    for (double fill : {0.5, 0.6, 0.7, 0.8, 0.9, 1.0, 1.0}) us += us_at(std::max(1, (int)(fill * M)));
    return us;
}

static TileChoice choice_for(const TileFamily& f, int N, int nk, bool gelu, int S, bool rest) {
    TileChoice c{};
    for (int i = 0; i < FAM_TILES; ++i) {
        const TileCost& t = f.t[i];
        if (t.bm == 0) continue;                 // a family of fewer tiles
        const float k = (float)nk / (float)S * (rest ? 1.0f + 0.5f * t.rest : 1.0f), e = t.epi + (gelu ? t.epi_gelu : 0.0f);
        c.t[i] = {t.bm == 256 ? 8 : (t.bm == 128 ? 7 : 6), (N + t.bn - 1) / t.bn * S, t.wpc == 2, t.launch,
                  k * t.kt[t.wpc - 1] + e * (float)t.wpc, k * t.kt[0] + e};
    }
    c.inv_cus = 1.0f / (float)device_cu_count();
    return c;
}

static double family_us(const TileChoice& c, int M) {
    double best = 1e30;
    for (int i = 0; i < FAM_TILES; ++i) best = std::min(best, (double)choice_us(c, i, M));
    return best;
}

Gemm16Plan gemm16_pair_plan(int M, bool exact, int N, int K, bool gelu, int min_splits, int max_splits, bool rest,
                            double* us_out) {
    Gemm16Plan best{0, 1};
    double best_us = 1e30;
    for (int i = 0; i < FAMILIES; ++i)
        for (int S : {1, 2, 3, 4, 6, 8}) {
            if (S < min_splits || S > std::max(max_splits, 1) || K % ((rest ? 128 : 64) * S)) continue;
            const TileChoice c = choice_for(kPairFamilies[i], N, K / 32, gelu, S, rest);
            const double us = over_fills(M, exact, [&](int m) {
                return family_us(c, m) + (S - 1) * ((double)m * N * 4e-6 / 4.0);
            });
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
// (measured at 256 .. 40,000 rows, 1 .. 12 splits).  Back to back the two forms
// are within 10% of one another from 6,000 to 33,000 rows of I = 1536 (us, fused
// in its best splits against the products: 6,124 rows 50.7 / 55.4, 10,000 73.6 /
// 77.6, 14,313 102.0 / 102.3, 32,768 206 / 205).  The estimate is weighed at
// 0.95, which decides between forms that close.  In forwards, against no weight:
// full batches of 6,144 and 8,192 rows 1-2% faster, ragged ones of 60-85% of them
// 2-6% slower (649 against 611 us at 3,817 of 6,144), and, since this kernel then
// runs in more splits than the products would, vectors 3% closer to float64.
static double ffn_us(int M, int I, int S) {
    const int cus = device_cu_count();
    const int64_t items = (int64_t)((M + 127) / 128) * S;
    const double chunks = (double)(I / 128) / S;
    auto round = [&](int64_t n) {
        return 3.0 + chunks * 12.6 * (1.0 + 0.64 * std::max(0.0, (double)n / cus - 0.5));
    };
    double us = (double)(items / cus) * round(cus) + (S - 1) * ((double)M * 384 * 4e-6 / 4.0);
    if (items % cus) us += round(items % cus);
    return us;
}

FfnPairPlan ffn_pair_plan(int M, bool exact, int H, int I, int min_splits, int max_splits, bool rest) {
    FfnPairPlan best{};
    double up_us = 0.0, best_us = 1e30;
    best.up = gemm16_pair_plan(M, exact, I, H, true, 1, 1, rest, &up_us);
    best.down = gemm16_pair_plan(M, exact, H, I, false, min_splits, max_splits, rest, &best_us);
    best_us += up_us;
    best.fused = false;
    best.splits = best.down.splits;
    if (rest || !ffn_pair_shape_ok(H, I)) return best;
    for (int S : {1, 2, 3, 4, 6}) {
        if (S < min_splits || S > std::max(max_splits, 1) || (I / 128) % S) continue;
        const double us = 0.95 * over_fills(M, exact, [&](int m) { return ffn_us(m, I, S); });
        if (us < best_us) {
            best_us = us;
            best.fused = true;
            best.splits = S;
        }
    }
    return best;
}

// One family's kernel: enough workgroups for the smallest of its tiles, or all
// that are resident at a time.
template <bool PAIR, bool REST, int EPI, int OUT>
static hipError_t launch_family(Gemm16Args a, int family, hipStream_t s) {
    const TileFamily& f = (PAIR ? kPairFamilies : kBf16Families)[family];
    const int S = a.splits > 1 ? a.splits : 1;
    int64_t items = 0;
    for (const TileCost& t : f.t)
        items = std::max(items, (int64_t)((a.M_max + t.bm - 1) / t.bm) * ((a.N + t.bn - 1) / t.bn) * S);
    if (items == 0) return hipSuccess;
    const TileChoice c = choice_for(f, a.N, a.K / (PAIR ? 32 : 64), EPI == EPI_BIAS_GELU, S, REST);
    const dim3 grid((unsigned)std::min<int64_t>(items, (int64_t)device_cu_count() * (family == 0 ? 1 : 2)));
    if (family == 0) hipLaunchKernelGGL((gemm16_kernel<PAIR, REST, 0, EPI, OUT>), grid, dim3(512), 0, s, a, c);
    else hipLaunchKernelGGL((gemm16_kernel<PAIR, REST, 1, EPI, OUT>), grid, dim3(256), 0, s, a, c);
    return hipGetLastError();
}

hipError_t launch_gemm16_pair(const Gemm16Args& a, int epi, bool out_pair, int family, hipStream_t s) {
    auto al16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
    const int S = a.splits > 1 ? a.splits : 1;
    const bool ok = a.M_max >= 0 && a.N > 0 && a.K > 0 && a.N % 8 == 0 && a.K % ((a.rest ? 128 : 64) * S) == 0 && a.lda % 8 == 0 &&
                    a.ldw % 8 == 0 && a.ldc % 8 == 0 && a.lda >= a.K && a.ldw >= a.K + (a.rest ? a.K / 2 : 0) &&
                    a.ldc >= a.N &&
                    al16(a.A) && al16(a.W) && al16(a.C) && (S == 1 || (epi == EPI_NONE && a.split_stride % 8 == 0)) &&
                    (epi == EPI_NONE || (a.bias && al16(a.bias))) && gemm_offsets_fit32(a.lda, a.ldw, 4) &&
                    a.ldc <= gemm_stride_max(4) && family >= 0 && family < FAMILIES && a.tile < FAM_TILES;
    if (!ok) return hipErrorInvalidValue;
    const bool r = a.rest;
    if (epi == EPI_BIAS && out_pair)
        return r ? launch_family<true, true, EPI_BIAS, OUT_PAIR>(a, family, s) : launch_family<true, false, EPI_BIAS, OUT_PAIR>(a, family, s);
    if (epi == EPI_BIAS_GELU && out_pair)
        return r ? launch_family<true, true, EPI_BIAS_GELU, OUT_PAIR>(a, family, s)
                 : launch_family<true, false, EPI_BIAS_GELU, OUT_PAIR>(a, family, s);
    if (epi == EPI_NONE && !out_pair)
        return r ? launch_family<true, true, EPI_NONE, OUT_F32>(a, family, s) : launch_family<true, false, EPI_NONE, OUT_F32>(a, family, s);
    return hipErrorInvalidValue;
}

bool launch_gemm16_bf16(const GemmArgs& g, int epi, hipStream_t s, hipError_t* err) {
    if (g.M_max <= 0 || g.K % 128 || g.lda < g.K || g.ldw < g.K || g.ldc < g.N || g.ldc > gemm_stride_max(4)) return false;
    const bool exact = g.M_dev == nullptr, gelu = epi == EPI_BIAS_GELU;
    int best = -1;
    // The ring kernel's estimate is weighed at 0.92: its three A stages hide what
    // a forward's cold operands cost the others (measured at one shape: 131,072
    // rows, FFN down, 481 us against 523, where back to back they are within 2%).
    const TileChoice ring = choice_for(kBf16Ring, g.N, g.K / 64, gelu, 1, false);
    double best_us = 0.92 * over_fills(g.M_max, exact, [&](int m) { return (double)choice_us(ring, 0, m); });
    for (int i = 0; i < FAMILIES; ++i) {
        const TileChoice c = choice_for(kBf16Families[i], g.N, g.K / 64, gelu, 1, false);
        const double us = over_fills(g.M_max, exact, [&](int m) { return family_us(c, m); });
        if (us < best_us) {
            best_us = us;
            best = i;
        }
    }
    if (best < 0) return false;
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
    a.tile = -1;
    switch (epi) {
        case EPI_BIAS: *err = launch_family<false, false, EPI_BIAS, OUT_BF16>(a, best, s); break;
        case EPI_BIAS_GELU: *err = launch_family<false, false, EPI_BIAS_GELU, OUT_BF16>(a, best, s); break;
        case EPI_NONE: *err = launch_family<false, false, EPI_NONE, OUT_BF16>(a, best, s); break;
        default: return false;
    }
    return true;
}

}  // namespace ebh
