// gemm16.hpp -- GEMM tiles on the 16-bit matrix cores: fp32 products from
// fp16 pairs, and bf16 products.
//
// Pair format.  An fp32 value x of a matrix with scale s (a power of two) is
// held as two fp16 numbers h = fp16(s x) and l = fp16(s x - h), both rounded
// to nearest even; s x - h is exact in fp32, and h + l is s x to within one
// unit of its 24th bit.  Eight consecutive elements of a row take 32 bytes,
// h0..h7 then l0..l7, so a row of K values takes 4 K bytes as in fp32 and an
// MFMA operand (8 k-consecutive fp16) is one aligned 16-byte chunk.
//
// s a . t b = ah.bh + ah.bl + al.bh, three v_mfma_f32_16x16x32_f16 with every
// product exact in fp32 and sums in fp32; al.bl, below 2^-22 of |a b|, is left
// out.  Measured against float64 the relative error of such a product is 0.62
// of the fp32 MFMA's (K = 384: 2.2e-7 against 3.5e-7; K = 3072: 6.2e-7 against
// 9.9e-7; the same on GELU outputs and on rows with outlier features), because
// the fp32 form rounds its sum every k and this one every 32: the pairs'
// own rounding is a small part of either.  (h and l hold 23 of a value's 24
// bits: three values in four exactly, the fourth off by one unit of the 24th,
// at most 2^-23 of it.)  The error is flat for scales from 2^4 to 2^10, so one
// scale per matrix, taken from a bound of its values, is enough.
//
// The rest.  Rounding errors differ from token to token, and a mean over a
// sequence takes them out; a weight's is the same for every token and stays.
// Over long sequences it is what is left (MiniLM-L6, 512 tokens: 0.9e-7 of the
// vector's 1.5e-7, where fp32 MFMA products give 1.2e-7).  So weight rows carry
// their rest, r = fp16(s w - h - l), which makes them exact, behind their pairs
// (launch_to_pair_rest), and products that are told to add ah.br, one more
// v_mfma_f32_16x16x32_f16 per 32 k: k-tiles of 64 rests against the h of 64 k,
// before the pairs', while the sums are small.  They take 1.2-1.25 times as long
// (forwards: 256 x 128 2.75 -> 3.42 ms, 16 x 512 907 -> 1,094 us, fp32 MFMA 5.7 ms
// and 1,642 us).
//
// The fp16 MFMA rounds its aligned terms down (towards minus infinity), so its
// sums sit 1e-8 (K = 384) to 4e-8 (K = 1536) of their size low on average, a
// small part of a sum's own error and nearly the same for every column, which
// the LayerNorm after the attention-output and FFN-down products takes out.
#pragma once
#include <type_traits>

#include "kernels.hpp"

namespace ebh {

typedef float g16_v4f __attribute__((ext_vector_type(4)));
typedef __bf16 g16_v8bf __attribute__((ext_vector_type(8)));
typedef unsigned int u4v_t __attribute__((ext_vector_type(4)));

enum Out16 : int { OUT_F32 = 0, OUT_PAIR = 1, OUT_BF16 = 2 };

// C = epi(A . W^T + bias), one list of work items (C tiles, N-fastest, times
// the K splits) walked by a persistent grid.  A [M, K] and W [N, K] rows are
// K-contiguous, in pairs (PAIR) or bf16; a k-tile is 128 bytes of each row
// (32 pairs or 64 bf16), staged unpadded in LDS with the row's eight 16-byte
// chunks XOR-swizzled, by direct-to-LDS buffer loads whose descriptors end at
// the last real row (rows past it read as zeros).
//
// Lane group q's operands are chunks 2q and 2q + 1 of a row (pairs: h and l of
// k = 8q .. 8q + 7), or q and q + 4 (bf16: two 32-deep slices of k, in order).
// bf16 sums start at the bias and run over the slices, as the ring kernel's
// (gemm.hip) do, so every tile there is gives a row the same bits, and the tile
// that a batch's size picks does not show in its vectors.  Pairs add the bias
// last: their sums hold a scale of their own.  The MFMAs take W
// as their first operand, so lane (r, q) of a 16 x 16 block holds C row r and
// the block's W rows 4q .. 4q + 3.  W rows are permuted on their way into LDS
// (within each 32, LDS row 16 jj + 4q + e holds column 8q + 4 jj + e), so a lane
// holds eight consecutive columns across two blocks: 32 bytes of fp32 or
// of a pair chunk, stored straight from the accumulators, four lanes to a
// 128-byte line.  The epilogue needs no LDS pass and no barrier, and the next
// k-tile's loads are in flight ahead of its stores.
// fp32 and pair outputs are stored through the caches, whose last level hands
// them to the next kernel (non-temporal: 256 x 128 tokens of MiniLM 2.71 ->
// 3.25 ms, 99 x 250 ragged 1.52 -> 1.65 ms); bf16 outputs non-temporal (through
// the caches 64 x 128 289 -> 296 us, 1024 x 128 of BERT-base 24.45 -> 25.0 ms).
//
// What bounds it: the matrix cores (a 256 x 256 k-tile is 64 KB of loads for
// 3,072 cycles of MFMAs per SIMD).  A k-tile's fragments are read a step (SB
// row blocks) ahead and its last step's MFMAs run after the next k-tile's
// barrier, so that the pipes work while the barrier releases and the first
// fragments arrive; two sets of W fragments make that possible, and k-tiles
// come in pairs so that the sets have fixed registers.
//
// Bias row segments ride in with their tile's first W k-tile, up to nsw - 1
// k-tiles before it is computed.  A tile has at least two k-tiles, so at a tile's
// last k-tile that reaches (nsw - 2) / 2 tiles past the next one: a slot for
// each of those, for the next tile and for the one whose epilogue comes.
constexpr int gemm16_bias_slots(int nsw) { return 2 + (nsw - 2) / 2; }
constexpr int gemm16_lds(int bm, int bn, int waves, int nsa, int nsw, bool bias) {
    return (nsa * bm + nsw * bn) * 128 + (bias ? gemm16_bias_slots(nsw) * waves * 1024 : 0);
}

template <bool PAIR, bool REST, int BM, int BN, int WAVES_M, int WAVES_N, int NSA, int NSW, int EPI, int OUT>
__device__ __forceinline__ void gemm16_body(const Gemm16Args& p, const int M, char* const smem) {
    constexpr int NT = 64 * WAVES_M * WAVES_N, NW = WAVES_M * WAVES_N;
    constexpr int WM = BM / WAVES_M, WN = BN / WAVES_N;
    constexpr int FM = WM / 16, FN = WN / 16;
    static_assert(FM * 16 == WM && FN * 16 == WN && FN % 2 == 0, "wave tile of 16 x 32 blocks");
    constexpr int SB = FM >= 8 ? 2 : 1, NS = FM / SB;
    static_assert(NS % 2 == 0, "steps alternate between two A sets");
    constexpr int ES = PAIR ? 4 : 2, KT = 128 / ES;
    constexpr int RPT = NT / 8;                   // tile rows a pass of loads covers
    constexpr int LA = BM / RPT, LW = BN / RPT;
    static_assert(LA * RPT == BM && LW * RPT == BN && RPT % 32 == 0, "every wave issues the same loads");
    constexpr int ST_A = BM * 128, ST_W = BN * 128;   // bytes of a stage
    constexpr int W_OFF = NSA * ST_A, B_OFF = W_OFF + NSW * ST_W;
    // k-tiles in flight ahead.  A streams from HBM (a forward's operands have left
    // the last-level cache by the time they are read), W comes from the caches:
    // where the LDS is short A has the deeper ring.
    constexpr int DA = NSA - 1, DW = NSW - 1;
    static_assert(DA == DW || DA == DW + 1, "load order");
    constexpr bool HAS_BIAS = EPI != EPI_NONE;
    constexpr int CES = OUT == OUT_BF16 ? 2 : 4;
    constexpr int NSTO = FM * (FN / 2) * (OUT == OUT_BF16 ? 1 : 2);   // stores per lane and tile
    constexpr int BIAS_BYTES = 1024;              // one wave's 64 x 16-byte bias chunks
    constexpr int NBIAS = gemm16_bias_slots(NSW);
    static_assert(gemm16_lds(BM, BN, NW, NSA, NSW, HAS_BIAS) <= (NW == 8 ? 160 : 80) * 1024, "LDS");

    const int N = p.N;
    const int ntn = (N + BN - 1) / BN, ntiles = ((M + BM - 1) / BM) * ntn;
    const int S = EPI == EPI_NONE && p.splits > 1 ? p.splits : 1;
    const int nwork = ntiles * S, nk = p.K / KT / S;   // nk is even and at least 2
    const int nr = REST ? nk / 2 : 0, nkt = nr + nk;   // k-tiles of the rest, even, and of the tile
    // Workgroup b runs on XCD b % 8; each XCD's workgroups take consecutive
    // tiles, which share A row panels in that XCD's L2.  Whole rounds: 32
    // consecutive tiles per XCD and round; otherwise an eighth of the items
    // per XCD, so that the last, partial round spreads over all of them.
    int G = gridDim.x;
    asm("" : "+s"(G));   // opaque: the tiles' bodies share nothing derived from it, which would be held (and spilled) across them
    int u0 = blockIdx.x, ustep = G, uend = nwork;
    if ((G & 7) == 0 && nwork % G == 0) {
        u0 = (blockIdx.x & 7) * (G >> 3) + (blockIdx.x >> 3);
    } else if ((G & 7) == 0) {
        const int x = blockIdx.x & 7;
        ustep = G >> 3;
        u0 = (int)((int64_t)x * nwork / 8) + (blockIdx.x >> 3);
        uend = (int)((int64_t)(x + 1) * nwork / 8);
    }
    const int my_tiles = u0 < uend ? (uend - u0 + ustep - 1) / ustep : 0;
    if (my_tiles == 0) return;  // uniform over the workgroup

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WAVES_N, wn = wave % WAVES_N;
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem;

    // Lane share of a k-tile's loads: tile row r0 + i * RPT, LDS chunk tid % 8.
    const int r0 = tid >> 3;
    const uint32_t chunk = 16 * ((tid & 7) ^ chunk_swizzle16<8>(r0));
    const int rw = (r0 & ~31) + 8 * ((r0 >> 2) & 3) + 4 * ((r0 >> 4) & 1) + (r0 & 3);
    const uint32_t lda_b = (uint32_t)p.lda * ES, ldw_b = (uint32_t)p.ldw * ES;
    const uint32_t avoff = r0 * lda_b + chunk, wvoff = rw * ldw_b + chunk;
    uint32_t avo = REST ? avoff + chunk : avoff;  // k-tiles of the rest: A's h chunks, every other one of 64 k

    // Load cursors: the next k-tile of A and of W to load, their panels'
    // descriptors and k offsets.
    g16_v4i arsrc, wrsrc;
    uint32_t ako = 0, wko = 0;
    const float* bias_src = nullptr;
    int akt = 0, at_ = 0, wkt = 0, wt_ = 0;       // k-tile within the tile, tile
    auto a_at = [&](int t) __attribute__((always_inline)) {
        const int u = u0 + t * ustep, split = u / ntiles, tile = u - split * ntiles, m0 = (tile / ntn) * BM;
        arsrc = make_rsrc(static_cast<const char*>(p.A) + (int64_t)m0 * p.lda * ES, (uint32_t)min(M - m0, BM) * lda_b);
        ako = (uint32_t)(split * nk) * 128;
    };
    auto w_at_tile = [&](int t) __attribute__((always_inline)) {
        const int u = u0 + t * ustep, split = u / ntiles, tile = u - split * ntiles, n0 = (tile - (tile / ntn) * ntn) * BN;
        wrsrc = make_rsrc(static_cast<const char*>(p.W) + (int64_t)n0 * p.ldw * ES, (uint32_t)min(N - n0, BN) * ldw_b);
        wko = REST ? (uint32_t)p.K * 4 + (uint32_t)(split * nk) * 64 : (uint32_t)(split * nk) * 128;
        if (HAS_BIAS) bias_src = p.bias + min(n0 + wn * WN + 4 * lane, N - 4);
    };
    int vm = 0;                                    // vector memory instructions issued by this wave
    // vm after the last load that the next k-tiles to enter need: their W where A
    // runs further ahead, else their A.
    int mark[DW];
#pragma unroll
    for (int d = 0; d < DW; ++d) mark[d] = 0;
    auto issue_w = [&](int iw) __attribute__((always_inline)) {   // the workgroup's iw-th k-tile
        if (wt_ >= my_tiles) return;
        const uint32_t st = lds0 + W_OFF + (uint32_t)(iw % NSW) * ST_W + (uint32_t)wave * 1024;
#pragma unroll
        for (int i = 0; i < LW; ++i) load_lds16_buf(wrsrc, wvoff + i * RPT * ldw_b, wko, st + i * RPT * 128);
        vm += LW;
        if (HAS_BIAS && wkt == 0) {
            load_lds16_async(bias_src, reinterpret_cast<const float*>(smem + B_OFF + ((wt_ % NBIAS) * NW + wave) * BIAS_BYTES));
            ++vm;
        }
        if constexpr (DA > DW) mark[DW - 1] = vm;
        wko += 128;
        ++wkt;
        if (REST && wkt == nr) wko = 2 * (wko - (uint32_t)p.K * 4) - nk * 128;   // from the rest's end to the pairs' start
        if (wkt == nkt) {
            wkt = 0;
            if (++wt_ < my_tiles) w_at_tile(wt_);
        }
    };
    auto issue_a = [&](int ia) __attribute__((always_inline)) {
        if (at_ >= my_tiles) return;
        const uint32_t st = lds0 + (uint32_t)(ia % NSA) * ST_A + (uint32_t)wave * 1024;
#pragma unroll
        for (int i = 0; i < LA; ++i) load_lds16_buf(arsrc, avo + i * RPT * lda_b, ako, st + i * RPT * 128);
        vm += LA;
        if constexpr (DA == DW) mark[DW - 1] = vm;
        ako += REST && akt < nr ? 256 : 128;
        ++akt;
        if (REST && akt == nr) {
            ako -= nk * 128;
            avo = avoff;
        }
        if (akt == nkt) {
            akt = 0;
            if (REST) avo = avoff + chunk;
            if (++at_ < my_tiles) a_at(at_);
        }
    };

    const int r16 = lane & 15, q16 = lane >> 4;
    constexpr uint32_t FX = PAIR ? 16 : 64;       // from a lane's first chunk to its second
    const uint32_t frag = r16 * 128 + 16 * ((PAIR ? 2 * q16 : q16) ^ chunk_swizzle16<8>(r16));
    const uint32_t a_off = wm * WM * 128 + frag, w_off = wn * WN * 128 + frag;
    g16_v4f acc[FM][FN];
    g16_v4f af[2][SB][2], wf[2][FN][2];

    int it = 0;
    auto enter = [&]() __attribute__((always_inline)) {
        const int n = vm - mark[0];
        constexpr auto c = [](int v) { return v > 63 ? 63 : v; };
        // issued after the loads waited for: later k-tiles' A and W (and a bias),
        // and a tile's stores
        constexpr int AH = DA > DW ? LA : (DW - 1) * (LA + LW);
        if constexpr (AH == 0) wait_vmcnt_of<c(NSTO)>(n);
        else if constexpr (DA > DW) wait_vmcnt_of<c(NSTO + AH), AH>(n);
        else wait_vmcnt_of<c(NSTO + AH + 1), c(NSTO + AH), AH + 1, AH>(n);
#pragma unroll
        for (int d = 0; d + 1 < DW; ++d) mark[d] = mark[d + 1];
        lds_barrier();
    };
    auto mfma_step = [&](int s, int as, int ws, auto two) __attribute__((always_inline)) {
        // smallest products first; consecutive MFMAs on different accumulators;
        // two: a lane's two chunks are two runs of k (bf16, the rest), not h and l
        constexpr bool TWO = decltype(two)::value;
#pragma unroll
        for (int pr = TWO ? 1 : 0; pr < 3; ++pr)
#pragma unroll
            for (int i = 0; i < SB; ++i)
#pragma unroll
                for (int j = 0; j < FN; ++j) {
                    g16_v4f& d = acc[s * SB + i][j];
                    if constexpr (PAIR) {
                        const g16_v4f& w = wf[ws][j][TWO ? pr - 1 : (pr == 1 ? 1 : 0)];
                        const g16_v4f& a = af[as][i][TWO ? pr - 1 : (pr == 0 ? 1 : 0)];
                        d = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, w), __builtin_bit_cast(v8h, a), d, 0, 0, 0);
                    } else {
                        d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(g16_v8bf, wf[ws][j][pr - 1]),
                                                                    __builtin_bit_cast(g16_v8bf, af[as][i][pr - 1]), d, 0, 0, 0);
                    }
                }
    };
    auto run_ktile = [&](auto pset, bool first, auto two) __attribute__((always_inline)) {
        constexpr int P = decltype(pset)::value;
        const char *sa = smem + (it % NSA) * ST_A, *sw = smem + W_OFF + (it % NSW) * ST_W;
        auto rd_a = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < SB; ++i) {
                af[s & 1][i][0] = *reinterpret_cast<const g16_v4f*>(sa + a_off + (s * SB + i) * 16 * 128);
                af[s & 1][i][1] = *reinterpret_cast<const g16_v4f*>(sa + (a_off ^ FX) + (s * SB + i) * 16 * 128);
            }
        };
        rd_a(0);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            wf[P][j][0] = *reinterpret_cast<const g16_v4f*>(sw + w_off + j * 16 * 128);
            wf[P][j][1] = *reinterpret_cast<const g16_v4f*>(sw + (w_off ^ FX) + j * 16 * 128);
        }
        if (!first) mfma_step(NS - 1, 1, P ^ 1, two);   // the previous k-tile's last step
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s == 0) issue_w(it + DW);
            if (s == 1) issue_a(it + DA);
            if (s + 1 < NS) rd_a(s + 1);
            if (s + 1 < NS) mfma_step(s, s & 1, P, two);
        }
        ++it;
    };

    // This wave's bias row segment of local tile t.
    auto bias_of = [&](int t) __attribute__((always_inline)) { return smem + B_OFF + ((t % NBIAS) * NW + wave) * BIAS_BYTES; };
    auto epilogue = [&](int t) __attribute__((always_inline)) {
        const int u = u0 + t * ustep, split = u / ntiles, tile = u - split * ntiles;
        const int mt = tile / ntn, wrow = mt * BM + wm * WM, n0 = (tile - mt * ntn) * BN;
        char* const cb = static_cast<char*>(p.C) + (EPI == EPI_NONE ? (int64_t)split * p.split_stride * CES : 0);
        const int64_t rowb = p.ldc * CES;
        // lane-derived values opaque here: formed at the epilogue, not held across the k-loop
        int el = lane;
        asm volatile("" : "+v"(el));
        const int er = el & 15, eq = el >> 4;
        const char* bs = bias_of(t) + 32 * eq;
        const float sc = p.acc_scale, so = p.out_scale;
        g16_v4f bb0[FN / 2], bb1[FN / 2]; uint32_t vo[FN / 2];
#pragma unroll
        for (int jp = 0; jp < FN / 2; ++jp) {
            bb0[jp] = bb1[jp] = g16_v4f{0, 0, 0, 0};
            if (PAIR && HAS_BIAS) {
                bb0[jp] = *reinterpret_cast<const g16_v4f*>(bs + jp * 128);
                bb1[jp] = *reinterpret_cast<const g16_v4f*>(bs + jp * 128 + 16);
            }
            const int col = n0 + wn * WN + 32 * jp + 8 * eq;
            vo[jp] = col < N ? (uint32_t)(er * (int)rowb + col * CES) : 0xFFFFFFE0u;   // N % 8 == 0
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
#pragma unroll
            for (int jp = 0; jp < FN / 2; ++jp) {
                const g16_v4f b0 = bb0[jp], b1 = bb1[jp];
                const uint32_t voff = vo[jp];
                float v[8];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    if constexpr (PAIR) {
                        v[e] = HAS_BIAS ? fmaf(acc[i][2 * jp][e], sc, b0[e]) : acc[i][2 * jp][e] * sc;
                        v[4 + e] = HAS_BIAS ? fmaf(acc[i][2 * jp + 1][e], sc, b1[e]) : acc[i][2 * jp + 1][e] * sc;
                    } else {
                        v[e] = acc[i][2 * jp][e];
                        v[4 + e] = acc[i][2 * jp + 1][e];
                    }
                    if constexpr (EPI == EPI_BIAS_GELU) {
                        v[e] = gelu_tanh_fast(v[e]);
                        v[4 + e] = gelu_tanh_fast(v[4 + e]);
                    }
                }
                const int left = __builtin_amdgcn_readfirstlane(M - wrow - 16 * i);
                const int bytes = (left >= 16 ? 16 : (left > 0 ? left : 0)) * (int)rowb;
                const __amdgpu_buffer_rsrc_t cr = __builtin_amdgcn_make_buffer_rsrc(
                    cb + (int64_t)__builtin_amdgcn_readfirstlane(wrow + 16 * i) * rowb, (short)0, bytes, G16_RSRC_WORD3);
                if constexpr (OUT == OUT_F32) {
                    __builtin_amdgcn_raw_buffer_store_b128(
                        u4v_t{__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])}, cr, voff, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b128(
                        u4v_t{__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])}, cr, voff + 16, 0, 0);
                } else if constexpr (OUT == OUT_PAIR) {
                    u4v_t h, l;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        uint32_t hw, lw;
                        split_f16x2(v[2 * e] * so, v[2 * e + 1] * so, hw, lw);
                        h[e] = hw;
                        l[e] = lw;
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(h, cr, voff, 0, 0);
                    __builtin_amdgcn_raw_buffer_store_b128(l, cr, voff + 16, 0, 0);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b128(
                        u4v_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]), pack_bf16x2(v[6], v[7])},
                        cr, voff, 0, 2 /* nt */);
                }
            }
        }
        vm += NSTO;
    };

    // Prologue, in the order of the loop: k-tile d's A before its W where A runs
    // ahead (whose mark is its W), else W first.
    a_at(0);
    w_at_tile(0);
    if constexpr (DA > DW) issue_a(0);
#pragma unroll
    for (int d = 0; d < DW; ++d) {
        issue_w(d);
        issue_a(d + DA - DW);
        if constexpr (DA == DW) mark[d] = vm;
    }
    if constexpr (DA > DW) static_assert(DW == 1, "one mark");
    typedef std::integral_constant<int, 0> set0;
    typedef std::integral_constant<int, 1> set1;
    for (int t = 0; t < my_tiles; ++t) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] = g16_v4f{0.0f, 0.0f, 0.0f, 0.0f};
        enter();
        if constexpr (!PAIR && HAS_BIAS) {         // it came with the tile's first W
#pragma unroll
            for (int j = 0; j < FN; ++j) {
                const g16_v4f b = *reinterpret_cast<const g16_v4f*>(bias_of(t) + 32 * q16 + (j >> 1) * 128 + (j & 1) * 16);
#pragma unroll
                for (int i = 0; i < FM; ++i) acc[i][j] = b;
            }
        }
        if constexpr (REST) {                      // the smallest products, while the sums are small
            run_ktile(set0{}, true, std::true_type{});
            enter();
            run_ktile(set1{}, false, std::true_type{});
            for (int kt = 2; kt < nr; kt += 2) {
                enter();
                run_ktile(set0{}, false, std::true_type{});
                enter();
                run_ktile(set1{}, false, std::true_type{});
            }
            mfma_step(NS - 1, 1, 1, std::true_type{});
            enter();
        }
        typedef std::integral_constant<bool, !PAIR> two;
        run_ktile(set0{}, true, two{});
        enter();
        run_ktile(set1{}, false, two{});
        for (int kt = 2; kt < nk; kt += 2) {
            enter();
            run_ktile(set0{}, false, two{});
            enter();
            run_ktile(set1{}, false, two{});
        }
        mfma_step(NS - 1, 1, 1, two{});
        epilogue(t);
    }
}

// ---------------------------------------------------------------------------
// The tiles, in two families that each are one kernel: a device-buffer call
// knows only the padded row count, so the host picks the family and the kernel,
// which reads the real count, the tile.  Cost model (us; host and device): with
// n items on the busiest CU, wpc of them resident at a time,
//   launch + sum over rounds of (k-tiles * kt[resident] + resident * epi).
// ---------------------------------------------------------------------------
struct TileCost {
    int bm, bn, wpc;
    float launch, epi, epi_gelu, kt[2];
    float rest;                                  // a k-tile of the rest, in pair k-tiles
};
constexpr int FAM_TILES = 4;                     // tiles per family
struct TileFamily {
    TileCost t[FAM_TILES];
};

// The model for one shape as the kernel evaluates it: few operations, no
// divisions, since every launch waits for the choice.
struct TileChoice {
    struct {
        int bm_shift, cols;                      // log2 of the tile's rows; column tiles times splits
        int two;                                 // two workgroups per CU
        float launch, full, rem;                 // us: fixed, a full round, a last round of one per CU
    } t[FAM_TILES];
    float inv_cus;
};

__host__ __device__ inline float choice_us(const TileChoice& c, int i, int M) {
    const int items = ((M + (1 << c.t[i].bm_shift) - 1) >> c.t[i].bm_shift) * c.t[i].cols;
    const int per = (int)((float)items * c.inv_cus + 0.9999f);
    const int full = c.t[i].two ? per >> 1 : per, rem = c.t[i].two ? per & 1 : 0;
    return c.t[i].launch + (float)full * c.t[i].full + (float)rem * c.t[i].rem;
}

template <bool PAIR, bool REST, int FAM, int EPI, int OUT>
__global__ __launch_bounds__(FAM == 0 ? 512 : 256, 2) void gemm16_kernel(Gemm16Args p, TileChoice f) {
    constexpr bool HB = EPI != EPI_NONE;
    // With no bias row to keep, 256 x 256 and 128 x 128 have room for a third A stage.
    constexpr int NA0 = HB ? 2 : 3;
    __shared__ __attribute__((aligned(16))) char smem[FAM == 0 ? 160 * 1024 : 80 * 1024];
    const int M = p.M_dev ? *p.M_dev : p.M_max;
    int tile = p.tile;
    if (tile < 0) {
        float best = 1e30f;
#pragma unroll
        for (int i = 0; i < FAM_TILES; ++i) {
            const float us = choice_us(f, i, M);
            if (us < best) {
                best = us;
                tile = i;
            }
        }
    }
    tile = __builtin_amdgcn_readfirstlane(tile);
    if constexpr (FAM == 0) {
        if (tile == 0) gemm16_body<PAIR, REST, 256, 256, 2, 4, NA0, 2, EPI, OUT>(p, M, smem);
        else if (tile == 1) gemm16_body<PAIR, REST, 256, 192, 4, 2, 3, 2, EPI, OUT>(p, M, smem);
        else if (tile == 2) gemm16_body<PAIR, REST, 256, 128, 4, 2, 3, 3, EPI, OUT>(p, M, smem);
        else gemm16_body<PAIR, REST, 128, 128, 2, 4, 4, 4, EPI, OUT>(p, M, smem);
    } else {
        if (tile == 0) gemm16_body<PAIR, REST, 128, 128, 2, 2, NA0, 2, EPI, OUT>(p, M, smem);
        else if (tile == 1) gemm16_body<PAIR, REST, 128, 96, 4, 1, 3, 2, EPI, OUT>(p, M, smem);
        else if (tile == 2) gemm16_body<PAIR, REST, 64, 128, 2, 2, 3, 3, EPI, OUT>(p, M, smem);
        else gemm16_body<PAIR, REST, 64, 64, 2, 2, 4, 4, EPI, OUT>(p, M, smem);
    }
}

}  // namespace ebh
