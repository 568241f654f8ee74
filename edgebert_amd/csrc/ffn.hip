// ffn.hip -- FFN up + GELU + FFN down of the fp32 pair forward in one launch
// (src/lib.rs:739-750, 958-978; H = 384).
//
// As two products, the GELU output goes through HBM twice: at 32k tokens of
// MiniLM-L6 201 MB out and 201 MB in, and its stores alone are a fifth of the
// up product's time.  Here a workgroup (8 waves, one per CU) takes 128 rows and
// a range of the intermediate columns, 128 at a time, and each chunk of GELU
// output lives in LDS only:
//   1. U = X . W1[chunk]^T over K = 384: 12 k-tiles of 32 pairs, waves 4 x 2 of
//      32 x 64;
//   2. gelu(U + b1) as pairs into LDS (64 KB, laid out as four A k-tiles);
//   3. Y += G . W2[:, chunk]^T: 4 k-tiles, waves 2 x 4 of 64 x 96, the 128 x 384
//      sums in registers (96 a lane) for the whole range.
// A row block's ranges (splits) are workgroups of their own, writing partial
// sums that the LayerNorm adds in order, as split-K products do.
//
// LDS is all 160 KB (so there is no room for the weights' rest, and products
// that need it run as two): G, and 96 KB that step 1 uses as three stages of 32 KB (X
// and W1, two k-tiles in flight ahead) and step 3 as two of 48 KB (W2).  The
// steps hand it over without a gap: W2's first k-tile is loaded during step 1's
// last k-tile (into the two stages that are done), its second during the GELU,
// and the next chunk's first k-tile during step 3's last.  b1 rides into the
// part of G that its own wave will write.  Products, fragment order and the
// deferred last step of each k-tile are those of gemm16.hpp, so the sums are
// the same as theirs.
#include "gemm16.hpp"

#include <algorithm>

namespace ebh {

namespace {

constexpr int FH = 384, FBM = 128, FBC = 128;          // width, rows, chunk columns
constexpr int K1T = FH / 32;                           // k-tiles of step 1
constexpr int G_BYTES = FBM * FBC * 4, ST1 = (FBM + FBC) * 128, ST2 = FH * 128;
constexpr int FFN_LDS = G_BYTES + 3 * ST1;
static_assert(2 * ST2 == 3 * ST1 && FFN_LDS == 160 * 1024, "the two steps share one region");

__global__ __launch_bounds__(512, 2) void ffn_pair_kernel(FfnPairArgs p) {
    __shared__ __attribute__((aligned(16))) char smem[FFN_LDS];
    char* const G = smem;
    char* const R = smem + G_BYTES;

    const int M = p.M_dev ? *p.M_dev : p.M_max;
    const int nblk = (M + FBM - 1) / FBM;
    // Item = (split, row block).  Workgroup b runs on XCD b % 8; an XCD takes an
    // eighth of the items in a row, so its workgroups walk the same weights.
    const int nitems = nblk * p.splits, per = (nitems + 7) >> 3;
    const int local = blockIdx.x >> 3, item = (blockIdx.x & 7) * per + local;
    if (local >= per || item >= nitems) return;  // uniform over the workgroup
    const int split = item / nblk, m0 = (item - split * nblk) * FBM;
    const int nch = p.I / FBC / p.splits, c0 = split * nch;

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, q16 = lane >> 4;
    const int wm1 = wave >> 1, wn1 = wave & 1;          // step 1: 32 x 64 per wave
    const int wm2 = wave >> 2, wn2 = wave & 3;          // step 3: 64 x 96 per wave
    const uint32_t lds0 = (uint32_t)(uintptr_t)smem, ldsR = lds0 + G_BYTES;

    // Lane share of every load: tile row r0 + 64 i, chunk tid % 8; W rows permuted
    // within each 32 as in gemm16.hpp.
    const int r0 = tid >> 3;
    const uint32_t chunk = 16 * ((tid & 7) ^ chunk_swizzle16<8>(r0));
    const int rw = (r0 & ~31) + 8 * ((r0 >> 2) & 3) + 4 * ((r0 >> 4) & 1) + (r0 & 3);
    constexpr uint32_t XB = FH * 4;
    const uint32_t w1b = (uint32_t)p.ldw1 * 4, w2b = (uint32_t)p.ldw2 * 4;
    const uint32_t xvo = r0 * XB + chunk, w1vo = rw * w1b + chunk, w2vo = rw * w2b + chunk;
    const g16_v4i xr = make_rsrc(p.X + (int64_t)m0 * FH, (uint32_t)min(M - m0, FBM) * XB);
    const g16_v4i w2r = make_rsrc(p.W2, (uint32_t)FH * w2b);
    auto issue_k = [&](int c, int j) __attribute__((always_inline)) {   // step 1's k-tile j of chunk c: 4 loads
        const g16_v4i w1r = make_rsrc(p.W1 + (int64_t)c * FBC * p.ldw1, FBC * w1b);
        const uint32_t st = ldsR + (uint32_t)(j % 3) * ST1 + wave * 1024, ko = j * 128;
#pragma unroll
        for (int i = 0; i < 2; ++i) load_lds16_buf(xr, xvo + i * 64 * XB, ko, st + i * 8192);
#pragma unroll
        for (int i = 0; i < 2; ++i) load_lds16_buf(w1r, w1vo + i * 64 * w1b, ko, st + FBM * 128 + i * 8192);
    };
    auto issue_w = [&](int c, int kt) __attribute__((always_inline)) {  // step 3's k-tile kt: 6 loads
        const uint32_t st = ldsR + (uint32_t)(kt & 1) * ST2 + wave * 1024, ko = (uint32_t)(c * FBC + kt * 32) * 4;
#pragma unroll
        for (int i = 0; i < 6; ++i) load_lds16_buf(w2r, w2vo + i * 64 * w2b, ko, st + i * 8192);
    };
    // b1 of this wave's 64 columns (lanes past them load copies) into the first
    // KB of the part of G that it writes: rows 32 wm1 .. of k-tile 2 wn1.
    char* const gw = G + 2 * wn1 * (FBM * 128) + wm1 * 32 * 128;
    auto issue_b = [&](int c) __attribute__((always_inline)) {          // 1 load
        load_lds16_async(p.b1 + c * FBC + wn1 * 64 + 4 * r16, reinterpret_cast<const float*>(gw));
    };

    const uint32_t frag = r16 * 128 + 16 * ((2 * q16) ^ chunk_swizzle16<8>(r16));
    g16_v4f acc2[4][6];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 6; ++j) acc2[i][j] = g16_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    g16_v4f af[2][2], wf[2][6][2];
    auto rd = [&](const char* at, uint32_t off, g16_v4f (&f)[2]) __attribute__((always_inline)) {
        f[0] = *reinterpret_cast<const g16_v4f*>(at + off);
        f[1] = *reinterpret_cast<const g16_v4f*>(at + (off ^ 16));
    };
    auto products = [&](auto& acc, int i, auto fn, int as, int ws) __attribute__((always_inline)) {
        constexpr int FN = decltype(fn)::value;
#pragma unroll
        for (int pr = 0; pr < 3; ++pr)
#pragma unroll
            for (int j = 0; j < FN; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, wf[ws][j][pr == 1 ? 1 : 0]),
                                                                   __builtin_bit_cast(v8h, af[as][pr == 0 ? 1 : 0]),
                                                                   acc[i][j], 0, 0, 0);
    };
    typedef std::integral_constant<int, 4> n4;
    typedef std::integral_constant<int, 6> n6;
    auto enter = [&](auto n) __attribute__((always_inline)) {   // at most n loads of this wave in flight
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n)::value) : "memory");
        lds_barrier();
    };
    typedef std::integral_constant<int, 0> w0;
    typedef std::integral_constant<int, 5> w5;

    issue_k(c0, 0);
    for (int c = c0; c < c0 + nch; ++c) {
        // Step 1.
        g16_v4f acc1[2][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc1[i][j] = g16_v4f{0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t a1 = wm1 * 32 * 128 + frag, b1 = FBM * 128 + wn1 * 64 * 128 + frag;
        auto ktile1 = [&](int j, auto set, bool first) __attribute__((always_inline)) {
            constexpr int P = decltype(set)::value;
            const char* st = R + (j % 3) * ST1;
            rd(st, a1, af[0]);
#pragma unroll
            for (int jj = 0; jj < 4; ++jj) rd(st, b1 + jj * 16 * 128, wf[P][jj]);
            if (!first) products(acc1, 1, n4{}, 1, P ^ 1);
        };
        auto rest1 = [&](int j, auto set) __attribute__((always_inline)) {
            rd(R + (j % 3) * ST1, a1 + 16 * 128, af[1]);
            products(acc1, 0, n4{}, 0, decltype(set)::value);
        };
        typedef std::integral_constant<int, 0> s0;
        typedef std::integral_constant<int, 1> s1;
        // k-tile j waits for its own loads; issued after them: j = 1: k-tile 2
        // and b1; 2: b1 and k-tile 3; 3 .. 10: k-tile j + 1; 0 and 11: nothing.
        enter(w0{});
        ktile1(0, s0{}, true);
        issue_k(c, 1);
        issue_k(c, 2);
        issue_b(c);
        rest1(0, s0{});
        enter(w5{});
        ktile1(1, s1{}, false);
        issue_k(c, 3);
        rest1(1, s1{});
        enter(w5{});
        ktile1(2, s0{}, false);
        issue_k(c, 4);
        rest1(2, s0{});
#pragma unroll 1
        for (int j = 3; j < 11; j += 2) {
            enter(n4{});
            ktile1(j, s1{}, false);
            issue_k(c, j + 2);
            rest1(j, s1{});
            enter(n4{});
            ktile1(j + 1, s0{}, false);
            if (j + 3 < K1T) issue_k(c, j + 3);
            rest1(j + 1, s0{});
        }
        enter(w0{});
        ktile1(11, s1{}, false);
        issue_w(c, 0);                       // k-tiles 9 and 10 are done: the first 64 KB are free
        rest1(11, s1{});
        products(acc1, 1, n4{}, 1, 1);
        lds_barrier();                       // k-tile 11's stage is free too
        issue_w(c, 1);

        // Step 2: this wave's 32 x 64 of G.
        {
            const float sc = p.scale1, so = p.scale_g;
            g16_v4f bv[2][2];
#pragma unroll
            for (int jp = 0; jp < 2; ++jp) {
                bv[jp][0] = *reinterpret_cast<const g16_v4f*>(gw + 128 * jp + 32 * q16);
                bv[jp][1] = *reinterpret_cast<const g16_v4f*>(gw + 128 * jp + 32 * q16 + 16);
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // before this wave's rows overwrite it
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int jp = 0; jp < 2; ++jp) {
                    float v[8];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        v[e] = gelu_tanh_fast(fmaf(acc1[i][2 * jp][e], sc, bv[jp][0][e])) * so;
                        v[4 + e] = gelu_tanh_fast(fmaf(acc1[i][2 * jp + 1][e], sc, bv[jp][1][e])) * so;
                    }
                    uint4 h, l;
                    split_f16x2(v[0], v[1], h.x, l.x);
                    split_f16x2(v[2], v[3], h.y, l.y);
                    split_f16x2(v[4], v[5], h.z, l.z);
                    split_f16x2(v[6], v[7], h.w, l.w);
                    char* const at = gw + jp * (FBM * 128) + i * 16 * 128;
                    *reinterpret_cast<uint4*>(at + frag) = h;
                    *reinterpret_cast<uint4*>(at + (frag ^ 16)) = l;
                }
        }

        // Step 3.  k-tile kt waits for its W2; after it at most the next one's.
        const uint32_t a2 = wm2 * 64 * 128 + frag, b2 = wn2 * 96 * 128 + frag;
        auto ktile2 = [&](int kt, auto set, bool first) __attribute__((always_inline)) {
            constexpr int P = decltype(set)::value;
            const char *ga = G + kt * (FBM * 128), *st = R + (kt & 1) * ST2;
            rd(ga, a2, af[0]);
#pragma unroll
            for (int jj = 0; jj < 6; ++jj) rd(st, b2 + jj * 16 * 128, wf[P][jj]);
            if (!first) products(acc2, 3, n6{}, 1, P ^ 1);
        };
        auto rest2 = [&](int kt, auto set) __attribute__((always_inline)) {
            const char* ga = G + kt * (FBM * 128);
#pragma unroll
            for (int s = 0; s < 3; ++s) {
                rd(ga, a2 + (s + 1) * 16 * 128, af[(s + 1) & 1]);
                products(acc2, s, n6{}, s & 1, decltype(set)::value);
            }
        };
        enter(n6{});
        ktile2(0, s0{}, true);
        rest2(0, s0{});
        enter(w0{});
        ktile2(1, s1{}, false);
        issue_w(c, 2);
        rest2(1, s1{});
        enter(w0{});
        ktile2(2, s0{}, false);
        issue_w(c, 3);
        rest2(2, s0{});
        enter(w0{});
        ktile2(3, s1{}, false);
        if (c + 1 < c0 + nch) issue_k(c + 1, 0);   // k-tile 2's W2 stage is free
        rest2(3, s1{});
        products(acc2, 3, n6{}, 1, 1);
    }

    // Partial `split` of Y: lane (r16, q16) holds row r16 of a block and eight
    // consecutive columns of each 32.
    float* const Y = p.Y + (int64_t)split * p.split_stride;
    const float sc = p.scale2;
    const uint32_t vo = r16 * XB + (wn2 * 96 + 8 * q16) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = __builtin_amdgcn_readfirstlane(m0 + wm2 * 64 + 16 * i), left = M - row;
        const int bytes = (left >= 16 ? 16 : (left > 0 ? left : 0)) * (int)XB;
        const __amdgpu_buffer_rsrc_t cr =
            __builtin_amdgcn_make_buffer_rsrc(Y + (int64_t)row * FH, (short)0, bytes, G16_RSRC_WORD3);
#pragma unroll
        for (int jp = 0; jp < 3; ++jp)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const g16_v4f a = acc2[i][2 * jp + h];
                __builtin_amdgcn_raw_buffer_store_b128(
                    u4v_t{__float_as_uint(a[0] * sc), __float_as_uint(a[1] * sc), __float_as_uint(a[2] * sc), __float_as_uint(a[3] * sc)},
                    cr, vo + 128 * jp + 16 * h, 0, 0);
            }
    }
}

}  // namespace

constexpr int FFN_MAX_I = (1 << 20) / 4;   // 384 rows of W2, 6 bytes an element, below 2^32 bytes

bool ffn_pair_shape_ok(int H, int I) { return H == FH && I > 0 && I % FBC == 0 && I <= FFN_MAX_I; }

hipError_t launch_ffn_pair(const FfnPairArgs& a, hipStream_t s) {
    auto al16 = [](const void* q) { return ((uintptr_t)q & 15) == 0; };
    if (a.M_max < 0 || a.I <= 0 || a.I % FBC || a.splits < 1 || (a.I / FBC) % a.splits || a.I > FFN_MAX_I ||
        a.ldw1 < FH || a.ldw2 < a.I || a.ldw1 % 4 || a.ldw2 % 4 || a.ldw1 > (1 << 20) || a.ldw2 > (1 << 20) ||
        !al16(a.X) || !al16(a.W1) || !al16(a.W2) || !al16(a.b1) || !al16(a.Y) || a.split_stride % 4)
        return hipErrorInvalidValue;
    const int64_t items = (int64_t)((a.M_max + FBM - 1) / FBM) * a.splits;
    if (items == 0) return hipSuccess;
    hipLaunchKernelGGL(ffn_pair_kernel, dim3((unsigned)(8 * ((items + 7) / 8))), dim3(512), 0, s, a);
    return hipGetLastError();
}

}  // namespace ebh
