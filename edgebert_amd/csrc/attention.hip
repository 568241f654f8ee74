// attention.hip -- masked multi-head self-attention over packed sequences.
//
// Replaces, per (sequence, head), the reference chain
//   q.k^T (matmul_4d, src/lib.rs:713, 898-956) -> * scale (714) ->
//   key-padding mask to -inf (717, 872-896) -> row softmax (720, 851-870) ->
//   P.V (723) -> permute back (726-730)
// without materialising the [S, S] score matrix in HBM.  Tokens are packed
// (only mask == 1 tokens exist), so the key-padding mask becomes "key index <
// sequence length"; a padded key contributes exactly 0, as exp(-inf) does in
// the reference.
//
// Work split: workgroup = (head, 128-query block, sequence), 4 waves of 32
// queries.  K and V of the sequence stream through LDS in 64-key chunks
// (sequences of at most 128 tokens) or 128-key chunks; softmax is online
// across chunks.  The grid's
// sequence index goes through `order` when the caller has one (the packing
// scan writes the sequences longest first), so that the long sequences'
// workgroups start first.
//
// Transposed scores: each wave computes S^T = K . Q^T with
// v_mfma_f32_32x32x2_f32, so lane l owns query l%32 and, for each 32-key
// block, keys 8*(r/4) + 4*(l/32) + r%4 (r = 0..15).  Row max / sum are then
// per-lane reductions plus one exchange with lane l^32, and the
// probabilities already sit in an operand layout of the P.V MFMA (query =
// l%32, one key per lane half), so P never leaves registers.  The context is
// accumulated transposed too, O^T = V^T . P^T: lane l then holds dims
// 8*(r/4) + 4*(l/32) + r%4 of its own query l%32, so the online-softmax
// rescale and the final division use the lane's own statistics, and the
// context leaves as 16-byte stores of four consecutive dims.
#include <algorithm>

#include "kernels.hpp"

namespace ebh {

typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));

// One key chunk (up to 128 keys, in 32-key blocks) of the fp32 kernel below
// for the wave's 32 queries: S^T = K . Q^T, the key-padding mask, the
// online-softmax update and context^T += V^T . P^T.  lim = real keys in the
// chunk (1..128); c2 = scale log2(e).  Fewer VALU instructions matter here: on this chip the VALU does
// not issue while an fp32 MFMA of the same SIMD runs, so the softmax's
// instructions add to the MFMA time instead of hiding behind it.
template <int HD>
__device__ __forceinline__ void attend_chunk(const float* Ks, const float* Vs, const v4f* qf, float c2, int l32,
                                             int half, int lim, v16f* o, float& m_run, float& l_run, bool first) {
    constexpr int KS = HD + 4, NJ = HD / 32;
    v16f sc[4];
    float cmax = -INFINITY;
    const int lim_h = lim - 4 * half;   // key kb*32 + 8(r/4) + r%4 + 4 half is real iff kb*32 + 8(r/4) + r%4 < lim_h
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb * 32 < lim) {
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[kb][r] = 0.0f;
            const float* kr = Ks + (kb * 32 + l32) * KS + 4 * half;
#pragma unroll
            for (int s = 0; s < HD / 8; ++s) {
                const v4f kf = *reinterpret_cast<const v4f*>(kr + s * 8);
#pragma unroll
                for (int q = 0; q < 4; ++q) sc[kb] = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[q], qf[s][q], sc[kb], 0, 0, 0);
            }
            // Key-padding mask (src/lib.rs:887-891), only in the block that
            // straddles the sequence end; the row max is taken over the raw
            // scores (scale > 0 commutes with max).
            if ((kb + 1) * 32 > lim) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (kb * 32 + 8 * (r >> 2) + (r & 3) >= lim_h) sc[kb][r] = -INFINITY;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) cmax = fmaxf(cmax, sc[kb][r]);
        }
    }
    cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
    // exp(scale (s - m)) as 2^(s c - m c), c = scale log2(e): the scale after
    // q.k^T (src/lib.rs:714) folded into one FMA per score.  m and m_run are
    // raw-score maxima; alpha = 0 on the first chunk.  The exponent is off by
    // at most 3 eps |s c - m c| + eps |m c| (the roundings of c, m c and the
    // FMA; eps = 2^-24), which exp2 turns into a relative error of that times
    // ln 2 plus its own 1 ulp.
    const float m_new = fmaxf(m_run, cmax);
    const float mc = m_new * c2;
    const float alpha = __builtin_amdgcn_exp2f(m_run * c2 - mc);
    float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb * 32 < lim) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pr = __builtin_amdgcn_exp2f(fmaf(sc[kb][r], c2, -mc));
                sc[kb][r] = pr;
                ps[r & 3] += pr;
            }
        }
    }
    l_run = l_run * alpha + ((ps[0] + ps[1]) + (ps[2] + ps[3]));
    m_run = m_new;
    if (!first) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[j][r] *= alpha;
    }
    // context^T += V^T . P^T: A = V^T (row = dim l32, one key per lane half),
    // B = P^T (that key, column = query l32).
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb * 32 < lim) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = kb * 32 + 8 * (r >> 2) + 4 * half + (r & 3);
#pragma unroll
                for (int j = 0; j < NJ; ++j)
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x2f32(Vs[key * HD + j * 32 + l32], sc[kb][r], o[j], 0, 0, 0);
            }
        }
    }
}

// KC = keys per LDS chunk.  With 64-key chunks (sequences of at most 128
// tokens) the next chunk's K and V are loaded into registers while the
// current chunk's MFMAs run, and the smaller chunk leaves room for four
// workgroups per CU (c3: 69.5 -> 65.8 us per layer against one 128-key chunk);
// longer sequences keep 128-key chunks, loaded when they are needed, three
// workgroups per CU (c4: 53.1 against 53.9 us with 64-key chunks).
template <int HD, int KC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HD == 32 ? (KC == 64 ? 4 : 3) : 2))) void attention_kernel(
    const float* __restrict__ qkv, const int* __restrict__ cu_seqlens, float* __restrict__ ctx_out, int H, float scale,
    const int* __restrict__ order) {
    constexpr bool PREFETCH = KC == 64;
    constexpr int KS = HD + 4;     // K row stride (floats): conflict-free 16-B reads
    constexpr int NJ = HD / 32;    // 32-wide output blocks of the context
    __shared__ __attribute__((aligned(16))) float Ks[KC * KS];
    __shared__ __attribute__((aligned(16))) float Vs[KC * HD];

    const int head = blockIdx.x, qb = blockIdx.y, b = order ? order[blockIdx.z] : (int)blockIdx.z;
    const int start = cu_seqlens[b];
    const int len = cu_seqlens[b + 1] - start;
    if (qb * 128 >= len) return;  // uniform over the workgroup

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int64_t ld = 3 * (int64_t)H;
    const float* Qg = qkv + (int64_t)start * ld + head * HD;
    const float* Kg = Qg + H;
    const float* Vg = Qg + 2 * H;

    // K and V of a chunk, float4 pieces in registers (with PREFETCH the next
    // chunk's loads go out before the current chunk's MFMAs, so only the first
    // chunk waits for memory).
    constexpr int F4 = KC * HD / 4;       // float4 pieces of K (and of V)
    constexpr int PT = F4 / 256;          // per thread
    static_assert(PT * 256 == F4, "whole pieces per thread");
    float4 kv[PT], vv[PT];
    auto load_chunk = [&](int kbase) {
#pragma unroll
        for (int pi = 0; pi < PT; ++pi) {
            const int i = tid + 256 * pi, key = kbase + i / (HD / 4), cc = i % (HD / 4);
            kv[pi] = vv[pi] = make_float4(0, 0, 0, 0);
            if (key < len) {
                kv[pi] = *reinterpret_cast<const float4*>(Kg + (int64_t)key * ld + cc * 4);
                vv[pi] = *reinterpret_cast<const float4*>(Vg + (int64_t)key * ld + cc * 4);
            }
        }
    };
    if (PREFETCH) load_chunk(0);

    // This lane's query row as the B operand of S^T = K . Q^T.
    const int q0 = qb * 128 + wave * 32;
    const int qi = min(q0 + l32, len - 1);
    v4f qf[HD / 8];
#pragma unroll
    for (int s = 0; s < HD / 8; ++s)
        qf[s] = *reinterpret_cast<const v4f*>(Qg + (int64_t)qi * ld + s * 8 + 4 * half);

    v16f o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[j][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    const float c_exp = scale * 1.4426950408889634f;   // exponent scale of the softmax (base 2)

    const int nchunks = (len + KC - 1) / KC;
    for (int c = 0; c < nchunks; ++c) {
        __syncthreads();  // previous chunk fully consumed
        if (!PREFETCH) load_chunk(c * KC);
#pragma unroll
        for (int pi = 0; pi < PT; ++pi) {
            const int i = tid + 256 * pi, r = i / (HD / 4), cc = i % (HD / 4);
            *reinterpret_cast<float4*>(&Ks[r * KS + cc * 4]) = kv[pi];
            *reinterpret_cast<float4*>(&Vs[r * HD + cc * 4]) = vv[pi];
        }
        __syncthreads();
        if (PREFETCH && c + 1 < nchunks) load_chunk((c + 1) * KC);
        // A wave whose 32 queries all lie past the sequence end (the last
        // query block of a ragged sequence) only helps load K and V.
        if (q0 < len)
            attend_chunk<HD>(Ks, Vs, qf, c_exp, l32, half, min(len - c * KC, KC), o, m_run, l_run, c == 0);
    }

    // Normalise by the row sum (both lane halves hold partial sums) and store:
    // lane holds dims j*32 + 8*g + 4*half + 0..3 (g = r / 4) of query l32.
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const int q = q0 + l32;
    if (q < len) {
        const float inv = 1.0f / l_tot;
        const int64_t at = (int64_t)(start + q) * H + head * HD + 4 * half;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const float c0 = o[j][4 * g] * inv, c1 = o[j][4 * g + 1] * inv;
                const float c2 = o[j][4 * g + 2] * inv, c3 = o[j][4 * g + 3] * inv;
                *reinterpret_cast<float4*>(ctx_out + at + j * 32 + 8 * g) = make_float4(c0, c1, c2, c3);
            }
    }
}

typedef short v8s_t __attribute__((ext_vector_type(8)));
typedef __bf16 v8bf_t __attribute__((ext_vector_type(8)));

// ---------------------------------------------------------------------------
// bf16 attention for sequences of at most 128 tokens: one key chunk and one
// query block per (head, sequence) workgroup.  Q, K and V go straight from
// HBM into LDS (global_load_lds_dwordx4, no staging registers, no transposing
// copy), so a workgroup needs 48 KB of LDS and at most 110 VGPRs: three
// workgroups per CU, whose load phases overlap each other's MFMAs and
// softmax; within a workgroup the scores wait for Q and K only.
//
// K rows sit unpadded with 16-byte chunk c of row r at c ^ chunk_swizzle16(r)
// (conflict-free fragment reads down 32 rows), as the GEMM tiles do.  V stays
// row-major ([key][dim]): the A operand of O^T = V^T . P^T needs, per lane,
// one dim at 8 keys, which ds_read_b64_tr_b16 delivers.  Within each 16-lane
// group that instruction hands lane i element i % 4 of the 8-byte reads of
// lanes i / 4, 4 + i / 4, 8 + i / 4 and 12 + i / 4; so when lane j of the
// group addresses key k0 + j / 4, dims d0 + 4 (j % 4) .. +3, lane i receives
// dim d0 + i at the four keys k0 .. k0 + 3.  Two such reads give a lane its 8
// keys of one MFMA.  V chunk c of row r sits at c ^ 4 ((r >> 1) & 1) (64-dim
// rows), so the four rows a half-wave reads fall in different banks.
// ---------------------------------------------------------------------------
typedef short v4s_t __attribute__((ext_vector_type(4)));

template <int HD>
__device__ __forceinline__ int v_swizzle(int r) {
    return HD == 64 ? 4 * ((r >> 1) & 1) : 0;
}

template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void attention_bf16_short_kernel(
    const uint16_t* __restrict__ qkv, const int* __restrict__ cu_seqlens, uint16_t* __restrict__ ctx, int H,
    float scale, const int* __restrict__ order) {
    constexpr int KC = 128;                 // keys (and queries) per sequence at most
    constexpr int CPR = HD / 8;             // 16-byte chunks per K / V row
    constexpr int TILE = KC * HD;           // bf16 elements of the K or V tile
    constexpr int NLD = KC * CPR / 256;     // 16-byte loads per thread per tile
    constexpr int NJ = HD / 32;             // 32-wide blocks of the context
    constexpr int NS = HD / 16;             // 16-dim slices of q.k
    __shared__ __attribute__((aligned(16))) uint16_t Ks[TILE];
    __shared__ __attribute__((aligned(16))) uint16_t Vs[TILE];
    __shared__ __attribute__((aligned(16))) uint16_t Qs[TILE];

    const int head = blockIdx.x, b = order ? order[blockIdx.y] : (int)blockIdx.y;
    const int start = cu_seqlens[b];
    const int len = cu_seqlens[b + 1] - start;
    if (len == 0) return;  // uniform over the workgroup
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int l32 = lane & 31, half = lane >> 5;
    const int64_t ld = 3 * (int64_t)H;
    const uint16_t* Qg = qkv + (int64_t)start * ld + head * HD;
    const uint16_t* Kg = Qg + H;
    const uint16_t* Vg = Qg + 2 * H;

    // Q, K and V into LDS, in that order: wave w's load i fills 16-byte slots
    // (4 i + w) * 64 + lane, i.e. row P / CPR, stored chunk P % CPR.  Rows
    // past the sequence re-read its last row (their keys are masked, their V
    // rows meet zero probabilities, their queries are not stored).  The scores
    // wait for Q and K only; V lands while they and the softmax run.
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int P = (i * 4 + wave) * 64 + lane;
        const int r = P / CPR, pc = P % CPR;
        const int64_t row = (int64_t)min(r, len - 1) * ld;
        load_lds16_async(Qg + row + 8 * (pc ^ chunk_swizzle16<CPR>(r)),
                         reinterpret_cast<const float*>(Qs + (i * 4 + wave) * 512));
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int P = (i * 4 + wave) * 64 + lane;
        const int r = P / CPR, pc = P % CPR;
        const int64_t row = (int64_t)min(r, len - 1) * ld;
        load_lds16_async(Kg + row + 8 * (pc ^ chunk_swizzle16<CPR>(r)),
                         reinterpret_cast<const float*>(Ks + (i * 4 + wave) * 512));
    }
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int P = (i * 4 + wave) * 64 + lane;
        const int r = P / CPR, pc = P % CPR;
        const int64_t row = (int64_t)min(r, len - 1) * ld;
        load_lds16_async(Vg + row + 8 * (pc ^ v_swizzle<HD>(r)),
                         reinterpret_cast<const float*>(Vs + (i * 4 + wave) * 512));
    }
    wait_vmcnt(NLD);   // this wave's Q and K loads (its V loads may be in flight)
    __syncthreads();
    // A wave whose 32 queries all lie past the sequence end skips the scores
    // and P.V; it still meets the barrier below.
    const bool active = wave * 32 < len;
    // This lane's query as the B operand: dims 16s + 8*half .. +7.
    const int qr = wave * 32 + l32;
    v8s_t qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
        qf[s] = *reinterpret_cast<const v8s_t*>(Qs + qr * HD + 8 * ((2 * s + half) ^ chunk_swizzle16<CPR>(qr)));

    const int nkb = active ? (len + 31) / 32 : 0;   // 32-key blocks holding real keys
    // S^T = K . Q^T: the four 32-key blocks' MFMA chains side by side.
    v16f sc[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) sc[kb][r] = 0.0f;
#pragma unroll
    for (int s = 0; s < NS; ++s)
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
            if (kb < nkb) {
                const int kr = kb * 32 + l32;
                const v8s_t kf = *reinterpret_cast<const v8s_t*>(
                    Ks + kr * HD + 8 * ((2 * s + half) ^ chunk_swizzle16<CPR>(kr)));
                sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, kf),
                                                                  __builtin_bit_cast(v8bf_t, qf[s]), sc[kb], 0, 0, 0);
            }
    // Row max of the raw scores (scale > 0 commutes with max); keys past the
    // sequence (only in its last block) are masked to -inf (src/lib.rs:887-891).
    float cmax = -INFINITY;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb < nkb) {
            if ((kb + 1) * 32 > len) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (kb * 32 + 8 * (r >> 2) + 4 * half + (r & 3) >= len) sc[kb][r] = -INFINITY;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) cmax = fmaxf(cmax, sc[kb][r]);
        }
    }
    cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
    // p = exp(scale * (s - max)) as exp2(s * c - max * c), c = scale * log2(e):
    // the scale after q.k^T (src/lib.rs:714) folded into one FMA.
    const float c2 = scale * 1.4426950408889634f, off = -cmax * c2;
    float psum = 0.0f;
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb < nkb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pr = __builtin_amdgcn_exp2f(fmaf(sc[kb][r], c2, off));
                sc[kb][r] = pr;
                psum += pr;
            }
        }
    }
    v16f o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[j][r] = 0.0f;
    wait_vmcnt(0);     // this wave's V loads
    __syncthreads();   // and everyone else's
    // context^T += V^T . P^T, two 16-key MFMAs per 32-key block.  Lane half h
    // of the B operand (P) holds keys 16 mm + 4 h + 0..3 and 16 mm + 8 + 4 h +
    // 0..3; the A operand (V^T) gets the same keys at dim l32 from two
    // transposing reads.  16-lane group g reads dims 16 (g % 2) .. +15 of its
    // 32-dim block at keys k0 .. k0 + 3.
    const int g16 = lane >> 4, i16 = lane & 15;
    const int vrow = i16 >> 2, vdim = 16 * (g16 & 1) + 4 * (i16 & 3);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
        if (kb < nkb) {
#pragma unroll
            for (int mm = 0; mm < 2; ++mm) {
                const float* pf = reinterpret_cast<const float*>(&sc[kb]) + 8 * mm;
                const v8s_t pa = __builtin_bit_cast(
                    v8s_t, make_uint4(pack_bf16x2(pf[0], pf[1]), pack_bf16x2(pf[2], pf[3]),
                                      pack_bf16x2(pf[4], pf[5]), pack_bf16x2(pf[6], pf[7])));
                const int k0 = kb * 32 + 16 * mm + 4 * (g16 >> 1);   // this group's first key
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int d = j * 32 + vdim;                     // this lane's 4 dims to address
                    const int ra = k0 + vrow, rb = k0 + 8 + vrow;
                    const v4s_t va = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) v4s_t*)(Vs + ra * HD + 8 * ((d >> 3) ^ v_swizzle<HD>(ra)) + (d & 7)));
                    const v4s_t vb = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (__attribute__((address_space(3))) v4s_t*)(Vs + rb * HD + 8 * ((d >> 3) ^ v_swizzle<HD>(rb)) + (d & 7)));
                    const v8s_t vf = {va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
                    o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, vf),
                                                                    __builtin_bit_cast(v8bf_t, pa), o[j], 0, 0, 0);
                }
            }
        }
    }
    // Lane holds dims j*32 + 8*g + 4*half + 0..3 (g = r / 4) of query l32.
    const float l_tot = psum + __shfl_xor(psum, 32);
    const int q = wave * 32 + l32;
    if (q < len) {
        const float inv = 1.0f / l_tot;
        uint16_t* dst = ctx + (int64_t)(start + q) * H + head * HD + 4 * half;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                *reinterpret_cast<uint2*>(dst + j * 32 + 8 * g) =
                    make_uint2(pack_bf16x2(o[j][4 * g] * inv, o[j][4 * g + 1] * inv),
                               pack_bf16x2(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv));
            }
    }
}

// ---------------------------------------------------------------------------
// bf16 attention of sequences of more than 128 tokens (the kernel above takes
// the shorter ones): Q, K, V, the context and the probabilities bf16, scores,
// softmax and sums fp32.
//
// Work split: workgroup = (head, 128-query block, sequence), 4 waves of 32
// queries.  Softmax is online over 128-key chunks.  K and V go straight into
// LDS (buffer loads; rows past the sequence read as zeros), K in two stages, so
// that chunk c + 1's is on its way while chunk c is computed, V in one: it lands
// while the scores and the softmax run, behind a barrier of its own.  That is
// 48 KB with heads of 64, three workgroups per CU.  A lane's query goes straight
// to registers; layouts, swizzles and the transposing V read are those of the
// kernel above.
//
// What bounds it: the softmax's VALU work, of which the scale, the subtraction
// of the maximum and the factor log2 e are an operation each: folded into one
// FMA, on 64-key chunks, they would be 3 us less (39.9) but other bits.  40
// sequences of 200-512, heads of 64: 66.2 -> 43.2 us (heads of 32: 40.4 -> 31.7)
// against the same sums with both chunks staged through registers and V
// transposed on its way into LDS.
// ---------------------------------------------------------------------------
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3))) void attention_bf16_long_kernel(
    const uint16_t* __restrict__ qkv, const int* __restrict__ cu_seqlens, uint16_t* __restrict__ ctx, int H,
    float scale, const int* __restrict__ order) {
    constexpr int KC = 128, NB = KC / 32;   // keys per chunk, 32-key blocks
    constexpr int RB = 2 * HD;              // bytes per K / V row
    constexpr int CPR = RB / 16;            // 16-byte chunks per K / V row
    constexpr int NLD = KC * CPR / 256;     // 16-byte loads per thread for K (and for V)
    constexpr int NJ = HD / 32, NS = HD / 16;
    __shared__ __attribute__((aligned(16))) char Ks[2][KC * RB];
    __shared__ __attribute__((aligned(16))) char Vs[KC * RB];

    const int head = blockIdx.x, qb = blockIdx.y, b = order ? order[blockIdx.z] : (int)blockIdx.z;
    const int start = cu_seqlens[b];
    const int len = cu_seqlens[b + 1] - start;
    if (qb * 128 >= len) return;  // uniform over the workgroup
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const int64_t ld = 3 * (int64_t)H;
    const uint32_t ldb = 3 * (uint32_t)H * 2;

    uint32_t kvo[NLD], vvo[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int P = i * 256 + tid, r = P / CPR, pc = P % CPR;
        kvo[i] = r * ldb + (H + head * HD) * 2 + 16 * (pc ^ chunk_swizzle16<CPR>(r));
        vvo[i] = r * ldb + (2 * H + head * HD) * 2 + 16 * (pc ^ v_swizzle<HD>(r));
    }
    auto rows_of = [&](int c) __attribute__((always_inline)) {
        return make_rsrc(qkv + (start + c * KC) * ld, (uint32_t)min(len - c * KC, KC) * ldb);
    };
    auto issue_k = [&](int c) __attribute__((always_inline)) {
        const g16_v4i rsrc = rows_of(c);
        const uint32_t ks = (uint32_t)(uintptr_t)&Ks[c & 1][0] + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLD; ++i) load_lds16_buf(rsrc, kvo[i], 0, ks + i * 4096);
    };
    auto issue_v = [&](int c) __attribute__((always_inline)) {
        const g16_v4i rsrc = rows_of(c);
        const uint32_t vs = (uint32_t)(uintptr_t)&Vs[0] + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLD; ++i) load_lds16_buf(rsrc, vvo[i], 0, vs + i * 4096);
    };

    // This lane's query as the B operand: dims 16 s + 8 half .. +7.
    const int q0 = qb * 128 + wave * 32;
    v8s_t qf[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s)
        qf[s] = *reinterpret_cast<const v8s_t*>(qkv + (start + min(q0 + l32, len - 1)) * ld + head * HD + 16 * s + 8 * half);
    issue_k(0);
    issue_v(0);

    v16f o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[j][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    const bool active = q0 < len;   // a wave past the sequence's queries only helps load
    const int g16 = lane >> 4, i16 = lane & 15;
    const int vrow = i16 >> 2, vdim = 16 * (g16 & 1) + 4 * (i16 & 3);
    const int nchunks = (len + KC - 1) / KC;
    for (int c = 0; c < nchunks; ++c) {
        if (c == 0) wait_vmcnt(NLD);   // K is here, V(0) may be in flight
        else wait_vmcnt(0);
        lds_barrier();                 // everyone's K, and everyone is done with chunk c - 1
        if (c > 0) issue_v(c);
        if (c + 1 < nchunks) issue_k(c + 1);
        const int lim = len - c * KC, nkb = active ? min(NB, (lim + 31) / 32) : 0;
        const char* K = Ks[c & 1];
        v16f sc[NB];
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[kb][r] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int kb = 0; kb < NB; ++kb)
                if (kb < nkb) {
                    const int kr = kb * 32 + l32;
                    const v8s_t kf = *reinterpret_cast<const v8s_t*>(K + kr * RB + 16 * ((2 * s + half) ^ chunk_swizzle16<CPR>(kr)));
                    sc[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, kf),
                                                                      __builtin_bit_cast(v8bf_t, qf[s]), sc[kb], 0, 0, 0);
                }
        // The scale after q.k^T (src/lib.rs:714), rounded by itself, and the
        // key-padding mask (src/lib.rs:887-891).
        float cmax = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) sc[kb][r] *= scale;
                if ((kb + 1) * 32 > lim) {             // the block that straddles the sequence end
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (kb * 32 + 8 * (r >> 2) + (r & 3) >= lim - 4 * half) sc[kb][r] = -INFINITY;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) cmax = fmaxf(cmax, sc[kb][r]);
            }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
        const float m_new = fmaxf(m_run, cmax);
        const float alpha = fast_exp(m_run - m_new);   // 0 on the first chunk
        float psum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float pr = fast_exp(sc[kb][r] - m_new);
                    sc[kb][r] = pr;
                    psum += pr;
                }
            }
        l_run = l_run * alpha + psum;
        m_run = m_new;
        if (c > 0) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[j][r] *= alpha;
        }
        if (c + 1 < nchunks) wait_vmcnt(NLD);          // V is here, K(c + 1) may be in flight
        else wait_vmcnt(0);
        lds_barrier();                                 // and everyone else's
        // context^T += V^T . P^T, 16 keys a step, as in the kernel above.
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
#pragma unroll
                for (int mm = 0; mm < 2; ++mm) {
                    const float* pf = reinterpret_cast<const float*>(&sc[kb]) + 8 * mm;
                    const v8s_t pa = __builtin_bit_cast(
                        v8s_t, make_uint4(pack_bf16x2(pf[0], pf[1]), pack_bf16x2(pf[2], pf[3]),
                                          pack_bf16x2(pf[4], pf[5]), pack_bf16x2(pf[6], pf[7])));
                    const int ra = kb * 32 + 16 * mm + 4 * (g16 >> 1) + vrow, rb = ra + 8;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const int d = j * 32 + vdim;
                        auto rd = [&](int r) __attribute__((always_inline)) {
                            return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                (__attribute__((address_space(3))) v4s_t*)(Vs + r * RB + 16 * ((d >> 3) ^ v_swizzle<HD>(r)) + 2 * (d & 7)));
                        };
                        const v4s_t va = rd(ra), vb = rd(rb);
                        const v8s_t vf = {va[0], va[1], va[2], va[3], vb[0], vb[1], vb[2], vb[3]};
                        o[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf_t, vf),
                                                                        __builtin_bit_cast(v8bf_t, pa), o[j], 0, 0, 0);
                    }
                }
            }
    }

    // Lane holds dims j*32 + 8*g + 4*half + 0..3 (g = r / 4) of query l32.
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const int q = q0 + l32;
    if (q < len) {
        const float inv = 1.0f / l_tot;
        uint16_t* dst = ctx + (int64_t)(start + q) * H + head * HD + 4 * half;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<uint2*>(dst + j * 32 + 8 * g) =
                    make_uint2(pack_bf16x2(o[j][4 * g] * inv, o[j][4 * g + 1] * inv),
                               pack_bf16x2(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv));
    }
}

// ---------------------------------------------------------------------------
// Attention on fp16 pairs, for any length: the fp32 forward above 64 tokens.
// Q, K, V and the context are in the pair format (gemm16.hpp; a head's row is
// 4 HD bytes, as in fp32), every product from three v_mfma_f32_32x32x16_f16
// with fp32 sums.
//
// Work split: workgroup = (head, 128-query block, sequence), 4 waves of 32
// queries; 64-key chunks of K and V in two LDS stages, chunk c + 1 on its way
// (direct-to-LDS buffer loads; rows past the sequence read as zeros) while
// chunk c is computed.  A lane's query goes straight to registers.
//
// The layouts are those of the kernels above: S^T = K . Q^T, so a lane owns one
// query's scores; the probabilities (scaled by 2^12 in the exponent, so that l
// of small ones stays out of fp16's subnormals, and split in registers)
// are the B operand of O^T = V^T . P^T, whose A operand comes from row-major V
// through ds_read_b64_tr_b16.  K chunks are swizzled as GEMM rows are.  A
// half-wave's transposing read takes the h (or l) chunks, every other 16 bytes,
// of four rows; V's swizzle moves rows that share banks (r and r + 2 of 128-byte
// rows, all four of 256-byte ones) apart.
//
// What bounds it: HBM at c3 (201 MB a layer), the softmax's VALU work (the
// split of P included, it outweighs the twelve MFMAs per 32 x 32 block) on long
// sequences.  Unlike fp32 MFMAs, fp16 ones leave the VALU free meanwhile.
// Against the fp32 kernel above, in the forward, per layer: 256 sequences of
// 128 tokens 76 -> 47 us (4.3 TB/s), 16 of 256-512 53 -> 26 us, 32 of 8-128
// 12.4 -> 8.3 us; heads of 64, 48 of 16-128 24.9 -> 15.2 us.
// ---------------------------------------------------------------------------
template <int HD>
__device__ __forceinline__ int v_pair_swizzle(int r) {
    return HD == 32 ? ((r >> 1) & 1) : (r & 1) | ((r >> 1) & 1) << 3;
}

template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HD == 32 ? 4 : 2))) void attention_stream_kernel(
    const uint32_t* __restrict__ qkv_, const int* __restrict__ cu_seqlens, uint32_t* __restrict__ ctx_, int H, float c2,
    float out_mul, const int* __restrict__ order) {
    constexpr int KC = 64, NB = KC / 32;    // keys per chunk, 32-key blocks
    constexpr int ES = 4;                   // bytes per element
    constexpr int RB = ES * HD;             // bytes per K / V row
    constexpr int CPR = RB / 16;            // 16-byte chunks per K / V row
    const char* qkv = reinterpret_cast<const char*>(qkv_);
    constexpr int NLD = KC * CPR / 256;     // 16-byte loads per thread for K (and for V)
    constexpr int NJ = HD / 32, NS = HD / 16;
    constexpr float P_LOG2 = 12.0f;         // probabilities are held times 2^12
    __shared__ __attribute__((aligned(16))) char Ks[2][KC * RB];
    __shared__ __attribute__((aligned(16))) char Vs[2][KC * RB];

    const int head = blockIdx.x, qb = blockIdx.y, b = order ? order[blockIdx.z] : (int)blockIdx.z;
    const int start = cu_seqlens[b];
    const int len = cu_seqlens[b + 1] - start;
    if (qb * 128 >= len) return;  // uniform over the workgroup
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l32 = lane & 31, half = lane >> 5;
    const uint32_t ldb = 3 * (uint32_t)H * ES;

    uint32_t kvo[NLD], vvo[NLD];
#pragma unroll
    for (int i = 0; i < NLD; ++i) {
        const int P = i * 256 + tid, r = P / CPR, pc = P % CPR;
        kvo[i] = r * ldb + (H + head * HD) * ES + 16 * (pc ^ chunk_swizzle16<CPR>(r));
        vvo[i] = r * ldb + (2 * H + head * HD) * ES + 16 * (pc ^ v_pair_swizzle<HD>(r));
    }
    auto issue = [&](int c) __attribute__((always_inline)) {
        const g16_v4i rsrc = make_rsrc(qkv + (int64_t)(start + c * KC) * ldb, (uint32_t)min(len - c * KC, KC) * ldb);
        const uint32_t ks = (uint32_t)(uintptr_t)&Ks[c & 1][0] + wave * 1024, vs = (uint32_t)(uintptr_t)&Vs[c & 1][0] + wave * 1024;
#pragma unroll
        for (int i = 0; i < NLD; ++i) load_lds16_buf(rsrc, kvo[i], 0, ks + i * 4096);
#pragma unroll
        for (int i = 0; i < NLD; ++i) load_lds16_buf(rsrc, vvo[i], 0, vs + i * 4096);
    };

    // One 32 x 32 x 16 product step of (h, l) operands.
    auto mul = [](const v8h& ah, const v8h& al, const v8h& bh, const v8h& bl, v16f d) __attribute__((always_inline)) {
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, d, 0, 0, 0);
        d = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, d, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, d, 0, 0, 0);
    };
    // This lane's query: dims 16 s + 8 half .. +7 (h and l).
    const int q0 = qb * 128 + wave * 32;
    v8h qh[NS], ql[NS];
    {
        const char* qr = qkv + (int64_t)(start + min(q0 + l32, len - 1)) * ldb + (head * HD + 8 * half) * ES;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            qh[s] = *reinterpret_cast<const v8h*>(qr + 16 * ES * s);
            ql[s] = *reinterpret_cast<const v8h*>(qr + 16 * ES * s + 16);
        }
    }
    issue(0);

    v16f o[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[j][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    const bool active = q0 < len;   // a wave past the sequence's queries only helps load
    const int g16 = lane >> 4, i16 = lane & 15;
    const int vrow = i16 >> 2, vdim = 16 * (g16 & 1) + 4 * (i16 & 3);
    const int nchunks = (len + KC - 1) / KC;
    for (int c = 0; c < nchunks; ++c) {
        wait_vmcnt(0);
        lds_barrier();   // chunk c is here, and everyone is done with chunk c - 1
        if (c + 1 < nchunks) issue(c + 1);
        if (!active) continue;
        const char *K = Ks[c & 1], *V = Vs[c & 1];
        const int lim = len - c * KC, nkb = min(NB, (lim + 31) / 32);
        v16f sc[NB];
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) sc[kb][r] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int kb = 0; kb < NB; ++kb)
                if (kb < nkb) {
                    const int kr = kb * 32 + l32, ch = (2 * (2 * s + half)) ^ chunk_swizzle16<CPR>(kr);
                    const v8h kh = *reinterpret_cast<const v8h*>(K + kr * RB + 16 * ch);
                    const v8h kl = *reinterpret_cast<const v8h*>(K + kr * RB + 16 * (ch ^ 1));
                    sc[kb] = mul(kh, kl, qh[s], ql[s], sc[kb]);
                }
        // Key-padding mask (src/lib.rs:887-891), only in the block that
        // straddles the sequence end; the max is taken over the raw scores.
        float cmax = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
                if ((kb + 1) * 32 > lim) {
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (kb * 32 + 8 * (r >> 2) + 4 * half + (r & 3) >= lim) sc[kb][r] = -INFINITY;
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) cmax = fmaxf(cmax, sc[kb][r]);
            }
        cmax = fmaxf(cmax, __shfl_xor(cmax, 32));
        // exp(scale (s - m)) as 2^(s c2 - m c2), times 2^12; c2 holds the scale,
        // log2 e and the operands' scales.
        const float m_new = fmaxf(m_run, cmax), mc = m_new * c2, off = P_LOG2 - mc;
        const float alpha = __builtin_amdgcn_exp2f(m_run * c2 - mc);   // 0 on the first chunk
        float ps[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const float pr = __builtin_amdgcn_exp2f(fmaf(sc[kb][r], c2, off));
                    sc[kb][r] = pr;
                    ps[r & 3] += pr;
                }
            }
        l_run = l_run * alpha + ((ps[0] + ps[1]) + (ps[2] + ps[3]));
        m_run = m_new;
        if (c > 0) {
#pragma unroll
            for (int j = 0; j < NJ; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[j][r] *= alpha;
        }
        // context^T += V^T . P^T, 16 keys a step: lane half h of P holds keys
        // 16 mm + 4 h + 0..3 and 16 mm + 8 + 4 h + 0..3.
#pragma unroll
        for (int kb = 0; kb < NB; ++kb)
            if (kb < nkb) {
#pragma unroll
                for (int mm = 0; mm < 2; ++mm) {
                    uint32_t hw[4], lw[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float p0 = sc[kb][8 * mm + 2 * e], p1 = sc[kb][8 * mm + 2 * e + 1];
                        split_f16x2(p0, p1, hw[e], lw[e]);
                    }
                    const v8h ph = __builtin_bit_cast(v8h, make_uint4(hw[0], hw[1], hw[2], hw[3]));
                    const v8h pl = __builtin_bit_cast(v8h, make_uint4(lw[0], lw[1], lw[2], lw[3]));
                    const int ra = kb * 32 + 16 * mm + 4 * (g16 >> 1) + vrow, rb = ra + 8;
#pragma unroll
                    for (int j = 0; j < NJ; ++j) {
                        const int d = j * 32 + vdim, ch = 2 * (d >> 3), in = 2 * (d & 7);
                        auto rd = [&](int r, int part) __attribute__((always_inline)) {
                            return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                (__attribute__((address_space(3))) v4s_t*)(V + r * RB + 16 * ((ch + part) ^ v_pair_swizzle<HD>(r)) + in));
                        };
                        const v4s_t ha = rd(ra, 0), hb = rd(rb, 0);
                        const v8h vh = __builtin_bit_cast(v8h, (v8s_t){ha[0], ha[1], ha[2], ha[3], hb[0], hb[1], hb[2], hb[3]});
                        const v4s_t la = rd(ra, 1), lb = rd(rb, 1);
                        const v8h vl = __builtin_bit_cast(v8h, (v8s_t){la[0], la[1], la[2], la[3], lb[0], lb[1], lb[2], lb[3]});
                        o[j] = mul(vh, vl, ph, pl, o[j]);
                    }
                }
            }
    }

    // Lane holds dims j*32 + 8*g + 4*half + 0..3 (g = r / 4) of query l32.
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    const int q = q0 + l32;
    if (q < len) {
        const float inv = out_mul / l_tot;   // ctx scale / qkv scale; the 2^12 cancels
        char* dst = reinterpret_cast<char*>(ctx_) + ((int64_t)(start + q) * H + head * HD) * ES + 8 * half;
#pragma unroll
        for (int j = 0; j < NJ; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                uint2 h, l;
                split_f16x2(o[j][4 * g] * inv, o[j][4 * g + 1] * inv, h.x, l.x);
                split_f16x2(o[j][4 * g + 2] * inv, o[j][4 * g + 3] * inv, h.y, l.y);
                *reinterpret_cast<uint2*>(dst + 128 * j + 32 * g) = h;
                *reinterpret_cast<uint2*>(dst + 128 * j + 32 * g + 16) = l;
            }
    }
}

hipError_t launch_attention_pair(const uint32_t* qkv, const int* cu_seqlens, int B, int max_len, int H, int nh,
                                 int head_dim, float scale, float qkv_scale, uint32_t* ctx, float ctx_scale,
                                 hipStream_t s, const int* order) {
    if (B <= 0 || max_len <= 0) return hipSuccess;
    const dim3 grid(nh, (max_len + 127) / 128, B), block(256);
    const float c2 = scale * 1.4426950408889634f / (qkv_scale * qkv_scale), mul = ctx_scale / qkv_scale;
    if (head_dim == 32)
        hipLaunchKernelGGL((attention_stream_kernel<32>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, c2, mul, order);
    else if (head_dim == 64)
        hipLaunchKernelGGL((attention_stream_kernel<64>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, c2, mul, order);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_attention_bf16(const uint16_t* qkv, const int* cu_seqlens, int B, int max_len,
                                 int H, int nh, int head_dim, float scale, uint16_t* ctx,
                                 hipStream_t s, const int* order) {
    if (B <= 0 || max_len <= 0) return hipSuccess;
    if (max_len <= 128) {
        // One key chunk per sequence: K and V straight into LDS, three
        // workgroups per CU.
        const dim3 grid(nh, B), block(256);
        if (head_dim == 32)
            hipLaunchKernelGGL(attention_bf16_short_kernel<32>, grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
        else if (head_dim == 64)
            hipLaunchKernelGGL(attention_bf16_short_kernel<64>, grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
        else
            return hipErrorInvalidValue;
        return hipGetLastError();
    }
    const dim3 grid(nh, (max_len + 127) / 128, B), block(256);
    if (head_dim == 32)
        hipLaunchKernelGGL(attention_bf16_long_kernel<32>, grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else if (head_dim == 64)
        hipLaunchKernelGGL(attention_bf16_long_kernel<64>, grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

hipError_t launch_attention(const float* qkv, const int* cu_seqlens, int B, int max_len, int H,
                            int nh, int head_dim, float scale, float* ctx, hipStream_t s, const int* order) {
    if (B <= 0 || max_len <= 0) return hipSuccess;
    const dim3 grid(nh, (max_len + 127) / 128, B), block(256);
    const bool short_seqs = max_len <= 128;
    if (head_dim == 32 && short_seqs)
        hipLaunchKernelGGL((attention_kernel<32, 64>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else if (head_dim == 32)
        hipLaunchKernelGGL((attention_kernel<32, 128>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else if (head_dim == 64 && short_seqs)
        hipLaunchKernelGGL((attention_kernel<64, 64>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else if (head_dim == 64)
        hipLaunchKernelGGL((attention_kernel<64, 128>), grid, block, 0, s, qkv, cu_seqlens, ctx, H, scale, order);
    else
        return hipErrorInvalidValue;
    return hipGetLastError();
}

}  // namespace ebh
