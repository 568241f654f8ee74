"""fp32 products from fp16 pairs, with and without the weights' rest
(ebh_op_to_pair, ebh_op_gemm_pair and their _rest forms), against float64 on every
tile, at tile edges and remainders and over several tiles a workgroup; bf16
products at the sizes between which their tile changes, bit for bit against the
ring kernel's; which products a model takes for a batch's shape; and models whose
weights lie at the ends of the range the pair operands' scales are taken from, or
outside it (those keep the fp32 kernels), against the CPU oracle."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EPI_BIAS, EPI_GELU, EPI_NONE = 0, 1, 3


@pytest.fixture(scope="module")
def env():
    import torch
    import edgebert_amd as eb
    from edgebert_amd import _native as N
    assert torch.cuda.is_available(), "gpu tests need a GPU"
    return torch, eb, N, eb.lib()


def vp(t):
    return ctypes.c_void_p(t.data_ptr())


def to_pair(torch, N, L, x, scale, s):
    y = torch.empty_like(x)
    N.check(L.ebh_op_to_pair(vp(x), vp(y), x.numel(), scale, s))
    return y


def to_pair_rest(torch, N, L, w, scale, s):
    y = torch.empty(w.shape[0], w.shape[1] * 3 // 2, device="cuda")
    N.check(L.ebh_op_to_pair_rest(vp(w), vp(y), w.shape[0], w.shape[1], scale, s))
    return y


def unpair(torch, y, scale):
    h = y.view(torch.float16).view(y.shape[0], -1, 2, 8).double()
    return ((h[:, :, 0] + h[:, :, 1]) / scale).reshape(y.shape[0], -1)


def test_to_pair_keeps_23_bits(env):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    x = torch.randn(64, 264, device="cuda")
    scale = 2.0 ** 12
    got = unpair(torch, to_pair(torch, N, L, x, scale, s), scale)
    # l is rounded to 11 bits of at most half a unit of h's 11: 2^-23 of |x|,
    # or half of fp16's smallest step where l is subnormal
    bound = np.maximum(2.0 ** -23 * x.abs().double().cpu().numpy(), 2.0 ** -25 / scale)
    assert (np.abs((got - x.double()).cpu().numpy()) <= bound).all()
    assert L.ebh_op_to_pair(vp(x), vp(x), 12, scale, s) == N.EBH_ERR_INVALID_ARG


# rows below, at and just over every tile height; columns that are not whole
# tiles; one, two and several k-tile pairs; splits
SHAPES = [(1, 64, 64, 1), (63, 96, 128, 2), (65, 200, 192, 3), (129, 392, 384, 1), (257, 1152, 384, 2),
          (300, 1536, 384, 1), (513, 384, 1536, 4), (1000, 264, 448, 1)]


@pytest.mark.parametrize("tile", range(-1, 8))
@pytest.mark.parametrize("M,Nn,K,S", SHAPES)
def test_gemm_pair(env, M, Nn, K, S, tile):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(M + Nn + K)
    lda, ldc = K + 8, Nn + 16
    A = torch.randn(M, lda, device="cuda", generator=g)
    A[:, 3] *= 30                                  # an outlier feature
    W = 0.04 * torch.randn(Nn, K, device="cuda", generator=g)
    b = torch.randn(Nn, device="cuda", generator=g)
    sa, sw, sc = 2.0 ** 8, 2.0 ** 14, 2.0 ** 4
    Ap, Wp = to_pair(torch, N, L, A, sa, s), to_pair(torch, N, L, W, sw, s)
    Ad, Wd = A[:, :K].double(), W.double()
    ref = Ad @ Wd.t()
    # operands 2^-23 each, al.bl 2^-24, and 3 K / 32 sums each rounded (down)
    # a few times within 2^-22 of the terms' size
    tol = (2.0 ** -21 + 3 * K / 32 * 2.0 ** -22) * (Ad.abs() @ Wd.abs().t())

    def run(epi, C, c_scale, bias, splits=1, stride=0):
        N.check(L.ebh_op_gemm_pair(vp(Ap), lda, vp(Wp), K, 1 / (sa * sw), bias, vp(C), ldc, c_scale, M, Nn, K, epi,
                                   splits, stride, tile, s))
        torch.cuda.synchronize()

    def padding_kept(D):
        return (D[M:] == 7).all() and (D[:M, Nn:] == 7).all()

    C = torch.full((M + 2, ldc), 7.0, device="cuda")
    run(EPI_BIAS, C, sc, vp(b))
    got = unpair(torch, C[:M], sc)[:, :Nn]
    u = ref + b.double()
    assert ((got - u).abs() <= tol + 2.0 ** -22 * (ref.abs() + b.abs().double()) + 2.0 ** -25 / sc).all()
    assert padding_kept(C)
    if tile > 0:      # every tile sums in the same order
        C0 = torch.full((M + 2, ldc), 7.0, device="cuda")
        N.check(L.ebh_op_gemm_pair(vp(Ap), lda, vp(Wp), K, 1 / (sa * sw), vp(b), vp(C0), ldc, sc, M, Nn, K, EPI_BIAS,
                                   1, 0, 0, s))
        torch.cuda.synchronize()
        assert torch.equal(C0.view(torch.int32), C.view(torch.int32))
    stride = (M + 1) * ldc
    P = torch.full((S * stride,), 7.0, device="cuda")
    if K % (64 * S) == 0:
        run(EPI_NONE, P, 0.0, None, S, stride)
        got = sum(P[i * stride:i * stride + M * ldc].view(M, ldc)[:, :Nn].double() for i in range(S))
        assert ((got - ref).abs() <= tol + 2.0 ** -23 * ref.abs() * S).all()
    D = torch.full((M + 2, ldc), 7.0, device="cuda")
    run(EPI_GELU, D, sc, vp(b))
    want = 0.5 * u * (1 + torch.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3)))
    got = unpair(torch, D[:M], sc)[:, :Nn]
    # GELU's slope is below 1.13; its own error (8 ln2 |t| + 8) 2^-24 |gelu|
    gtol = 1.13 * (tol + 2.0 ** -23 * u.abs()) + (2.0 ** -22 + 2.0 ** -20) * want.abs() + 2.0 ** -25 / sc
    assert ((got - want).abs() <= gtol + 1e-6 * (u < -4)).all()
    assert padding_kept(D)


# K: two, three and twelve pairs of the rest's k-tiles, split and not
@pytest.mark.parametrize("K,S", [(128, 1), (256, 2), (384, 1), (384, 3), (1536, 4)])
def test_rest_makes_weights_exact(env, K, S):
    """Rows of the identity pick out the weights: with the rest every one of them
    comes back as it is, at every k, on every tile; without it, a quarter do not."""
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(K)
    W = 0.04 * torch.randn(200, K, device="cuda", generator=g)
    sw = 2.0 ** 16
    A = to_pair(torch, N, L, torch.eye(K, device="cuda"), 1.0, s)
    Wr = to_pair_rest(torch, N, L, W, sw, s)
    halves = Wr[:, K:].contiguous().view(torch.float16).double()
    # below 1/2 (scaled) a value's 24th bit is less than fp16's smallest step, 2^-24
    exact = W.abs() * sw >= 0.5
    assert exact.float().mean().item() > 0.999
    assert torch.equal((unpair(torch, Wr[:, :K].contiguous(), sw) + halves / sw)[exact], W.double()[exact])

    def product(f, W, ldw, tile):
        C = torch.empty(S, K, 200, device="cuda")
        N.check(f(vp(A), K, vp(W), ldw, 1 / sw, None, vp(C), 200, 0.0, K, 200, K, EPI_NONE, S, K * 200, tile, s))
        return C.sum(0).t()            # one split holds the value, the others zeros

    for tile in range(-1, 8):
        assert torch.equal(product(L.ebh_op_gemm_pair_rest, Wr, K * 3 // 2, tile)[exact], W[exact])
    off = product(L.ebh_op_gemm_pair, Wr, K * 3 // 2, -1) != W
    assert 0.2 < off.float().mean().item() < 0.3
    assert L.ebh_op_gemm_pair_rest(vp(A), K, vp(Wr), K, 1 / sw, None, vp(Wr), 200, 0.0, K, 200, K, EPI_NONE, 1, 0, -1,
                                   s) == N.EBH_ERR_INVALID_ARG      # rows without room for the rest
    assert L.ebh_op_gemm_pair_rest(vp(A), K, vp(Wr), K * 3 // 2, 1 / sw, None, vp(Wr), 200, 0.0, K, 200, 64, EPI_NONE, 1,
                                   0, -1, s) == N.EBH_ERR_INVALID_ARG


def test_products_by_length_and_depth(env, weights_for):
    """Where fp32 models take pairs, pairs with the rest and fp32 MFMA products."""
    torch, eb, N, L = env
    mfma, pair, rest = 0, 1, 2
    wide = dict(vocab_size=50, max_position_embeddings=512, layer_norm_eps=1e-12)
    deep = eb.BertConfig(hidden_size=128, num_attention_heads=4, num_hidden_layers=12, intermediate_size=256, **wide)
    narrow = eb.BertConfig(hidden_size=64, num_attention_heads=2, num_hidden_layers=2, intermediate_size=256, **wide)
    for cfg, want in ((eb.MINILM_L6, {(1, 64): mfma, (1, 65): pair, (300, 128): pair, (1, 129): rest, (8, 512): rest}),
                      (narrow, {(30, 128): pair, (30, 129): mfma}),       # K = 64: no rest
                      (deep, {(2, 64): pair, (2, 65): rest, (2, 192): rest, (2, 193): mfma, (1, 64): mfma})):
        m = eb.Model.from_weights(weights_for(cfg), cfg, "fp32")
        try:
            got = {k: L.ebh_op_products(m._h, *k) for k in want}
        finally:
            m.close()
        assert got == want


# at least three items for every workgroup on every tile, in whole rounds of
# 256 x 256 tiles and not, rows and columns ending inside a tile; tiles of two
# k-tiles, of four and of more.  The columns of a workgroup's items differ, and so
# do their biases.
@pytest.mark.parametrize("M,Nn", [(8187, 6136), (8450, 6392)])
@pytest.mark.parametrize("K,S,rest", [(64, 1, False), (128, 2, False), (384, 3, False), (128, 1, True), (384, 3, True)])
def test_gemm_pair_many_tiles(env, M, Nn, K, S, rest):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(M + K)
    A, W = torch.randn(M, K, device="cuda", generator=g), 0.04 * torch.randn(Nn, K, device="cuda", generator=g)
    b = 3 * torch.randn(Nn, device="cuda", generator=g)
    sa, sw, sc = 2.0 ** 8, 2.0 ** 14, 2.0 ** 4
    Ap, Wp = to_pair(torch, N, L, A, sa, s), (to_pair_rest if rest else to_pair)(torch, N, L, W, sw, s)
    product = L.ebh_op_gemm_pair_rest if rest else L.ebh_op_gemm_pair

    def run(tile, epi, splits=1):
        C = torch.empty(splits, M, Nn, device="cuda")
        N.check(product(vp(Ap), K, vp(Wp), Wp.shape[1], 1 / (sa * sw), vp(b) if epi != EPI_NONE else None, vp(C), Nn,
                        sc if epi != EPI_NONE else 0.0, M, Nn, K, epi, splits, M * Nn, tile, s))
        return C

    ref = A.double() @ W.double().t()
    tol = (2.0 ** -21 + 3 * K / 32 * 2.0 ** -22) * (A.abs().double() @ W.abs().double().t())   # as in test_gemm_pair
    for epi, splits in ((EPI_BIAS, 1), (EPI_GELU, 1), (EPI_NONE, S)):
        first = run(0, epi, splits)
        if epi == EPI_BIAS:
            u = ref + b.double()
            assert ((unpair(torch, first[0], sc) - u).abs() <= tol + 2.0 ** -22 * (ref.abs() + b.abs().double()) + 2.0 ** -25 / sc).all()
        elif epi == EPI_NONE:
            assert ((first.double().sum(0) - ref).abs() <= tol + 2.0 ** -23 * ref.abs() * S).all()
        for tile in range(1, 8):
            for _ in range(2):
                assert torch.equal(run(tile, epi, splits).view(torch.int32), first.view(torch.int32)), (tile, epi)


@pytest.mark.parametrize("M,I,S", [(1, 128, 1), (127, 256, 2), (129, 384, 1), (300, 1536, 3), (1000, 1536, 12), (2600, 1536, 1)])
def test_ffn_pair(env, M, I, S):
    """Against float64, and bit for bit against the two products that it stands
    for (the same fragments in the same order), split by split."""
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(M + I)
    X = torch.randn(M, 384, device="cuda", generator=g)
    W1 = 0.04 * torch.randn(I, 384, device="cuda", generator=g)
    W2 = 0.04 * torch.randn(384, I, device="cuda", generator=g)
    b1 = 0.1 * torch.randn(I, device="cuda", generator=g)
    sx, sw, sg = 2.0 ** 9, 2.0 ** 15, 2.0 ** 10
    Xp, W1p, W2p = (to_pair(torch, N, L, t, sc, s) for t, sc in ((X, sx), (W1, sw), (W2, sw)))
    stride = M * 384 + 64
    Y = torch.full((S * stride,), 7.0, device="cuda")
    N.check(L.ebh_op_ffn_pair(vp(Xp), vp(W1p), vp(b1), vp(W2p), 1 / (sx * sw), sg, 1 / (sg * sw), vp(Y), M, I, S, stride, s))
    F = torch.empty(M, I, device="cuda")
    N.check(L.ebh_op_gemm_pair(vp(Xp), 384, vp(W1p), 384, 1 / (sx * sw), vp(b1), vp(F), I, sg, M, I, 384, EPI_GELU, 1, 0, -1, s))
    P = torch.full((S * stride,), 7.0, device="cuda")
    N.check(L.ebh_op_gemm_pair(vp(F), I, vp(W2p), I, 1 / (sg * sw), None, vp(P), 384, 0.0, M, 384, I, EPI_NONE, S, stride, -1, s))
    torch.cuda.synchronize()
    assert torch.equal(Y, P)
    u = X.double() @ W1.double().t() + b1.double()
    f = 0.5 * u * (1 + torch.tanh(0.7978845608028654 * (u + 0.044715 * u ** 3)))
    want = f @ W2.double().t()
    got = sum(Y[i * stride:i * stride + M * 384].view(M, 384).double() for i in range(S))
    assert ((got - want).norm() / want.norm()).item() <= 8e-7     # an fp32 MFMA chain over 1,536 is at 7e-7
    bad = N.EBH_ERR_INVALID_ARG
    args = (1 / (sx * sw), sg, 1 / (sg * sw), vp(Y), M)
    assert L.ebh_op_ffn_pair(vp(Xp), vp(W1p), vp(b1), vp(W2p), *args, I, 5, stride, s) == bad
    assert L.ebh_op_ffn_pair(vp(Xp), vp(W1p), vp(b1), vp(W2p), *args, I + 64, 1, stride, s) == bad


def test_gemm_pair_refuses(env):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    t = torch.zeros(1 << 16, device="cuda")

    def call(M=8, Nn=64, K=64, epi=EPI_NONE, c_scale=0.0, splits=1, tile=-1, ldc=64, bias=None, A=None):
        return L.ebh_op_gemm_pair(A or vp(t), K, vp(t), K, 1.0, bias, vp(t), ldc, c_scale, M, Nn, K, epi, splits, 64 * 8,
                                  tile, s)

    bad = N.EBH_ERR_INVALID_ARG
    assert call(K=96) == bad and call(Nn=60) == bad and call(ldc=60) == bad and call(tile=8) == bad
    assert call(epi=EPI_GELU) == bad and call(c_scale=2.0) == bad and call(splits=2) == bad
    assert call(epi=EPI_BIAS, c_scale=2.0) == bad          # no bias
    assert call(A=ctypes.c_void_p(t.data_ptr() + 4)) == bad
    assert call(M=0) == N.EBH_OK and call() == N.EBH_OK
    torch.cuda.synchronize()


# the dispatch takes 64x64, 64x128, 128x96, 128x128 and 256x192 tiles and the
# ring kernel over these sizes; rows and columns end inside a tile
@pytest.mark.parametrize("M,Nn,K", [(1, 64, 128), (65, 264, 256), (130, 768, 3072), (1300, 2304, 768), (2050, 3072, 768),
                                    (4353, 768, 3072), (8200, 1544, 384), (8191, 3072, 768), (20481, 2304, 768)])
@pytest.mark.parametrize("epi", [EPI_BIAS, EPI_GELU, EPI_NONE])
def test_gemm_bf16_tiles(env, M, Nn, K, epi):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(M + Nn + K)
    A = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    W = (0.04 * torch.randn(Nn, K, device="cuda", generator=g)).bfloat16()
    b = torch.randn(Nn, device="cuda", generator=g)
    C = torch.full((M + 1, Nn), 7.0, device="cuda", dtype=torch.bfloat16)
    N.check(L.ebh_op_gemm_bf16(vp(A), K, vp(W), K, vp(b) if epi != EPI_NONE else None, vp(C), Nn, N.EBH_DTYPE_BF16, M,
                               Nn, K, epi, s))
    torch.cuda.synchronize()
    u = A.float() @ W.float().t() + (b if epi != EPI_NONE else 0.0)    # 24-bit sums of exact products
    want = torch.nn.functional.gelu(u, approximate="tanh") if epi == EPI_GELU else u
    # the result rounded to bf16, and two differently ordered fp32 sums
    tol = 2.0 ** -8 * want.abs() + 4e-6 * np.sqrt(K) + 1e-6
    assert ((C[:M].float() - want).abs() <= tol).all()
    assert (C[M:] == 7).all()


# M: rows of the one call that the ring kernel takes; fewer rows take the smaller
# tiles in turn (64x64, 64x128, 128x96, 128x128, 256x128, 256x192)
@pytest.mark.parametrize("M,Nn,K", [(20481, 2304, 768), (20481, 768, 3072), (20481, 3072, 768), (33000, 192, 128),
                                    (20481, 1544, 384)])
@pytest.mark.parametrize("epi", [EPI_BIAS, EPI_GELU, EPI_NONE])
def test_bf16_rows_do_not_depend_on_the_batch(env, M, Nn, K, epi):
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(Nn + K)
    A = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    W = (0.04 * torch.randn(Nn, K, device="cuda", generator=g)).bfloat16()
    b = torch.randn(Nn, device="cuda", generator=g)

    def product(m):
        C = torch.empty(m, Nn, device="cuda", dtype=torch.bfloat16)
        N.check(L.ebh_op_gemm_bf16(vp(A), K, vp(W), K, vp(b) if epi != EPI_NONE else None, vp(C), Nn, N.EBH_DTYPE_BF16, m,
                                   Nn, K, epi, s))
        return C.view(torch.int16)

    want = product(M)
    for m in (1, 65, 1300, 2050, 4353, 8191, 12000):
        assert torch.equal(product(m), want[:m]), m


@pytest.mark.parametrize("H,nh", [(384, 12), (768, 12), (64, 1)])
@pytest.mark.parametrize("lens", [[1], [31, 32, 33, 0, 64, 65], [127, 128, 129, 7], [192, 193, 512, 300]])
def test_attention_pair(env, H, nh, lens):
    """Against float64, every length around the 32-key blocks, 64-key chunks and
    128-query blocks; rows past the last sequence stay untouched."""
    torch, eb, N, L = env
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda").manual_seed(sum(lens) + H)
    T, hd = sum(lens), H // nh
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32, device="cuda")
    qkv = torch.randn(T, 3 * H, device="cuda", generator=g)
    qkv[:, :H] *= 2.0                                # peaked rows too
    sq, sc = 2.0 ** 9, 2.0 ** 10
    pairs = to_pair(torch, N, L, qkv, sq, s)
    ctx = torch.full((T + 3, H), 7.0, device="cuda")
    N.check(L.ebh_op_attention_pair(vp(pairs), sq, vp(cu), len(lens), max(lens), H, nh, vp(ctx), sc, s))
    torch.cuda.synchronize()
    got = unpair(torch, ctx[:T], sc)
    at = 0
    for n in lens:
        x = qkv[at:at + n].double().view(n, 3, nh, hd).permute(1, 2, 0, 3).contiguous()
        score = torch.matmul(x[0], x[1].transpose(1, 2).contiguous()) / np.sqrt(hd)
        p = torch.softmax(score, -1)
        want = torch.matmul(p, x[2]).transpose(0, 1).reshape(n, H)
        # a score is off by its products' 2^-21 |q||k| sum and the exponent's
        # few 2^-24 |s c|; that moves a probability by as much, relatively; the
        # products with V and their split add 2^-21
        big = (torch.matmul(x[0].abs(), x[1].abs().transpose(1, 2).contiguous()) / np.sqrt(hd)).amax(-1) if n else None
        if n:
            rel = 2.0 ** -20 * (1 + big).transpose(0, 1).repeat_interleave(hd, 1)
            size = torch.matmul(p, x[2].abs()).transpose(0, 1).reshape(n, H)
            assert ((got[at:at + n] - want).abs() <= rel * size + 2.0 ** -25 / sc).all()
        at += n
    assert (ctx[T:] == 7).all()


def _spread(w, how):
    """Weights moved towards or past an end of the pair operands' range."""
    w = {k: v.copy() for k, v in w.items()}
    for k in w:
        if how == "wide_gain" and k.endswith("LayerNorm.weight"):
            w[k] *= 40.0
        if how == "outlier_gain" and k == "embeddings.LayerNorm.weight":
            w[k][5] = 5.0e3                                # one feature far above the rest: fp32 kernels
        if how == "outlier_gain" and "layer.0.attention.self" in k and k.endswith("weight"):
            w[k][:, 5] /= 5.0e3
        if how == "zero_matrix" and k.endswith("attention.output.dense.weight"):
            w[k][:] = 0.0                                  # no scale: fp32 kernels
        if how == "tiny_row" and k.endswith("intermediate.dense.weight"):
            w[k][3] *= 1e-7                                # a row far below the rest: fp32 kernels
        if how == "small_values" and ".attention.self.value." in k:
            w[k] *= 2.0 ** -11                             # v far below the scale it shares with q and k: fp32 kernels
        if how == "small_weights" and k.endswith("dense.weight"):
            w[k] *= 2.0 ** -20
    return w


@pytest.mark.parametrize("how,products", [("wide_gain", 1), ("small_weights", 1), ("outlier_gain", 0), ("zero_matrix", 0),
                                          ("tiny_row", 0), ("small_values", 0)])
def test_models_at_the_ends_of_the_range(env, weights_for, how, products):
    import oracle
    torch, eb, N, L = env
    cfg = eb.TINY
    w = _spread(weights_for(cfg), how)
    rng = np.random.default_rng(5)
    B, S = 9, 31
    ids = rng.integers(10, cfg.vocab_size, (B, S)).astype(np.uint32)
    n = rng.integers(1, S + 1, B)
    mask = (np.arange(S)[None, :] < n[:, None]).astype(np.uint32)
    m = eb.Model.from_weights(w, cfg, "fp32")
    try:
        assert L.ebh_op_products(m._h, B, S) == products
        got = m.encode_ids(ids * mask, mask)
    finally:
        m.close()
    want = oracle.OracleModel(cfg, w).encode_unpadded(ids * mask, mask, normalize=True)
    assert np.isfinite(got).all()
    # fp32 against fp32: components of unit vectors of 64, each forward within a few
    # 2^-24 of them a layer (one feature 5,000 times the others leaves them 2^-12 less)
    assert np.abs(got - want).max() <= (5e-6 if how == "outlier_gain" else 5e-7)


def test_rows_too_long_for_the_pair_products(env):
    """An FFN of 1.9 million columns is beyond the pair products' 32-bit row offsets:
    the model keeps the fp32 kernels."""
    torch, eb, N, L = env
    cfg = eb.BertConfig(hidden_size=64, num_attention_heads=2, num_hidden_layers=1, intermediate_size=1_900_032,
                        vocab_size=50, max_position_embeddings=32, layer_norm_eps=1e-12)
    r = np.random.default_rng(1)
    shapes = {"embeddings.word_embeddings.weight": (50, 64), "embeddings.position_embeddings.weight": (32, 64),
              "embeddings.token_type_embeddings.weight": (2, 64)}
    w = {k: r.standard_normal(s).astype(np.float32) for k, s in shapes.items()}
    for k in ("embeddings.", "encoder.layer.0.attention.output.", "encoder.layer.0.output."):
        w[k + "LayerNorm.weight"], w[k + "LayerNorm.bias"] = np.ones(64, np.float32), np.zeros(64, np.float32)
    for k, n, m in (("attention.self.query", 64, 64), ("attention.self.key", 64, 64), ("attention.self.value", 64, 64),
                    ("attention.output.dense", 64, 64), ("intermediate.dense", cfg.intermediate_size, 64),
                    ("output.dense", 64, cfg.intermediate_size)):
        w["encoder.layer.0." + k + ".weight"] = np.float32(0.04) * r.standard_normal((n, m), dtype=np.float32)
        w["encoder.layer.0." + k + ".bias"] = np.zeros(n, np.float32)
    ids, mask = r.integers(0, 50, (5, 20)).astype(np.uint32), np.ones((5, 20), np.uint32)
    got = []
    for dtype in ("fp32", "fp32-bf16x6"):
        m = eb.Model.from_weights(w, cfg, dtype)
        try:
            got.append(m.encode_ids(ids, mask))
        finally:
            m.close()
    # Sums of n = 1.9 million terms of random signs in two orders: a partial sum S_k
    # is rounded by up to 2^-24 |S_k|, and |S_k|^2 grows as k, so each order is off
    # by some sqrt(n / 2) 2^-24 / sqrt(3) = 3e-5 of the sum's norm, at most the unit
    # vector's, and both by twice that at most
    assert np.isfinite(got[0]).all() and np.linalg.norm(got[0] - got[1], axis=1).max() <= 7e-5


# pairs; pairs with the rest; the few-token kernels (a partial per head) at the
# workspace sizes just above their own; products whose operands are not pairs
@pytest.mark.parametrize("dtype,B,S,after", [
    ("fp32", 3, 22, (6, 60)), ("fp32", 5, 128, (20, 67)), ("fp32", 40, 50, (43, 64)), ("fp32", 63, 128, (65, 128)),
    ("fp32", 5, 140, (4, 201)), ("fp32", 4, 16, (5, 16)), ("fp32", 1, 64, (1, 95)), ("fp32", 2, 31, (3, 31)),
    ("fp32-bf16x6", 4, 16, (5, 16)), ("fp32-bf16x6", 21, 64, (26, 64)), ("fp32-bf16x6", 3, 64, (67, 128))])
def test_vectors_do_not_depend_on_earlier_batches(env, weights_for, dtype, B, S, after):
    """A batch gives the same bits in a fresh model and in one whose workspace a
    larger batch has grown (a product's split count goes by the batch alone)."""
    torch, eb, N, L = env
    cfg = eb.MINILM_L6
    w = weights_for(cfg)
    rng = np.random.default_rng(7)

    def batch(b, s):
        return rng.integers(10, cfg.vocab_size, (b, s)).astype(np.uint32), np.ones((b, s), np.uint32)

    ids, mask = batch(B, S)
    fresh, grown = eb.Model.from_weights(w, cfg, dtype), eb.Model.from_weights(w, cfg, dtype)
    try:
        want = fresh.encode_ids(ids, mask)
        grown.encode_ids(*batch(*after))
        got = grown.encode_ids(ids, mask)
    finally:
        fresh.close()
        grown.close()
    assert np.array_equal(got, want)
