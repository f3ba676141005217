"""The GEMM kernel of the vLUT matmul (large batches of the decoded formats)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# exact products, fp32 sums of at most K terms in any order: well inside 2^-14
# of the summands' magnitude (the bound of the other matrix-core kernels)
RTOL = 2.0 ** -14


def _weight(rows, K, q, M, seed):
    import coset_amd as ca
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = 1.5 * torch.randn(rows * K // 8, 8, device="cuda", generator=g)
    words = ca.hnlq_encode(x, q, M, 1.0).reshape(rows, K // 8, M)
    W = ca.hnlq_decode(words.reshape(-1, M), q, M, None).reshape(rows, K).double()
    return words, W, g


@pytest.mark.parametrize("layout", ["decoded", "decoded6"])
@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("B,rows,K", [(1, 4, 8), (129, 40, 64), (257, 200, 72), (300, 259, 1064), (127, 193, 200)])
def test_gemm_shapes_vs_dense(layout, dt, shape, B, rows, K):
    """Every tile shape at the edges of its tiles (one token, one token past a
    tile, ragged rows and k-blocks, K below one stage), with a dividing scale,
    a bias and the LSQ epilogue, against the dense product in float64."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(rows, K, 4, 2, 7 * B + rows)
    w = ca.vlut_prepare(words, 4, layout=layout)
    a = torch.randn(B, K, device="cuda", generator=g).to(dt)
    sc = torch.rand(rows, device="cuda", generator=g) + 0.5
    bias = torch.randn(rows, device="cuda", generator=g)
    try:
        _lib.set_vlut_gemm(2 + shape)
        y = ca.vlut_matmul(w, a, scale=sc)
        yb = ca.vlut_matmul(w, a, scale=sc, scale_mode="div", bias=bias)
        alpha = torch.tensor(3.0, device="cuda")
        yl = ca.vlut_matmul(w, a, scale=sc, scale_mode="div", bias=bias, act_quant=(alpha, 127))
    finally:
        _lib.set_vlut_gemm(1)
    ref, mag = a.double() @ W.t(), a.double().abs() @ W.t().abs()
    assert ((y.double() - ref * sc).abs() <= RTOL * mag * sc).all()
    assert ((yb.double() - (ref / sc + bias)).abs() <= RTOL * (mag / sc + bias.abs())).all()
    m = ca.LSQActivation(bit_width=8, init_alpha=3.0).cuda()
    with torch.no_grad():
        assert torch.equal(yl, m(yb))          # the epilogue on the same sums


def test_gemm_inf_activation_and_padding():
    """An infinite activation reaches its own token only, and activations past
    K are zero (0 x inf in the padding would make NaN)."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(72, 200, 4, 2, 3)    # 25 k-blocks: a ragged last stage
    w = ca.vlut_prepare(words, 4, layout="decoded")
    a = torch.randn(130, 200, device="cuda", generator=g).half()
    a[7, 199] = float("inf")
    try:
        for shape in range(4):
            _lib.set_vlut_gemm(2 + shape)
            y = ca.vlut_matmul(w, a)
            fin = torch.isfinite(y)
            assert fin[:7].all() and fin[8:].all()
            nz = W[:, 199] != 0
            assert not fin[7][nz].any()
    finally:
        _lib.set_vlut_gemm(1)


@pytest.mark.parametrize("B,rows,K", [(128, 768, 768), (1000, 1000, 1000), (700, 3072, 264)])
def test_gemm_natural_plan_equals_deep(B, rows, K):
    """Where the plan takes the GEMM kernel, its outputs agree with the deep
    kernel's (the same exact products, summed in another order), for both
    decoded formats bit for bit with each other, and fp32 activations run
    through it as three planes."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(rows, K, 4, 2, B)
    d8, d6 = (ca.vlut_prepare(words, 4, layout=lay) for lay in ("decoded", "decoded6"))
    a = torch.randn(B, K, device="cuda", generator=g)
    mag = a.double().abs() @ W.t().abs()
    for act in (a.bfloat16(), a.half(), a):
        y = ca.vlut_matmul(d8, act)
        assert torch.equal(y, ca.vlut_matmul(d6, act))
        try:
            _lib.set_vlut_gemm(0)
            y0 = ca.vlut_matmul(d8, act)
        finally:
            _lib.set_vlut_gemm(1)
        assert ((y - y0).double().abs() <= 2.0 ** -16 * mag).all()


def test_gemm_under_graph_capture():
    """Replays equal the eager result (no workspace, no memset nodes)."""
    import coset_amd as ca
    words, W, g = _weight(768, 768, 4, 2, 5)
    w = ca.vlut_prepare(words, 4, layout="decoded")
    a = torch.randn(512, 768, device="cuda", generator=g).bfloat16()
    want = ca.vlut_matmul(w, a)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y = ca.vlut_matmul(w, a)
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)


@pytest.mark.parametrize("B,rows,K", [(48, 768, 3072), (49, 132, 2056), (200, 1000, 1000), (64, 130, 4096)])
def test_gemm_fp32_splits(B, rows, K):
    """fp32 activations over a wide range of magnitudes through the natural
    plan (many K splits at few tokens; rows % 4 != 0 takes the scalar reduce),
    with bias: within the fp32 bound, and no further from float64 than the three
    planes run as 3B tokens on the deep kernel (times 1.25: both are rounding
    noise)."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(rows, K, 4, 2, B)
    w = ca.vlut_prepare(words, 4, layout="decoded")
    a = torch.randn(B, K, device="cuda", generator=g)
    a *= torch.exp2(torch.randint(-6, 7, (B, 1), device="cuda", generator=g).float())
    sc = torch.rand(rows, device="cuda", generator=g) + 0.5
    bias = torch.randn(rows, device="cuda", generator=g)
    ref = (a.double() @ W.t()) * sc + bias
    mag = (a.double().abs() @ W.t().abs()) * sc + bias.abs()
    y = ca.vlut_matmul(w, a, scale=sc, bias=bias)
    try:
        _lib.set_vlut_gemm(0)
        y0 = ca.vlut_matmul(w, a, scale=sc, bias=bias)
    finally:
        _lib.set_vlut_gemm(1)
    assert ((y - ref).abs() <= RTOL * mag).all()
    assert (y - ref).norm() <= 1.25 * (y0 - ref).norm()


def test_gemm_fp32_special_values():
    """Infinities and NaN stay in their token, and an output is finite exactly
    where the deep kernel's is."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(768, 3072, 4, 2, 8)
    w = ca.vlut_prepare(words, 4, layout="decoded6")
    a = torch.randn(60, 3072, device="cuda", generator=g)
    a[3, 5], a[9, 3071], a[20, 100], a[30] = float("inf"), -float("inf"), float("nan"), 1e-40
    y = ca.vlut_matmul(w, a)
    try:
        _lib.set_vlut_gemm(0)
        y0 = ca.vlut_matmul(w, a)
    finally:
        _lib.set_vlut_gemm(1)
    assert torch.equal(torch.isfinite(y), torch.isfinite(y0))
    keep = [i for i in range(60) if i not in (3, 9, 20)]
    assert torch.isfinite(y[keep]).all()


@pytest.mark.parametrize("layout", ["decoded", "decoded6"])
@pytest.mark.parametrize("rows,K", [(256, 256), (768, 768), (1000, 1000), (768, 3072)])
def test_fp32_at_the_gemm_kernels_first_tokens(layout, rows, K):
    """42 fp32 tokens (126 plane tokens) run as planes on the deep kernel; 43 to
    48, whose planes would reach the GEMM kernel, run on it whole: a token's
    output is then the same whatever the call's token count (one token tile, the
    same K splits)."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(rows, K, 4, 2, rows)
    w = ca.vlut_prepare(words, 4, layout=layout)
    a = torch.randn(48, K, device="cuda", generator=g)
    sc = torch.rand(rows, device="cuda", generator=g) + 0.5
    bias = torch.randn(rows, device="cuda", generator=g)
    ref = (a.double() @ W.t()) * sc + bias
    mag = (a.double().abs() @ W.t().abs()) * sc + bias.abs()
    y = {B: ca.vlut_matmul(w, a[:B], scale=sc, bias=bias) for B in (42, 43, 47, 48)}
    try:
        _lib.set_vlut_gemm(0)
        deep = ca.vlut_matmul(w, a[:42], scale=sc, bias=bias)
    finally:
        _lib.set_vlut_gemm(1)
    assert torch.equal(y[42], deep)
    for B in (43, 47):
        assert torch.equal(y[B], y[48][:B])
    for B, v in y.items():
        assert ((v - ref[:B]).abs() <= RTOL * mag[:B]).all()


@pytest.mark.parametrize("dt", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,rows,K,shape", [(127, 768, 768, None), (160, 768, 3072, None), (129, 2048, 1000, 3),
                                            (160, 3072, 3072, None), (256, 768, 2048, None), (256, 256, 256, 3),
                                            (512, 3072, 768, 3), (1000, 3072, 768, 2), (4096, 512, 512, 2),
                                            (2000, 512, 2048, -1), (700, 4096, 4096, -1)])
def test_plan_takes_the_faster_kernel(dt, B, rows, K, shape):
    """Where the deep kernel is the faster one (its splits fill the chip in one
    round, and no unsplit launch is about as fast) the plan takes it, else this kernel in the named shape (-1: with K
    splits): told apart by the bits of the sums, which the two add in different
    orders."""
    import coset_amd as ca
    from coset_amd import _lib
    words, W, g = _weight(rows, K, 4, 2, B)
    w = ca.vlut_prepare(words, 4, layout="decoded")
    a = torch.randn(B, K, device="cuda", generator=g).to(dt)
    y = ca.vlut_matmul(w, a)
    try:
        _lib.set_vlut_gemm(0)
        deep = ca.vlut_matmul(w, a)
        if shape is not None and shape >= 0:
            _lib.set_vlut_gemm(2 + shape)
            forced = ca.vlut_matmul(w, a)
    finally:
        _lib.set_vlut_gemm(1)
    assert torch.equal(y, deep) == (shape is None)
    assert shape is None or shape < 0 or torch.equal(y, forced)
