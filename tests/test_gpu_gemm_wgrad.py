"""coset_gemm_wgrad: the weight gradient gy^T x at the shapes coset_gemm_tn
does not take.  As in test_gpu_gemm.py the pin is exactness: with small-integer
bf16 operands every partial sum is an integer below 2^24, so any summation order
gives the integer product itself."""
import pytest
import torch

from coset_amd import _lib, layers

pytestmark = pytest.mark.gpu

# (M, N, K): one block; one past a tile of either size, K one past a stage; one
# stage; several splits with a ragged last one; more tiles than a band of 4 rows
SHAPES = [(8, 8, 1), (200, 136, 65), (64, 1000, 64), (768, 320, 1000), (1000, 200, 4001), (1536, 1000, 300),
          (256, 256, 16384)]


@pytest.fixture
def tile():
    yield
    _lib.set_gemm_wgrad_tile(1)


@pytest.mark.parametrize("mode", [1, 2, 3])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_integer_operands_exact(M, N, K, mode, tile):
    _lib.set_gemm_wgrad_tile(mode)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randint(-4, 5, (K, M), device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randint(-4, 5, (K, N), device="cuda", generator=g).to(torch.bfloat16)
    exact = a.double().t() @ b.double()
    assert torch.equal(layers.gemm_wgrad(a, b, torch.float32).double(), exact)
    cs = torch.full((M,), float("nan"), device="cuda")
    c16 = layers.gemm_wgrad(a, b, torch.bfloat16, colsum=cs)
    assert torch.equal(c16, exact.float().to(torch.bfloat16))
    assert torch.equal(cs.double(), a.double().sum(0))


def test_gaussian_operands_and_repeatability():
    g = torch.Generator(device="cuda").manual_seed(4)
    a = torch.randn((5000, 776), device="cuda", generator=g).to(torch.bfloat16)
    b = torch.randn((5000, 320), device="cuda", generator=g).to(torch.bfloat16)
    ref, mag = a.double().t() @ b.double(), a.double().abs().t() @ b.double().abs()
    c = layers.gemm_wgrad(a, b, torch.float32)
    # fp32 sums of 5000 exact products: sqrt(K) 2^-24 typically, bounded by 2^-16
    assert ((c.double() - ref).abs() <= 2.0 ** -16 * mag).all()
    assert torch.equal(layers.gemm_wgrad(a, b, torch.float32), c)
    a[17, 3] = float("inf")
    c = layers.gemm_wgrad(a, b, torch.float32)
    assert torch.isfinite(c[:3]).all() and torch.isfinite(c[4:]).all() and not torch.isfinite(c[3]).any()


def test_refusals_fall_back():
    """Shapes, dtypes and alignments it does not take give None (the layer then
    uses torch.mm), and a short workspace is refused before any launch."""
    a = torch.zeros((100, 64), dtype=torch.bfloat16, device="cuda")
    assert layers.gemm_wgrad(a[:, :60].contiguous(), a) is None          # M not a multiple of 8
    assert layers.gemm_wgrad(a[:0], a[:0]) is None                       # no tokens
    assert layers.gemm_wgrad(a.float(), a.float()) is None
    flat = torch.zeros(100 * 64 + 1, dtype=torch.bfloat16, device="cuda")[1:].view(100, 64)
    assert flat.is_contiguous() and layers.gemm_wgrad(flat, a) is None   # 2-byte aligned
    assert not layers._gemm_wgrad_takes(flat, a, True)
    lib = _lib.load()
    need = int(lib.coset_gemm_wgrad_workspace_floats(64, 64, 100))
    ws = torch.zeros(need, device="cuda")
    out = torch.zeros((64, 64), dtype=torch.bfloat16, device="cuda")
    for ptr, n in ((0, 0), (ws.data_ptr(), need - 1)):
        assert lib.coset_gemm_wgrad(a.data_ptr(), 64, a.data_ptr(), 64, out.data_ptr(), 64, _lib.BF16, 64, 64, 100, 0,
                                    ptr, n, _lib.stream_of(a)) == -1


@pytest.mark.parametrize("kind", ["plain", "expanded", "strided", "misaligned", "3d"])
def test_layer_gradients_over_operand_forms(kind):
    """The layer's dW and db with the kernels on and off, for the forms of gy
    and x that autograd hands over: contiguous, an expanded gradient (sum),
    strided rows, a misaligned view, batched tokens."""
    import coset_amd as ca
    torch.manual_seed(3)
    layer = ca.create_e8_hnlq_linear(320, 264, Delta0=1.5)
    n = 1000
    x = torch.randn(n, 320, device="cuda").to(torch.bfloat16)
    gy = torch.randn(n, 264, device="cuda").to(torch.bfloat16)
    if kind == "expanded":
        gy = torch.ones((), dtype=torch.bfloat16, device="cuda").expand(n, 264)
    elif kind == "strided":
        x = torch.randn(n, 640, device="cuda").to(torch.bfloat16)[:, 320:]
        gy = torch.randn(264, n, device="cuda").to(torch.bfloat16).t()
    elif kind == "misaligned":
        x = torch.randn(n * 320 + 1, device="cuda").to(torch.bfloat16)[1:].view(n, 320)
    elif kind == "3d":
        x, gy = x.view(10, 100, 320), gy.view(10, 100, 264)
    got = {}
    for on in (True, False):
        layers.set_gemm_tn(on)
        try:
            layer.zero_grad(set_to_none=True)
            layer(x).backward(gy)
            got[on] = (layer.weight.grad.clone(), layer.bias.grad.clone())
        finally:
            layers.set_gemm_tn(True)
    g2, x2 = gy.reshape(n, 264).double(), x.reshape(n, 320).double()
    mag = g2.abs().t() @ x2.abs()
    d = (got[True][0] - got[False][0]).abs()
    # one bf16 rounding of fp32 sums that differ by their accumulation error
    assert (d <= 2.0 ** -7 * got[False][0].abs() + 2.0 ** -16 * mag).all()
    assert ((got[True][1].double() - g2.sum(0)).abs() <= 2.0 ** -16 * g2.abs().sum(0)).all()


def test_captured_step_replays_the_kernel():
    """A captured step whose dW runs on coset_gemm_wgrad: every replay equals
    the eager gradients bit for bit."""
    import coset_amd as ca
    torch.manual_seed(5)
    layer = ca.create_e8_hnlq_linear(320, 264, Delta0=1.5)
    x = torch.randn(1000, 320, device="cuda").to(torch.bfloat16)
    gy = torch.randn(1000, 264, device="cuda").to(torch.bfloat16)
    layer(x).backward(gy)
    want = layer.weight.grad.clone(), layer.bias.grad.clone()
    layer.step_count.zero_()
    layer._host_step = None
    step = ca.CapturedQATStep(layer, x.clone(), gy.clone())
    for _ in range(4):
        step.step()
        torch.cuda.synchronize()
        assert torch.equal(layer.weight.grad, want[0]) and torch.equal(layer.bias.grad, want[1])
        torch.zeros(1 << 20, device="cuda")


@pytest.mark.parametrize("tokens,fin,fout,need_x,kernel", [
    (1000, 256, 264, True, False), (1024, 1024, 2048, True, False), (2071, 256, 264, True, True),
    (2067, 256, 264, True, False), (8000, 3072, 2048, True, False), (5000, 320, 512, True, True),
    (1000, 256, 264, False, True), (1500, 512, 320, False, True),
    (1900, 3072, 2048, False, True), (5000, 3072, 2048, False, False), (5000, 2048, 3072, False, False),
    (5000, 3072, 3072, False, True)])
def test_rule_of_a_step_with_and_without_dx(tokens, fin, fout, need_x, kernel):
    """Which product takes the weight gradient, told by the bits of its K splits
    and column sums: with dX to compute, torch.mm below 2000 tokens and one more
    per 1000 outputs and for outputs above 4.8 M, without dX for these from 2000
    tokens unless one round of tiles holds them, else the kernel; the captured
    step's replays equal the eager step's gradients bit for bit on both sides."""
    import coset_amd as ca
    torch.manual_seed(7)
    layer = ca.create_e8_hnlq_linear(fin, fout, Delta0=1.5)
    with torch.no_grad():
        layer.weight.mul_(0.02)
    x = torch.randn(tokens, fin, device="cuda").to(torch.bfloat16).requires_grad_(need_x)
    gy = torch.randn(tokens, fout, device="cuda").to(torch.bfloat16)

    def grads():
        layer.zero_grad(set_to_none=True)
        x.grad = None
        layer(x).backward(gy)
        return [layer.weight.grad, layer.theta_beta.grad, layer.bias.grad, x.grad]

    want = grads()
    try:
        layers.set_gemm_tn(False)
        library = grads()
    finally:
        layers.set_gemm_tn(True)
    assert (torch.equal(want[0], library[0]) and torch.equal(want[2], library[2])) == (not kernel)
    step = ca.CapturedQATStep(layer, x.detach().clone().requires_grad_(need_x), gy.clone())
    for _ in range(3):
        step.step()
        torch.cuda.synchronize()
        got = [layer.weight.grad, layer.theta_beta.grad, layer.bias.grad, step.x.grad]
        for a, r in zip(got, want):
            assert (a is None) == (r is None) and (a is None or torch.equal(a, r))
