"""Second derivatives through the layer's linear (a backward with
create_graph=True: gradient penalties, Hessian-vector products), on the CPU
against plain torch autograd in float64.  The kernels are stood in for by torch
functions that, like them, leave no graph."""
import pytest
import torch
import torch.nn.functional as F

from coset_amd import layers


def _operands(shape, fin, fout, dtype=torch.float32):
    g = torch.Generator().manual_seed(3)
    x = torch.randn(*shape, fin, generator=g).to(dtype).requires_grad_()
    W = torch.randn(fout, fin, generator=g).to(dtype).requires_grad_()
    b = torch.randn(fout, generator=g).to(dtype).requires_grad_()
    return x, W, b


def _penalty(fn, leaves):
    """Gradients of sum |dL/dleaf|^2 for a nonlinear loss L of fn(*leaves)."""
    y = fn(*leaves)
    first = torch.autograd.grad((y.sin() * y).sum(), leaves, create_graph=True)
    return torch.autograd.grad(sum(t.square().sum() for t in first), leaves)


@pytest.fixture
def kernels(monkeypatch):
    """The weight-gradient kernels take every product; all leave no graph."""
    def wgrad(a, b, out_dtype=None, colsum=None):
        with torch.no_grad():
            if colsum is not None:
                colsum.copy_(a.float().sum(0))
            return a.t() @ b

    monkeypatch.setattr(layers, "_gemm_tn_takes", lambda a, b: False)
    monkeypatch.setattr(layers, "_gemm_wgrad_takes", lambda a, b, with_bias, with_dx=False: True)
    monkeypatch.setattr(layers, "gemm_wgrad", wgrad)
    monkeypatch.setattr(layers, "colsum", lambda a: a.detach().float().sum(0))


@pytest.mark.parametrize("fout", [8, 5])   # with and without the column-sum kernel's width
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("shape", [(7,), (2, 3)])
def test_linear_products_are_differentiable_again(kernels, shape, bias, fout):
    x, W, b = _operands(shape, 16, fout)
    leaves = [x, W] + ([b] if bias else [])
    got = _penalty(lambda x, W, b=None: layers.QATLinearFn.apply(x, W, b, None), leaves)
    want = _penalty(F.linear, [t.detach().double().requires_grad_() for t in leaves])
    for a, r in zip(got, want):
        # fp32: six products and a sine deep, |y| up to 10 multiplying its rounding;
        # a lost path is off by 1e-1
        assert (a - r).norm() <= 2.0 ** -13 * r.norm()


CFG = ((1.5, 0.1, 12.0, 2), 4, 2, 0.9, 1)   # QATLayerFn's: bounds, q, M, clip, blocks per tile


@pytest.fixture
def quantizer(monkeypatch):
    """A rounding quantizer with the fused one's interface and straight-through
    gradient: W_q = clamp(round(W beta) / beta, +-clip), beta = 1 + sigmoid(theta)."""
    def fwd(Wc, theta, sigma, xmax, step_count, bounds, q, M, clip, bpt, out_dtype, bias=None):
        s = torch.sigmoid(theta)
        beta = 1 + s
        r = torch.round(Wc * beta[:, None])
        Wq = (r / beta[:, None]).clamp(-clip, clip)
        return Wq.to(out_dtype), r, beta, s * (1 - s), None if bias is None else bias.to(out_dtype)

    def bwd(g, Wc, r, beta, dbdt, q, M, clip, bpt, theta_shape):
        g = g.detach()
        b = beta[:, None]
        g = g * ((r / b).abs() <= clip)
        return g, ((g / b * Wc - g * r / (b * b)).sum(1) * dbdt).view(theta_shape)

    monkeypatch.setattr(layers, "qat_fwd_theta", fwd)
    monkeypatch.setattr(layers, "qat_bwd_theta", bwd)


def _reference_layer(x, W, theta, b):
    """The same layer in torch operations autograd differentiates by itself."""
    beta = (1 + torch.sigmoid(theta))[:, None]
    t = W * beta
    q = t + (torch.round(t) - t).detach()
    return F.linear(x, (q / beta).clamp(-CFG[3], CFG[3]), b)


def _fused(x, W, theta, b):
    return layers.QATLayerFn.apply(x, W, theta, b, None, None, None, CFG)


def _two_functions(x, W, theta, b):
    Wq = layers.E8ThetaWeightQuant.apply(W, theta, None, None, None, *CFG, x.dtype)
    return layers.QATLinearFn.apply(x, Wq, b, None)


@pytest.mark.parametrize("layer", [_fused, _two_functions])
@pytest.mark.parametrize("linear_loss", [False, True])   # True: the gradient that arrives is a constant
@pytest.mark.parametrize("bias", [True, False])
def test_gradient_penalty_reaches_weight_and_theta(kernels, quantizer, layer, bias, linear_loss):
    """W.grad, theta.grad, x.grad and the bias's of |dL/dx|^2 + L, through the
    one node and through its two functions."""
    x, W, b = _operands((7,), 16, 8)
    theta = torch.linspace(-1, 1, 8).requires_grad_()
    c = torch.randn(7, 8, generator=torch.Generator().manual_seed(4))

    def grads(fn, x, W, theta, b, c):
        y = fn(x, W, theta, b if bias else None)
        loss = (y * c).sum() if linear_loss else (y.sin() * y).sum()
        dx, = torch.autograd.grad(loss, x, create_graph=True)
        return torch.autograd.grad(dx.square().sum() + loss, [x, W, theta] + ([b] if bias else []))

    got = grads(layer, x, W, theta, b, c)
    want = grads(_reference_layer, *(t.detach().double().requires_grad_() for t in (x, W, theta, b)), c.double())
    for a, r in zip(got, want):
        assert (a - r).norm() <= 2.0 ** -13 * r.norm()
