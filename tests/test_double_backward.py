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
    monkeypatch.setattr(layers, "_gemm_wgrad_takes", lambda a, b, with_bias: True)
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
