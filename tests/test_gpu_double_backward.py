"""Second derivatives through the layer on the GPU (a backward with
create_graph=True), where its products would otherwise run on the
weight-gradient kernels."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


# tokens x fin x fout that coset_gemm_tn (4096) and coset_gemm_wgrad take in bf16
@pytest.mark.parametrize("tokens,fin,fout", [(4096, 768, 768), (1000, 320, 264)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
def test_hessian_vector_product_without_the_quantizer(dt, tokens, fin, fout):
    """Warm-up epochs (quantizer off): the gradient of |dL/dW|^2 + |dL/db|^2 +
    |dL/dx|^2 reaches x, W and the bias as it does through F.linear."""
    import coset_amd as ca
    torch.manual_seed(2)
    layer = ca.create_e8_hnlq_linear(fin, fout, Delta0=1.5, warmup_epochs=1)
    x = torch.randn(tokens, fin, device="cuda").to(dt)
    with torch.no_grad():
        layer.weight.mul_(fin ** -0.5)
        layer.bias.normal_()

    def second(fn, x, W, b):
        y = fn(x)
        first = torch.autograd.grad(y.float().square().mean(), [x, W, b], create_graph=True)
        return torch.autograd.grad(sum(t.float().square().sum() for t in first), [x, W, b])

    x1 = x.clone().requires_grad_()
    got = second(layer, x1, layer.weight, layer.bias)
    x2, W, b = (t.detach().float().requires_grad_() for t in (x, layer.weight, layer.bias))
    want = second(lambda v: F.linear(v, W, b), x2, W, b)
    for a, r in zip(got, want):
        # six bf16 roundings deep (2^-9 each); a lost path is off by 1e-1
        tol = 2.0 ** -5 if dt == torch.bfloat16 else 1e-4
        assert (a.float() - r).norm() <= tol * r.norm()
