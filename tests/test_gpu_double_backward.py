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


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("tiling", ["row", "block"])
def test_gradient_penalty_equals_the_two_functions(dt, tiling):
    """The gradients of |dL/dx|^2 + L through the layer's one node are those of
    its two functions; also where the weight is not a leaf."""
    import coset_amd as ca
    from coset_amd import layers
    torch.manual_seed(6)
    layer = ca.create_e8_hnlq_linear(72, 40, Delta0=1.5, tiling=tiling)
    x = torch.randn(33, 72, device="cuda").to(dt).requires_grad_()
    c = torch.randn(33, 40, device="cuda").to(dt)
    bpt = layer.blocks_per_row if tiling == "row" else 1
    leaves = [x, layer.weight, layer.theta_beta, layer.bias]

    def two(x):
        Wq = layers.E8ThetaWeightQuant.apply(layer.weight, layer.theta_beta, layer.sigma_ema, layer.xmax_ema, None,
                                             (float(layer.Delta0), float(layer.eta), layer._ginv_f, int(layer.M)), 4, 2,
                                             float(layer.weight_clip_value), int(bpt), dt)
        return layers.QATLinearFn.apply(x, Wq, layer.bias, None)

    def scaled(x):   # the weight as a function of the parameter: one more node above the layer's
        return torch.func.functional_call(layer, {"weight": layer.weight * 1.0}, x)

    for loss_of in (lambda y: (y * c).float().sum(), lambda y: y.float().square().sum()):
        def grads(fn):
            loss = loss_of(fn(x))
            dx, = torch.autograd.grad(loss, x, create_graph=True)
            return torch.autograd.grad(dx.float().square().sum() + loss, leaves, allow_unused=True)

        want = grads(two)
        assert all(t is not None and t.abs().sum() > 0 for t in want[1:])
        for fn in (layer, scaled):
            for a, r in zip(grads(fn), want):
                assert (a is None) == (r is None)
                # the two functions add the weight's gradients before the quantizer's
                # backward, the node after it: a rounding of each, and theta sums 72 of them
                tol = 2.0 ** -7 if dt == torch.bfloat16 else 2.0 ** -19
                assert a is None or (a - r).float().norm() <= tol * r.float().norm()
