"""The fused layer's single autograd node against its two functions in turn."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("bias,train_theta,train_w,need_x", [(True, True, True, True), (False, True, True, False),
                                                             (True, False, True, True), (True, True, False, True),
                                                             (True, False, False, True), (True, False, False, False)])
@pytest.mark.parametrize("tiling", ["row", "block"])
def test_node_equals_the_two_functions(dt, bias, train_theta, train_w, need_x, tiling):
    """Output and every gradient bit for bit, for each choice of what trains."""
    import coset_amd as ca
    from coset_amd import layers
    torch.manual_seed(1)
    layer = ca.create_e8_hnlq_linear(72, 40, Delta0=1.5, bias=bias, theta_trainable=train_theta, tiling=tiling)
    layer.weight.requires_grad_(train_w)
    x = torch.randn(3, 33, 72, device="cuda").to(dt).requires_grad_(need_x)
    gy = torch.randn(3, 33, 40, device="cuda").to(dt)
    names = [n for n, p in layer.named_parameters() if p.requires_grad]

    def grads(y):
        if not y.requires_grad:
            return y, {}, None
        layer.zero_grad(set_to_none=True)
        x.grad = None
        y.backward(gy)
        return y.detach(), {n: getattr(layer, n).grad.clone() for n in names}, x.grad

    y1, g1, dx1 = grads(layer(x))
    assert int(layer.step_count) == 1 and layer._host_step == 1
    bpt = layer.blocks_per_row if tiling == "row" else 1
    out = layers.E8ThetaWeightQuant.apply(layer.weight, layer.theta_beta, layer.sigma_ema, layer.xmax_ema, None,
                                          (float(layer.Delta0), float(layer.eta), layer._ginv_f, int(layer.M)), 4, 2,
                                          float(layer.weight_clip_value), int(bpt), dt)
    y2, g2, dx2 = grads(layers.QATLinearFn.apply(x, out, layer.bias, None))
    assert torch.equal(y1, y2) and set(g1) == set(g2) == set(names)
    for n in names:
        assert torch.equal(g1[n], g2[n]), n
    assert (dx1 is None) == (dx2 is None) and (dx1 is None or torch.equal(dx1, dx2))


def test_in_place_weight_update_is_caught():
    """A weight changed between forward and backward still raises."""
    import coset_amd as ca
    layer = ca.create_e8_hnlq_linear(72, 40, Delta0=1.5)
    y = layer(torch.randn(8, 72, device="cuda"))
    with torch.no_grad():
        layer.weight.mul_(2.0)
    with pytest.raises(RuntimeError):
        y.sum().backward()


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("how", ["subclass", "instance"])
def test_overridden_weight_quantizer_is_called(dt, how):
    """A replaced weight quantizer (a subclass's method or one set on the
    layer) decides the weight of the training forward, and its gradient."""
    import types
    import coset_amd as ca
    from coset_amd.layers import HNLQLinearQAT

    class Halved(HNLQLinearQAT):
        def _quantize_weights_with_bias(self, out_dtype, cast_bias):
            W_q, b = super()._quantize_weights_with_bias(out_dtype, cast_bias)
            return W_q * 0.5, b

    torch.manual_seed(1)
    plain = ca.create_e8_hnlq_linear(72, 40, Delta0=1.5)
    layer = ca.create_e8_hnlq_linear(72, 40, Delta0=1.5)
    layer.load_state_dict(plain.state_dict())
    if how == "subclass":
        layer.__class__ = Halved
    else:
        def halved(self, out_dtype, cast_bias):
            W_q, b = HNLQLinearQAT._quantize_weights_with_bias(self, out_dtype, cast_bias)
            return W_q * 0.5, b
        layer._quantize_weights_with_bias = types.MethodType(halved, layer)
    x = torch.randn(33, 72, device="cuda").to(dt)
    y0, y = plain(x), layer(x)
    with torch.no_grad():
        assert torch.equal(y, y0 * 0.5)        # halving is exact; the bias is zero
    y0.sum().backward()
    y.sum().backward()
    assert torch.equal(layer.weight.grad, 0.5 * plain.weight.grad)
