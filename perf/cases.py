"""What the library is timed on: the calls its users make, over the sizes they make them at.

A case is a dict of plain values; ``kind`` names the path:

  head     a small layer's no-grad forward (the classification head of the
           reference's example), fp32 tokens
  codec    the native codec on a tensor of 8-wide blocks: one-pass round trip,
           encode, or decode
  vlut     vlut_matmul on a weight prepared once (token-by-token decoding and
           small batches)
  packed   PackedLinear, the served form of a trained layer (whole prompts)
  qat      one training step of a quantized layer, forward and backward, eager
  graph    the same step replayed through CapturedQATStep

Sizes are this repository's configurations (768 / 3072 layers, a 4096 x 4096
weight, 2^24 and 2^22 blocks, 32 x 128 tokens) and generic ones around them.
"""
import math

import torch

import coset_amd

# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # the 768 -> 10 classification head on a batch of 32: one small launch, bound by latency
        dict(name="head_768x10", kind="head", tokens=32, fin=768, fout=10),
        # bulk compression of a tensor, words and reconstruction in one pass
        dict(name="roundtrip_bulk", kind="codec", op="roundtrip", n=1 << 24, q=4, M=2, dtype="f32", scale="none",
             heavy=False, per_row=1),
        # heavy-tailed bf16 weights with a scale per row, three levels of q = 16
        dict(name="roundtrip_heavy", kind="codec", op="roundtrip", n=1 << 22, q=16, M=3, dtype="bf16", scale="row",
             heavy=True, per_row=512),
        # storing a bf16 checkpoint tensor (8191 rows of 4096) as words, a scale per row
        dict(name="encode_rows", kind="codec", op="encode", n=8191 * 512, q=4, M=2, dtype="bf16", scale="row",
             heavy=False, per_row=512),
        # loading it back to bf16
        dict(name="decode_rows", kind="codec", op="decode", n=8191 * 512, q=4, M=2, dtype="bf16", scale="row",
             heavy=False, per_row=512),
        # generating one token through a 4096 x 4096 layer
        dict(name="vlut_1", kind="vlut", tokens=1, rows=4096, cols=4096, q=4, M=2, dtype="f16", layout="decoded"),
        # a serving batch of 48 sequences through the same layer
        dict(name="vlut_48", kind="vlut", tokens=48, rows=4096, cols=4096, q=4, M=2, dtype="f16", layout="decoded"),
        # a served layer on whole sequences, 32 x 128 tokens
        dict(name="packed_4096", kind="packed", tokens=4096, fin=768, fout=3072, dtype="bf16", bias=True),
        # one sequence of 197 patches in fp32 (the layer's own dtype)
        dict(name="packed_197_f32", kind="packed", tokens=197, fin=3072, fout=768, dtype="f32", bias=True),
        # training in bf16 on 32 sequences of 512 tokens
        dict(name="qat_16384", kind="qat", tokens=16384, fin=3072, fout=768, dtype="bf16"),
        # training in fp32, a last batch of 1000 tokens
        dict(name="qat_1000_f32", kind="qat", tokens=1000, fin=768, fout=768, dtype="f32"),
        # the captured training step at 32 x 128 tokens
        dict(name="graph_4096", kind="graph", tokens=4096, fin=768, fout=3072, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_WIDTHS = [256, 320, 512, 768, 1000, 1024, 1536, 2048, 3072]


def draw(rng):
    kind = rng.choice(["head", "codec", "codec", "codec", "vlut", "vlut", "packed", "packed", "qat", "qat", "graph"])
    if kind == "head":
        return dict(kind=kind, tokens=_log(rng, 1, 64), fin=8 * _log(rng, 16, 512), fout=_log(rng, 2, 300))
    if kind == "codec":
        q, M = rng.choice([(4, 2), (4, 2), (4, 2), (4, 1), (2, 3), (8, 2), (16, 2), (16, 3)])
        scale = rng.choice(["none", "beta", "row", "row"])
        per_row = rng.choice([32, 96, 125, 384, 512]) if scale == "row" else 1
        n = max(1, _log(rng, 1000, (1 << 24) // 4) // per_row) * per_row
        return dict(kind=kind, op=rng.choice(["roundtrip", "encode", "decode"]), n=n, q=q, M=M,
                    dtype=rng.choice(["f32", "bf16"]), scale=scale, heavy=rng.random() < 0.3, per_row=per_row)
    if kind == "vlut":
        rows = rng.choice([768, 1000, 2048, 3072, 4096])
        cols = rng.choice([768, 1000, 2048, 3072, 4096])
        return dict(kind=kind, tokens=_log(rng, 1, 256), rows=rows, cols=cols, q=4, M=2,
                    dtype=rng.choice(["f16", "bf16", "f32"]), layout=rng.choice(["decoded", "decoded", "tiled"]))
    if kind == "packed":
        return dict(kind=kind, tokens=_log(rng, 16, 8192), fin=rng.choice(_WIDTHS), fout=rng.choice(_WIDTHS),
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]), bias=rng.random() < 0.7)
    fin, fout = rng.choice(_WIDTHS), rng.choice(_WIDTHS)
    if kind == "qat":
        dtype = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind=kind, tokens=_log(rng, 64, 16384 if dtype == "bf16" else 2048), fin=fin, fout=fout,
                    dtype=dtype)
    return dict(kind=kind, tokens=128 * _log(rng, 4, 64), fin=fin, fout=fout, dtype="bf16")


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_SIZE = {"f32": 4, "bf16": 2, "f16": 2}
_DELTA0, _ETA, _GINV, _CLIP = 1.5, 0.1, 12.0, 2.0


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape):
    return torch.randn(shape, device="cuda", generator=g)


def _blocks(case, g):
    """The values that a codec call takes: Gaussian, or Student's t(3) clipped at +-2."""
    n = case["n"]
    if not case["heavy"]:
        x = _randn(g, n, 8)
        return x * 0.02 if case["scale"] == "row" else x
    chi2 = _randn(g, n, 8).square_()
    chi2 += _randn(g, n, 8).square_()
    chi2 += _randn(g, n, 8).square_()
    return (_randn(g, n, 8) / (chi2 / 3).sqrt_()).clamp_(-2.0, 2.0)


def _scales(case, x, g):
    """hnlq_* keyword arguments of the case's scaling.  Per row: the layer's
    bounds from the row's own statistics, theta drawn uniformly in them;
    weights of q = 4 take a scale that brings them to unit variance."""
    if case["scale"] == "none":
        return dict(beta=None)
    if case["scale"] == "beta":
        return dict(beta=0.3)
    rows = case["n"] // case["per_row"]
    u = torch.rand(rows, device="cuda", generator=g)
    w = x.view(rows, -1).float()
    if not case["heavy"]:
        return dict(beta_row=(0.7 + 0.6 * u) / w.std(dim=1), blocks_per_row=case["per_row"])
    qm = float(case["q"] ** case["M"])
    sigma, xmax = w.std(dim=1), w.abs().amax(dim=1)
    hi = torch.minimum(_DELTA0 * (qm - 1) / (2 * _GINV * xmax), _DELTA0 * (qm - 1) / (2 * _ETA * _GINV * sigma))
    lo = torch.minimum((_DELTA0 / qm) / (_ETA * _GINV * sigma), hi * 0.9)
    return dict(beta_row=lo + u * (hi - lo), blocks_per_row=case["per_row"])


def _weight_words(g, rows, cols, q, M):
    """Level words [rows, cols / 8, M] and per-row beta of a Gaussian weight."""
    w = 0.02 * _randn(g, rows, cols)
    beta = (0.8 + 0.4 * torch.rand(rows, device="cuda", generator=g)) / 0.02
    words = _words(_encode((w * beta[:, None]).view(-1, 8), q, M), q)
    return words.view(rows, cols // 8, M), beta


def _layer(case, g):
    """A layer in mid-training: weights N(0, 0.02), statistics that have
    followed them, thetas that have moved."""
    fin, fout = case["fin"], case["fout"]
    layer = coset_amd.create_e8_hnlq_linear(fin, fout, device="cuda", Delta0=_DELTA0, weight_clip_value=_CLIP)
    with torch.no_grad():
        w = 0.02 * _randn(g, fout, fin)
        layer.weight.copy_(w)
        layer.bias.copy_(0.1 * _randn(g, fout))
        layer.theta_beta.copy_(1.0 + 0.5 * _randn(g, fout))
        layer.sigma_ema.copy_(w.std(dim=1))
        layer.xmax_ema.copy_(w.abs().amax(dim=1))
    return layer


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind == "codec":
        x = _blocks(case, g)
        kw = _scales(case, x, g)
        if case["op"] != "decode":
            return dict(case=case, x=x.to(_DT[case["dtype"]]), kw=kw)
        return dict(case=case, words=_words(_encode_scaled(x, kw, case["q"], case["M"]), case["q"]), kw=kw)
    if kind == "vlut":
        words, beta = _weight_words(g, case["rows"], case["cols"], case["q"], case["M"])
        act = _randn(g, case["tokens"], case["cols"]).to(_DT[case["dtype"]])
        return dict(case=case, act=act, scale=1.0 / beta, raw=words,
                    words=coset_amd.vlut_prepare(words, case["q"], layout=case["layout"]))
    if kind == "packed":
        words, beta = _weight_words(g, case["fout"], case["fin"], 4, 2)
        tensors = dict(words=words, beta=beta)
        if case["bias"]:
            tensors["bias"] = 0.1 * _randn(g, case["fout"])
        meta = dict(q=4, M=2, in_features=case["fin"], out_features=case["fout"])
        x = _randn(g, case["tokens"], case["fin"]).to(_DT[case["dtype"]])
        return dict(case=case, x=x, tensors=tensors, layer=coset_amd.PackedLinear(tensors, meta))
    layer = _layer(case, g)
    if kind == "head":
        return dict(case=case, layer=layer, x=_randn(g, case["tokens"], case["fin"]))
    dt = _DT[case["dtype"]]
    x = _randn(g, case["tokens"], case["fin"]).to(dt).requires_grad_()
    gy = _randn(g, case["tokens"], case["fout"]).to(dt)
    if kind == "qat":
        return dict(case=case, layer=layer, x=x, gy=gy)
    step = coset_amd.CapturedQATStep(layer, x.detach().clone().requires_grad_(), gy.clone())
    return dict(case=case, layer=layer, x=x.detach(), gy=gy, step=step)


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def _signed(words):
    """The words' bits as signed integers (torch indexes no unsigned ones)."""
    return words.view(torch.int16 if words.dtype == torch.uint16 else torch.int32)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "codec":
        q, M, kw = case["q"], case["M"], state["kw"]
        if case["op"] == "roundtrip":
            words, decoded = coset_amd.hnlq_roundtrip(state["x"], q, M, **kw)
            return _signed(words), decoded
        if case["op"] == "encode":
            return _signed(coset_amd.hnlq_encode(state["x"], q, M, **kw))
        return coset_amd.hnlq_decode(state["words"], q, M, out_dtype=_DT[case["dtype"]], **kw)
    if kind == "vlut":
        return coset_amd.vlut_matmul(state["words"], state["act"], scale=state["scale"])
    if kind == "packed":
        return state["layer"](state["x"])
    if kind == "head":
        with torch.no_grad():
            return state["layer"](state["x"])
    layer = state["layer"]
    if kind == "graph":
        y = state["step"].step(state["x"], state["gy"])
        x = state["step"].x
    else:
        layer.zero_grad(set_to_none=True)
        x = state["x"]
        x.grad = None
        y = layer(x)
        y.backward(state["gy"])
        y = y.detach()
    return dict(y=y, dx=x.grad, dW=layer.weight.grad, dtheta=layer.theta_beta.grad, db=layer.bias.grad)


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "codec":
        word = 2 if case["q"] <= 4 else 4
        word *= case["M"]
        value = 8 * _SIZE[case["dtype"]]
        per = {"roundtrip": value + word + 32, "encode": value + word, "decode": word + value}[case["op"]]
        rows = case["n"] // case["per_row"] if case["scale"] == "row" else 0
        return dict(bytes=case["n"] * per + 4 * rows, flops=0)
    if kind == "vlut":
        t, rows, cols = case["tokens"], case["rows"], case["cols"]
        codes = rows * cols // 8 * 2 * case["M"]
        return dict(bytes=codes + t * (cols * _SIZE[case["dtype"]] + 4 * rows) + 4 * rows, flops=2 * t * rows * cols)
    t, fin, fout = case["tokens"], case["fin"], case["fout"]
    if kind == "packed":
        return dict(bytes=fin * fout // 2 + t * (fin * _SIZE[case["dtype"]] + 4 * fout) + 8 * fout,
                    flops=2 * t * fin * fout)
    if kind == "head":
        return dict(bytes=4 * (fin * fout + t * (fin + fout) + 4 * fout), flops=2 * t * fin * fout)
    # x, gy read; y, dx written; weight read, its gradient written; statistics, theta, bias and their gradients
    size = _SIZE[case["dtype"]]
    return dict(bytes=2 * t * (fin + fout) * size + 8 * fin * fout + 24 * fout, flops=6 * t * fin * fout)


def tolerance(case):
    kind = case["kind"]
    if kind == "codec":
        return "exact"  # words, and sums of small dyadic values scaled once
    if kind in ("head", "vlut", "packed"):
        # exact products, 32-bit sums of up to 4096 terms: 5e-8 to 1e-7 off 64 bits
        return dict(rel=1e-6, max=1e-5)
    if case["dtype"] == "f32":
        # fp32 products of up to 3072 terms: 1e-7 to 2e-7 off 64 bits, the theta gradient (which cancels) 6e-7
        return dict(rel=4e-6, max=4e-5)
    # bf16 weights and results: 2.4e-3 off 64 bits
    return dict(rel=1e-2, max=5e-2)


# ---------------------------------------------------------------------------
# the results in 64 bits, in plain torch
# ---------------------------------------------------------------------------
_EPS = 2.0 ** -23
_CHUNK = 1 << 20


def _round(x):
    return torch.floor((x - torch.sign(x) * _EPS) + 0.5)


def _d8(x):
    """The D8 point of each row of x: every coordinate rounded and, if the
    sum is odd, the worst one stepped (up where x_k >= f_k >= 0, else down)."""
    f = _round(x)
    odd = f.sum(-1).remainder(2.0) != 0
    k = (x - f).abs().argmax(-1, keepdim=True)
    xk, fk = x.gather(-1, k), f.gather(-1, k)
    step = torch.where((xk >= 0) & (fk < xk), 1.0, -1.0)
    return f.scatter_add(-1, k, torch.where(odd[:, None], step, torch.zeros_like(step)))


def _project(x):
    """The nearest E8 point of each fp32 row (the D8 + 1/2 one on a tie)."""
    y0, y1 = _d8(x), _d8(x - 0.5) + 0.5
    xd = x.double()
    near = (xd - y0.double()).square().sum(-1) < (xd - y1.double()).square().sum(-1)
    return torch.where(near[:, None], y0, y1)


def _basis():
    G = torch.zeros(8, 8, dtype=torch.float64)
    G[0, 0] = 2.0
    for j in range(1, 7):
        G[j - 1, j], G[j, j] = -1.0, 1.0
    G[:, 7] = 0.5
    return G


def _encode(x, q, M):
    """Digits [n, M, 8] of the fp32 rows of x."""
    inv = torch.linalg.inv(_basis()).mul(2).round().div(2).to(x.device)
    out = torch.empty((x.shape[0], M, 8), dtype=torch.uint8, device=x.device)
    for i in range(0, x.shape[0], _CHUNK):
        c = x[i:i + _CHUNK].float()
        for m in range(M):
            out[i:i + _CHUNK, m] = (_project(c).double() @ inv.T).round().remainder(q).to(torch.uint8)
            c = c / q
    return out


def _encode_scaled(x, kw, q, M):
    if kw.get("beta_row") is not None:
        x = x * kw["beta_row"].repeat_interleave(kw["blocks_per_row"])[:, None]
    elif kw["beta"] is not None:
        x = x / torch.full((1,), kw["beta"], device=x.device)  # a true division, also on the GPU
    return _encode(x, q, M)


def _words(digits, q):
    p = torch.tensor([q ** (7 - j) for j in range(8)], dtype=torch.int64, device=digits.device)
    n, M = digits.shape[:2]
    out = torch.empty((n, M), dtype=torch.int16 if q <= 4 else torch.int32, device=digits.device)
    for i in range(0, n, _CHUNK):
        out[i:i + _CHUNK] = (digits[i:i + _CHUNK].long() * p).sum(-1).to(out.dtype)
    return out.view(torch.uint16 if q <= 4 else torch.uint32)


def _digits(words, q):
    n, M = words.shape
    w = _signed(words).long() & (0xffff if q <= 4 else 0xffffffff)
    p = torch.tensor([q ** (7 - j) for j in range(8)], dtype=torch.int64, device=words.device)
    return ((w[..., None] // p) % q).to(torch.uint8)


def _decode(digits, q):
    """sum_m q^m (G b_m - q P(G b_m / q)), fp64 [n, 8]."""
    n, M = digits.shape[:2]
    G = _basis().to(digits.device)
    out = torch.zeros((n, 8), dtype=torch.float64, device=digits.device)
    for i in range(0, n, _CHUNK):
        for m in range(M):
            p = digits[i:i + _CHUNK, m].double() @ G.T
            out[i:i + _CHUNK] += q ** m * (p - q * _project((p / q).float()).double())
    return out


def _unscale(v, kw):
    if kw.get("beta_row") is not None:
        return v / kw["beta_row"].double().repeat_interleave(kw["blocks_per_row"])[:, None]
    return v if kw["beta"] is None else v * float(torch.tensor(kw["beta"], dtype=torch.float32))


def _step64(layer, x, gy=None):
    """The layer's forward (and, with gy, its gradients) with all sums in 64
    bits; the scaled weight that chooses the lattice points is fp32."""
    W = layer.weight.detach()
    qm = 16.0
    hi = torch.minimum((_DELTA0 * (qm - 1)) / (2 * _GINV * layer.xmax_ema),
                       (_DELTA0 * (qm - 1)) / (2 * _ETA * _GINV * layer.sigma_ema))
    lo = torch.minimum((_DELTA0 / qm) / (_ETA * _GINV * layer.sigma_ema), hi * 0.9)
    s = torch.sigmoid(layer.theta_beta.detach().double())
    beta = lo + s.float() * (hi - lo)
    Q = _decode(_encode((W * beta[:, None]).view(-1, 8), 4, 2), 4).view(W.shape)
    b = beta.double()[:, None]
    Wq = (Q / b).clamp(-_CLIP, _CLIP)
    x = x.detach().double()
    y = x @ Wq.T + layer.bias.detach().double()
    if gy is None:
        return y
    gy = gy.double()
    g = (gy.T @ x) * ((Q / b).abs() <= _CLIP)
    dbeta = (g / b * W.double() - g * Q / (b * b)).sum(1)
    return dict(y=y, dx=gy @ Wq, dW=g, dtheta=dbeta * (hi - lo).double() * s * (1 - s), db=gy.sum(0))


def exact(case, seed):
    kind = case["kind"]
    if kind == "graph":  # its inputs without the capture
        return exact(dict(case, kind="qat"), seed)
    state = prepare(case, seed)
    if kind == "codec":
        q, M, kw = case["q"], case["M"], state["kw"]
        if case["op"] == "decode":
            return _unscale(_decode(_digits(state["words"], q), q), kw)
        digits = _encode_scaled(state["x"].float(), kw, q, M)
        words = _signed(_words(digits, q))
        return words if case["op"] == "encode" else (words, _unscale(_decode(digits, q), kw))
    if kind in ("vlut", "packed"):
        raw, x = (state["raw"], state["act"]) if kind == "vlut" else (state["tensors"]["words"], state["x"])
        rows, kb, M = raw.shape
        w = _decode(_digits(raw.reshape(-1, M), 4), 4).view(rows, kb * 8)
        if kind == "vlut":
            return (x.double() @ w.T) * state["scale"].double()
        y = (x.double() @ w.T) / state["tensors"]["beta"].double()
        return y + state["tensors"]["bias"].double() if case["bias"] else y
    if kind == "head":
        return _step64(state["layer"], state["x"])
    return _step64(state["layer"], state["x"], state["gy"])
