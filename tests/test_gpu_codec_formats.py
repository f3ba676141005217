"""The table codec's fixed-format kernels: bf16, per-row betas, dividing betas."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _both(fn):
    """fn() on the fixed-format table kernel and on the generic kernel."""
    from coset_amd import _lib
    out = []
    try:
        for path, plain in ((2, True), (1, False)):
            _lib.set_codec_path(path)
            _lib.set_codec_plain(plain)
            r = fn()
            out.append(r if isinstance(r, tuple) else (r,))
    finally:
        _lib.set_codec_path(0)
        _lib.set_codec_plain(True)
    for a, b in zip(*out):
        a, b = (v.view(torch.int16 if v.element_size() == 2 else torch.int32) for v in (a, b))
        assert torch.equal(a, b)
    return out[0]


def _x(n, seed, zeros=True):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = 2 * torch.randn(n, 8, device="cuda", generator=g)
    if zeros and n > 4:
        x[1] = 0.0
        x[2, ::2] = 0.0
        x[3] = torch.tensor([0.5, -0.5, 1.5, -2.5, 1e-30, -0.0, 3e-39, 2.0], device="cuda")
    return x


@pytest.mark.parametrize("q,M", [(4, 1), (4, 2), (2, 3), (2, 4)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,per_row", [(1, 1), (3, 21), (129, 512), (40, 65)])
def test_per_row_betas(q, M, dt, rows, per_row):
    """Encode, decode and round trip with stored per-row betas (ordinary, zero,
    negative, tiny, huge, non-finite) and a clip, against the generic kernel
    bit for bit in both output types."""
    import coset_amd as ca
    n = rows * per_row
    x = _x(n, n).to(dt)
    beta = 0.5 + torch.rand(rows, device="cuda")
    odd = torch.tensor([1e-30, 1e30, -0.7, float("inf"), 0.0, 3e38, 1e-44, float("nan")], device="cuda")
    k = min(rows, len(odd))
    if rows > 1:
        beta[:k] = odd[:k]
    kw = dict(beta_row=beta, blocks_per_row=per_row)
    words = _both(lambda: ca.hnlq_encode(x, q, M, **kw))[0]
    for od in (torch.float32, torch.bfloat16):
        for clip in (float("inf"), 1.25):
            _both(lambda: ca.hnlq_decode(words, q, M, clip=clip, out_dtype=od, **kw))
            _both(lambda: ca.hnlq_roundtrip(x, q, M, clip=clip, out_dtype=od, **kw))
        _both(lambda: ca.hnlq_decode(words, q, M, clip=0.0, out_dtype=od, **kw))


@pytest.mark.parametrize("q,M", [(4, 2), (4, 3), (2, 4)])
@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("beta", [None, 0.25, 0.3, 0.02, 7.1, 1e-7, 1e7])
def test_codec_betas_and_dtypes(q, M, dt, beta):
    """No scale, powers of two, and betas that divide (one inside, two outside
    the fixed-format kernel's range), values from denormal to 2^21 and beyond,
    infinities and NaN: bit for bit the generic kernel's."""
    import coset_amd as ca
    n = 3000
    x = _x(n, 5)
    x *= torch.exp2(torch.randint(-30, 20, (n, 1), device="cuda").float())
    x[7, 0], x[8, 1], x[9, 2] = float("inf"), float("nan"), 1e38
    x = x.to(dt)
    words = _both(lambda: ca.hnlq_encode(x, q, M, beta))[0]
    _both(lambda: ca.hnlq_roundtrip(x, q, M, beta))
    if dt == torch.float32:
        _both(lambda: ca.hnlq_encode(x, q, M, beta, return_codes=True))
    for od in (torch.float32, torch.bfloat16):
        _both(lambda: ca.hnlq_decode(words, q, M, beta, out_dtype=od))


def test_dividing_beta_matches_oracle():
    """x / beta through the shared reciprocal against the oracle's division."""
    import coset_amd as ca
    from coset_amd import _lib
    x = 3 * torch.randn(20000, 8, device="cuda")
    try:
        _lib.set_codec_path(2)
        for beta in (0.3, 0.02, 1.7, 123.4):
            b = float(np.float32(beta))
            words = ca.hnlq_encode(x * beta, 4, 2, b)
            codes = O.e8_encode((x * beta).cpu().numpy(), 4, 2, b)
            assert np.array_equal(words.cpu().numpy().astype(np.uint32), O.pack_words(codes, 4))
    finally:
        _lib.set_codec_path(0)


@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 19) + 77, (6 << 20) - 1, (6 << 20) + 1])
def test_sizes_around_the_dispatch_lines(n):
    """The natural route below and above each line (table kernel, counter
    tiles) equals the generic kernel."""
    import coset_amd as ca
    from coset_amd import _lib
    x = _x(n, 9)
    got = ca.hnlq_roundtrip(x, 4, 2, None)
    words = ca.hnlq_encode(x, 4, 2, None)
    dec = ca.hnlq_decode(words, 4, 2, None)
    try:
        _lib.set_codec_path(1)
        want = ca.hnlq_roundtrip(x, 4, 2, None)
    finally:
        _lib.set_codec_path(0)
    s = torch.int16
    assert torch.equal(got[0].view(s), want[0].view(s)) and torch.equal(words.view(s), want[0].view(s))
    assert torch.equal(got[1], want[1]) and torch.equal(dec, want[1])


@pytest.mark.parametrize("q,M", [(4, 2), (2, 3)])
@pytest.mark.parametrize("n", [1 << 21, (1 << 21) + 1, (1 << 21) + 1023 * 1024 + 3, (3 << 20) + 1025])
def test_float_codes_from_the_tile_counter(q, M, n):
    """Encode and round trip with float codes from their counter line on
    (tiles of one block per thread), last tiles full and ragged: bit for bit
    the grid stride's outputs, every element written."""
    import coset_amd as ca
    from coset_amd import _lib
    x = _x(n, 11)
    out = []
    try:
        for dynamic in (True, False):
            _lib.set_codec_dynamic(dynamic)
            rt = torch.full((n, M), -1, dtype=torch.int16, device="cuda")
            rc = torch.full((n, M, 8), -1.0, device="cuda")
            dec = torch.full((n, 8), float("nan"), device="cuda")
            w, c = ca.hnlq_encode(x, q, M, None, return_codes=True)
            _lib.call("coset_e8_hnlq_roundtrip", x.data_ptr(), _lib.F32, n, _lib.SCALE_NONE, 1.0, None, 0, 0.0, None, 0,
                      q, M, 1, rt.data_ptr(), rc.data_ptr(), dec.data_ptr(), _lib.F32, _lib.stream_of(x))
            out.append((w.view(torch.int16), c, rt, rc, dec))
    finally:
        _lib.set_codec_dynamic(True)
    for a, b in zip(*out):
        assert torch.equal(a, b)
    assert torch.equal(out[0][0], out[0][2]) and torch.equal(out[0][1], out[0][3])
    assert (out[0][3] >= 0).all() and torch.isfinite(out[0][4]).all()


@pytest.mark.parametrize("q,M,skip", [(4, 2, 1), (2, 4, 1), (2, 4, 2), (2, 3, 1), (4, 1, 1)])
def test_words_that_start_inside_a_load(q, M, skip):
    """Words at an address that is no multiple of a block's (a view into a
    larger buffer): decoded, and written through the C ABI, as elsewhere."""
    import coset_amd as ca
    from coset_amd import _lib
    n = (1 << 19) + 5                 # the table kernel's sizes for every mode
    x = _x(n, 9)
    words = ca.hnlq_encode(x, q, M, 0.25)
    buf = torch.zeros(n * M + skip, dtype=torch.int16, device="cuda")
    buf[skip:] = words.view(torch.int16).reshape(-1)
    view = buf[skip:].view(n, M)
    assert view.data_ptr() % (2 * M) != 0 or M == 1 or M == 3
    for od in (torch.float32, torch.bfloat16):
        want = ca.hnlq_decode(words, q, M, 0.25, out_dtype=od)
        assert torch.equal(ca.hnlq_decode(view.view(torch.uint16), q, M, 0.25, out_dtype=od), want)
    if view.data_ptr() % 4 == 0:      # the entry points take packed words from 4-byte addresses on
        view.zero_()
        _lib.call("coset_e8_hnlq_encode", _lib.ptr(x), _lib.F32, n, _lib.SCALE_CODEC, 0.25, None, 0, None, 0, q, M,
                  view.data_ptr(), None, _lib.stream_of(x))
        assert torch.equal(view, words.view(torch.int16))


@pytest.mark.parametrize("op,n,q,M,dt,beta,table", [
    ("encode", 300000, 4, 2, torch.float32, 0.25, False), ("encode", 300000, 4, 1, torch.bfloat16, "row", False),
    ("encode", 1 << 19, 4, 2, torch.float32, 0.3, True), ("encode", 1 << 19, 4, 2, torch.bfloat16, None, False),
    ("encode", 800000, 4, 1, torch.bfloat16, None, False), ("encode", (1 << 20) + 8, 4, 2, torch.bfloat16, None, True),
    ("roundtrip", 600000, 4, 1, torch.bfloat16, None, False), ("roundtrip", 600000, 4, 2, torch.float32, 0.3, True),
    ("roundtrip", 600000, 2, 3, torch.float32, "row", True), ("decode", 300000, 4, 2, torch.bfloat16, "row", True),
    ("decode", 200000, 4, 2, torch.float32, None, False)])
def test_kernel_of_a_call(op, n, q, M, dt, beta, table):
    """Which kernel takes a call of 2^18 to 2^20 blocks (both give the same
    bits): the names a profiler sees."""
    from torch.profiler import ProfilerActivity, profile
    import coset_amd as ca
    n = n // 8 * 8
    x = torch.randn(n, 8, device="cuda").to(dt)
    kw = dict(beta=beta)
    if beta == "row":
        kw = dict(beta_row=torch.rand(n // 8, device="cuda") + 0.5, blocks_per_row=8)
    words = ca.hnlq_encode(x, q, M, **kw)
    fn = {"encode": lambda: ca.hnlq_encode(x, q, M, **kw), "roundtrip": lambda: ca.hnlq_roundtrip(x, q, M, **kw),
          "decode": lambda: ca.hnlq_decode(words, q, M, out_dtype=dt, **kw)}[op]
    fn()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA]) as p:
        fn()
        torch.cuda.synchronize()
    names = [e.key for e in p.key_averages()]
    assert any("hnlq" in k for k in names), names
    assert any("hnlq_plain_kernel" in k or "hnlq_lut_kernel" in k for k in names) == table, names
