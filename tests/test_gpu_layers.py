"""The layer building blocks one by one (dense products, norms with convolution, window attention, linear attention,
sinusoidal embedding), each against its plain statement, in both number formats and at awkward sizes.  Inputs are made
so that a mistake shows: a key at the very edge of a window outweighs all others, states decay slowly."""
import ctypes

import numpy as np
import pytest

import kugilix_model as km
import kugilix_plain as plain
from test_host_rules import FORMS

pytestmark = pytest.mark.gpu

FORMATS = [False, True]  # f32


@pytest.fixture
def dev(torch_gpu):
    return Device(torch_gpu)


class Device:
    def __init__(self, torch):
        self.torch = torch
        self.stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def act(self, x, f32):
        """activations in the format under test; returns (tensor, the values it holds)"""
        x = np.ascontiguousarray(x, np.float32)
        if f32:
            return self.f(x), x.astype(np.float64)
        return self.torch.from_numpy(x).cuda().to(self.torch.bfloat16), km.bf16(x).astype(np.float64)

    def f(self, x):
        return self.torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda()

    def empty(self, shape, f32, fill=float("nan")):
        return self.torch.full(shape, fill, dtype=self.torch.float32 if f32 else self.torch.bfloat16, device="cuda")

    def host(self, t):
        self.torch.cuda.synchronize()
        return t.float().cpu().numpy().astype(np.float64)


def limit(f32):
    return 2e-5 if f32 else 0.012


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("tokens", [1, 2, 33, 65, 130, 300])
@pytest.mark.parametrize("shape", [(70, 90, 50), (300, 1536, 520)], ids=str)
def test_dense_two_segments(awq, lib, dev, f32, tokens, shape):
    """[A; B] in one block: silu on part of A's rows, xIELU on B's, each with an input of its own"""
    na, k, nb = shape
    print("dense", shape, tokens, f32, flush=True)
    rng = np.random.default_rng(tokens)
    up = lambda v, m: (v + m - 1) // m * m
    kp, row_b = up(k, 64), up(na, 256)
    rows = row_b + up(nb, 256)
    block = dev.torch.zeros(lib.awq_dense_weight_bytes(rows, kp, f32), dtype=dev.torch.uint8, device="cuda")
    wa, wb = km.bf16(rng.standard_normal((na, k)) / k ** 0.5), km.bf16(2 * rng.standard_normal((nb, k)) / k ** 0.5)
    for w, r0 in ((wa, 0), (wb, row_b)):
        d, _ = dev.act(w, False)
        awq.check(lib.awq_dense_pack(d.data_ptr(), 0, w.shape[0], k, block.data_ptr(), kp, r0, 0, f32, dev.stream))
    pad = lambda x: np.pad(x, ((0, 0), (0, kp - k)))
    xa, va = dev.act(pad(rng.standard_normal((tokens, k))), f32)
    xb, vb = dev.act(pad(rng.standard_normal((tokens, k))), f32)
    ya, yb = dev.empty((tokens, na + 3), f32), dev.empty((tokens, nb), f32)
    ws = dev.empty((1 << 22,), True)
    p, q = 0.4, -0.3
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), kp, tokens, 2, awq.DENSE_STORE
    sp = lambda z: float(plain.softplus(np.float64(z)))
    a.segment[0] = awq.AwqDenseSegment(xa.data_ptr(), ya.data_ptr(), kp, na + 3, 0, na, awq.ACT_SILU, na // 2, 0, 0)
    a.segment[1] = awq.AwqDenseSegment(xb.data_ptr(), yb.data_ptr(), kp, nb, row_b, nb, awq.ACT_XIELU, 0, sp(p), 0.5 + sp(q))
    a.workspace, a.workspace_floats = ws.data_ptr(), ws.numel()
    awq.check(lib.awq_dense(ctypes.byref(a), f32, dev.stream))
    za, zb = va[:, :k] @ wa.T, vb[:, :k] @ wb.T
    za[:, :na // 2] = plain.silu(za[:, :na // 2])
    got = dev.host(ya)
    assert km.rms_error(got[:, :na], za) < limit(f32) and np.isnan(got[:, na:]).all()
    assert km.rms_error(dev.host(yb), plain.xielu(zb, p, q)) < limit(f32)
    # residual form, with and without an addend; and as floats
    for addend in (None, rng.standard_normal((tokens, na))):
        y0 = rng.standard_normal((tokens, na))
        y = dev.f(y0)
        ad = dev.f(addend) if addend is not None else None
        a.n_segments, a.out, a.addend = 1, awq.DENSE_RESIDUAL, ad.data_ptr() if ad is not None else None
        a.segment[0] = awq.AwqDenseSegment(xa.data_ptr(), y.data_ptr(), kp, na, 0, na, 0, 0, 0, 0)
        awq.check(lib.awq_dense(ctypes.byref(a), f32, dev.stream))
        assert km.rms_error(dev.host(y), y0 + va[:, :k] @ wa.T + (0 if addend is None else addend)) < 2e-5
    y = dev.empty((tokens, na), True)
    a.out, a.addend = awq.DENSE_F32, None
    a.segment[0] = awq.AwqDenseSegment(xa.data_ptr(), y.data_ptr(), kp, na, 0, na, 0, 0, 0, 0)
    awq.check(lib.awq_dense(ctypes.byref(a), f32, dev.stream))
    assert km.rms_error(dev.host(y), va[:, :k] @ wa.T) < 2e-5


@pytest.mark.parametrize("tokens", [1, 2, 31, 32, 33, 64, 65, 96, 127, 129, 193])
@pytest.mark.parametrize("rows,k", [(1, 64), (70, 320), (257, 1088), (300, 1856), (8200, 256), (16401, 448)])
def test_binary32_products_at_the_edges_of_tiles(awq, lib, dev, tokens, rows, k):
    """every tile of tokens, shares of k down to one, one, two and four rows per wavefront for one token, inputs and outputs that are
    not aligned to 16 bytes.  A sum of k products
    in binary32 is off by about sqrt(k) roundings of 2^-24 of its size"""
    print("binary32", tokens, rows, k, flush=True)
    rng = np.random.default_rng(rows + tokens)
    padded = (rows + 255) // 256 * 256
    block = dev.torch.zeros(padded * k, dtype=dev.torch.float32, device="cuda")
    w = (rng.standard_normal((rows, k)) / k ** 0.5).astype(np.float32)
    d = dev.f(w)
    awq.check(lib.awq_dense_pack(d.data_ptr(), 1, rows, k, block.data_ptr(), k, 0, 0, 1, dev.stream))
    x = rng.standard_normal((tokens, k)).astype(np.float32)
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    ws = dev.empty((1 << 22,), True)
    for off in (0, 1):
        xd, y = dev.empty((tokens * k + 1,), True), dev.empty((tokens * rows + 5,), True)
        xd[off:off + tokens * k] = dev.f(x).reshape(-1)
        for floats in (ws.numel(), 0):
            y.fill_(float("nan"))
            a = awq.AwqDenseArgs()
            a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
            a.segment[0] = awq.AwqDenseSegment(xd.data_ptr() + 4 * off, y.data_ptr() + 4 * off, k, rows, 0, rows, 0, 0, 0, 0)
            a.workspace, a.workspace_floats = (ws.data_ptr() if floats else None), floats
            awq.check(lib.awq_dense(ctypes.byref(a), 1, dev.stream))
            got = dev.host(y)
            assert np.isnan(got[:off]).all() and np.isnan(got[off + tokens * rows:]).all()
            got = got[off:off + tokens * rows].reshape(tokens, rows)
            assert np.abs(got - want).max() < 8 * k ** 0.5 * 2.0 ** -24


# weights that are bfloat16 numbers, all of them, all but those of one step (the first, a middle one, the last) and none; sizes at
# which no term of a product leaves binary32's range; tiles of 32 tokens with k shared by wavefronts, of 64, and of 128 rows
@pytest.mark.parametrize("tokens,rows", [(5, 300), (70, 300), (300, 8200)])
@pytest.mark.parametrize("wide", ["none", "first", "middle", "last", "one", "all"])
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -90, 2.0 ** 100])
def test_binary32_products_of_weights_in_either_format(awq, lib, dev, tokens, rows, wide, scale):
    print("binary32 weights", tokens, rows, wide, scale, flush=True)
    k = 576
    rng = np.random.default_rng(rows)
    fine = (rng.standard_normal((rows, k)) / k ** 0.5).astype(np.float32)
    w = km.bf16(fine)
    steps = {"none": [], "first": [0], "middle": [7], "last": [17], "one": [7], "all": range(18)}[wide]
    for i in steps:
        w[:, 32 * i:32 * i + 32] = fine[:, 32 * i:32 * i + 32]
    if wide == "one":
        w = km.bf16(fine)
        w[rows - 2, 230] = fine[rows - 2, 230]
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.float32, device="cuda")
    d = dev.f(w)
    awq.check(lib.awq_dense_pack(d.data_ptr(), 1, rows, k, block.data_ptr(), k, 0, 0, 1, dev.stream))
    x = (rng.standard_normal((tokens, k)) * scale).astype(np.float32)
    for floats in (0, 1 << 22):
        ws, y = dev.empty((1 << 22,), True), dev.empty((tokens, rows), True)

        def run():
            a = awq.AwqDenseArgs()
            xd = dev.f(x)
            a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
            a.segment[0] = awq.AwqDenseSegment(xd.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
            a.workspace, a.workspace_floats = (ws.data_ptr() if floats else None), floats
            awq.check(lib.awq_dense(ctypes.byref(a), 1, dev.stream))
            return dev.host(y).astype(np.float64)
        want = x.astype(np.float64) @ w.T.astype(np.float64)
        # 36 sums of 16 products: 36 roundings of 2^-24 of partial sums, which are below 6 (2.5 million outputs of rms 1) and, in the
        # mean square over all, sqrt(i / 36) behind the i-th: 2^-24 sqrt(18).  What is left out of a product is 2^-30 of it.
        before = run()
        assert np.abs(before - want).max() < 36 * 6 * 2.0 ** -24 * scale
        assert np.sqrt(np.mean((before - want) ** 2)) < 18 ** 0.5 * 2.0 ** -24 * scale
        # what is not finite stays with its token (the others have the bits they had), and is what products and sums of binary32 make of it
        keep = x.copy()
        x[1, 3], x[2, 100], x[2, 101], x[3, 575], x[4, 40] = np.inf, np.inf, -np.inf, np.nan, -np.inf
        with np.errstate(invalid="ignore"):
            want = x.astype(np.float64) @ w.T.astype(np.float64)
        got = run()
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.sign(got[1]), np.sign(want[1])) and np.isinf(got[[1, 4]]).all()
        rest = [t for t in range(tokens) if not 1 <= t <= 4]
        assert np.array_equal(got[rest], before[rest])
        x = keep


def binary32_product(awq, lib, dev, w, x, floats):
    """x w^T by awq_dense in binary32, with a workspace of so many floats"""
    (rows, k), tokens = w.shape, len(x)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.float32, device="cuda")
    wd, xd, y, ws = dev.f(w), dev.f(x), dev.empty((tokens, rows), True), dev.empty((max(1, floats),), True)
    awq.check(lib.awq_dense_pack(wd.data_ptr(), 1, rows, k, block.data_ptr(), k, 0, 0, 1, dev.stream))
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
    a.segment[0] = awq.AwqDenseSegment(xd.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
    a.workspace, a.workspace_floats = (ws.data_ptr() if floats else None), floats
    awq.check(lib.awq_dense(ctypes.byref(a), 1, dev.stream))
    return dev.host(y)


# Operands whose last bits are below bfloat16's range, 2^-133.  288 instructions of two products, each rounding their sum and partial sums that are
# sqrt(i / 288) of the result's rms in the mean square: sqrt(288) x 2^-24 at most.
@pytest.mark.parametrize("tokens,rows", [(5, 300), (70, 300), (300, 1100)])
@pytest.mark.parametrize("of_w,of_x", [(0, -110), (0, -118), (0, -124), (-120, 0), (-60, -60)])
def test_binary32_products_of_tiny_operands(awq, lib, dev, tokens, rows, of_w, of_x):
    print("tiny operands", tokens, rows, of_w, of_x, flush=True)
    rng = np.random.default_rng(rows)
    w = (rng.standard_normal((rows, 576)) * 2.0 ** of_w).astype(np.float32)
    x = (rng.standard_normal((tokens, 576)) * 2.0 ** of_x).astype(np.float32)
    want = x.astype(np.float64) @ w.T.astype(np.float64)
    for floats in (0, 1 << 22):
        off = binary32_product(awq, lib, dev, w, x, floats) - want
        assert np.sqrt(np.mean(off ** 2)) < 288 ** 0.5 * 2.0 ** -24 * np.sqrt(np.mean(want ** 2))


# A product of two binary32 numbers rounds by 2^-24 of itself; their bfloat16 terms' sums by 2^-24 of what is 2^-6 of it, five times, and
# what is left out is 2^-30: an eighth more.  Where all terms have one sign, what were left out of the products would add up: roundings
# go either way, and the mean of many outputs' errors is far below one.  0x3f80ffff has the largest second and third terms.
@pytest.mark.parametrize("tokens,rows", [(5, 300), (33, 300), (70, 300), (300, 8200)])
@pytest.mark.parametrize("k", [64, 576])
def test_no_bits_of_a_binary32_product_are_left_out(awq, lib, dev, tokens, rows, k):
    print("binary32 bits", tokens, rows, k, flush=True)
    rng = np.random.default_rng(rows + k)
    worst = np.array([0x3f80ffff], np.uint32).view(np.float32)[0]
    w, x = rng.standard_normal((rows, k)).astype(np.float32), rng.standard_normal((tokens, k)).astype(np.float32)
    one = np.zeros_like(x)
    at = rng.integers(0, k, tokens)
    one[np.arange(tokens), at] = x[np.arange(tokens), at]
    for floats in (0, 1 << 22):
        for wv, xv in ((w, one), (np.full_like(w, worst), np.where(one != 0, worst, np.float32(0)))):
            want = xv.astype(np.float64) @ wv.T.astype(np.float64)
            assert (np.abs(binary32_product(awq, lib, dev, wv, xv, floats) - want) <= 1.125 * 2.0 ** -24 * np.abs(want)).all()
        wv, xv = np.abs(w), np.abs(x)
        want = xv.astype(np.float64) @ wv.T.astype(np.float64)
        off = np.mean((binary32_product(awq, lib, dev, wv, xv, floats) - want) / want)
        print("mean %.3f x 2^-24" % (off * 2 ** 24), flush=True)
        assert abs(off) < 0.3 * 2.0 ** -24


@pytest.mark.parametrize("k", [64, 192, 320, 448, 1024, 1088, 1152, 1536, 1792, 2048, 2112, 2560, 3072, 3584, 4160, 8192, 8256, 12352])
@pytest.mark.parametrize("rows", [1, 9, 1000, 2048, 2049])
def test_products_of_one_token(awq, lib, dev, rows, k):
    """8 and 16 rows per workgroup, 4, 8 and 16 wavefronts, runs of whole turns and every kind of rest, wavefronts without a
    step.  The operands are exact: a sum of k products in binary32 is off by about sqrt(k) roundings of 2^-24 of its size"""
    print("one token", rows, k, flush=True)
    rng = np.random.default_rng(rows + k)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((1, k)), False)
    y = dev.empty((2, rows), True)
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, 1, 1, awq.DENSE_F32
    a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
    awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
    got = dev.host(y)
    assert np.isnan(got[1]).all()
    assert np.abs(got[0] - (xv @ wv.T)[0]).max() < 8 * k ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("tokens", [2, 15, 16, 17, 24, 25, 31, 32])
@pytest.mark.parametrize("rows,k", [(1, 64), (47, 320), (300, 1088), (264, 8256), (8200, 192), (16400, 64)])
def test_products_of_few_tokens(awq, lib, dev, tokens, rows, k):
    """one and two tiles of 16 tokens, 16 and 32 rows per workgroup, 4, 8 and 16 wavefronts, rests of k.  The operands are
    exact: a sum of k products in binary32 is off by about sqrt(k) roundings of 2^-24 of its size"""
    print("few tokens", tokens, rows, k, flush=True)
    rng = np.random.default_rng(rows + tokens)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((tokens, k)), False)
    ws = dev.empty((1 << 20,), True)
    y = dev.empty((tokens + 1, rows), True)
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
    a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
    a.workspace, a.workspace_floats = ws.data_ptr(), ws.numel()
    awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
    got = dev.host(y)
    assert np.isnan(got[tokens]).all()
    assert np.abs(got[:tokens] - xv @ wv.T).max() < 8 * k ** 0.5 * 2.0 ** -24


@pytest.mark.parametrize("tokens", [2, 16, 17, 20, 32])
@pytest.mark.parametrize("k", [192, 1088, 8256])
def test_few_tokens_on_many_rows(awq, lib, dev, tokens, k):
    """32 rows per workgroup with 4, 8 and 16 wavefronts, for every kind of output: gated pairs, biases, another type, a residual.
    17,152 padded rows: the few-token kernel up to 8,256 inputs and 20 tokens at least, by its estimate against the other one."""
    torch = dev.torch
    print("few tokens, many rows", tokens, k, flush=True)
    rows0, glu, plain_rows, sig = [0, 16032, 16320], 8009, 261, 300   # at multiples of 32
    total = 17152
    gen = torch.Generator(device="cuda")
    gen.manual_seed(tokens + k)
    block = torch.zeros(total * k, dtype=torch.bfloat16, device="cuda")
    w = {n: (torch.randn(r, k, generator=gen, device="cuda") / k ** 0.5).bfloat16() for n, r in
         (("gate", glu), ("up", glu), ("plain", plain_rows), ("sig", sig))}
    for n, r0, form in (("gate", 0, 1), ("up", 0, 2), ("plain", rows0[1], 0), ("sig", rows0[2], 0)):
        awq.check(lib.awq_dense_pack_form(w[n].data_ptr(), 0, w[n].shape[0], k, block.data_ptr(), k, r0, 0, form, 0, dev.stream))
    x = torch.randn(tokens, k, generator=gen, device="cuda").bfloat16()
    z = {n: (x.double() @ v.double().t()).cpu().numpy() for n, v in w.items()}
    y = {n: dev.empty((tokens + 1, r + 3), n == "plain") for n, r in (("glu", glu), ("plain", plain_rows), ("sig", sig))}
    bias = torch.randn(sig, generator=gen, device="cuda")
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 3, awq.DENSE_STORE
    for i, (n, rows, act) in enumerate((("glu", 16032, awq.ACT_GLU), ("plain", plain_rows, awq.ACT_NONE), ("sig", sig, awq.ACT_SIGMOID))):
        a.segment[i] = awq.AwqDenseSegment(x.data_ptr(), y[n].data_ptr(), k, y[n].shape[1], rows0[i], rows, act)
    a.segment[0].glu_rows, a.segment[1].y_f32, a.segment[2].bias = glu, 1, bias.data_ptr()
    awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
    want = {"glu": plain.silu(z["gate"]) * z["up"], "plain": z["plain"], "sig": plain.sigmoid(z["sig"] + bias.double().cpu().numpy())}
    exact = 8 * k ** 0.5 * 2.0 ** -24  # a sum of k exact products in binary32; a result in bfloat16 is off by 2^-9 of its size more
    for n, v in want.items():
        got = dev.host(y[n])
        assert np.isnan(got[tokens]).all() and np.isnan(got[:, v.shape[1]:]).all(), n
        off = np.abs(got[:tokens, :v.shape[1]] - v)
        assert np.all(off <= 4 * exact * (1 + np.abs(v)) + (0 if n == "plain" else 2.0 ** -8 * np.abs(v))), n
    # the same rows as a residual: gate and up rows lie in eights
    r = dev.f(np.zeros((tokens, 16032)))
    r.normal_(generator=gen)
    before = dev.host(r)
    a.n_segments, a.out = 1, awq.DENSE_RESIDUAL
    a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), r.data_ptr(), k, 16032, 0, 16032)
    awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
    sums = np.zeros((tokens, 16032))
    at = np.arange(glu) // 8 * 16 + np.arange(glu) % 8
    sums[:, at], sums[:, at + 8] = z["gate"], z["up"]
    assert np.abs(dev.host(r) - (before + sums)).max() < exact + 8 * 2.0 ** -24   # and the residual's own rounding


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 9, 12, 13, 37])
@pytest.mark.parametrize("tokens", [33, 129, 700])
def test_products_of_every_number_of_steps(awq, lib, dev, tokens, steps):
    """the products of many tokens go six steps of 64 inputs at a time and end anywhere; with and without shares of k.  The
    operands are exact: a sum of k products in binary32 is off by about sqrt(k) roundings of 2^-24 of its size"""
    rows, k = 300, 64 * steps
    print("steps", tokens, steps, flush=True)
    rng = np.random.default_rng(steps + tokens)
    block = dev.torch.zeros(512 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((tokens, k)), False)
    ws = dev.empty((1 << 22,), True)
    for floats in (ws.numel(), 0):
        y = dev.empty((tokens + 1, rows), True)
        a = awq.AwqDenseArgs()
        a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
        a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
        a.workspace, a.workspace_floats = (ws.data_ptr() if floats else None), floats
        awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
        got = dev.host(y)
        assert np.isnan(got[tokens]).all()
        assert np.abs(got[:tokens] - xv @ wv.T).max() < 8 * k ** 0.5 * 2.0 ** -24


# tiles of 128 and 256 rows and of 64 and 128 tokens, each alone and with its k in shares (test_host_rules.py has which is which), rows
# and tokens that end inside a tile
@pytest.mark.parametrize("rows,k,tokens", sorted(FORMS))
def test_products_of_many_tokens_in_every_form(awq, lib, dev, rows, k, tokens):
    """all three outputs; the operands are exact: a sum of k products in binary32 is off by about sqrt(k) roundings of 2^-24 of its size"""
    print("forms", rows, k, tokens, flush=True)
    rng = np.random.default_rng(rows + tokens)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((tokens, k)), False)
    want = xv @ wv.T
    ws = dev.empty((1 << 25,), True)
    exact = 8 * k ** 0.5 * 2.0 ** -24
    for out in (awq.DENSE_F32, awq.DENSE_RESIDUAL, awq.DENSE_STORE):
        y = dev.empty((tokens + 1, rows), out != awq.DENSE_STORE, fill=0.5)
        y[tokens] = float("nan")
        a = awq.AwqDenseArgs()
        a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, out
        a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
        a.workspace, a.workspace_floats = ws.data_ptr(), ws.numel()
        awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
        got = dev.host(y)
        assert np.isnan(got[tokens]).all()
        off = np.abs(got[:tokens] - want - (0.5 if out == awq.DENSE_RESIDUAL else 0.0))
        # (the residual's own rounding; a bfloat16 output has 8 bits, half a unit of the last is at most 2^-8 of its value)
        assert (off <= exact + (2.0 ** -8 * np.abs(want) if out == awq.DENSE_STORE else 8 * 2.0 ** -24)).all()


# tiles of every size with a compute unit to each and an even number of steps, which two halves of a workgroup share: as many as there
# are units and some more, rows and tokens that end inside a tile, the fewest steps
@pytest.mark.parametrize("rows,k,tokens", [(1000, 512, 129), (2048, 1024, 1000), (2048, 1024, 1100), (8200, 2176, 400), (12300, 2048, 129), (4100, 2048, 1025), (300, 640, 34)])
def test_products_whose_k_two_halves_share(awq, lib, dev, rows, k, tokens):
    print("halves", rows, k, tokens, flush=True)
    rng = np.random.default_rng(rows + tokens)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((tokens, k)), False)
    want = xv @ wv.T
    for out in (awq.DENSE_F32, awq.DENSE_RESIDUAL, awq.DENSE_STORE):
        y = dev.empty((tokens + 1, rows), out != awq.DENSE_STORE, fill=0.5)
        y[tokens] = float("nan")
        a = awq.AwqDenseArgs()
        a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, out
        a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
        awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
        got = dev.host(y)
        assert np.isnan(got[tokens]).all()
        off = np.abs(got[:tokens] - want - (0.5 if out == awq.DENSE_RESIDUAL else 0.0))
        # exact operands: about sqrt(k) roundings of 2^-24 of a sum's size; then as in the test above
        assert (off <= 8 * k ** 0.5 * 2.0 ** -24 + (2.0 ** -8 * np.abs(want) if out == awq.DENSE_STORE else 8 * 2.0 ** -24)).all()


@pytest.mark.parametrize("k", [64, 320, 512, 576])
@pytest.mark.parametrize("rows,tokens", [(2000, 2001), (8200, 1030)])
def test_products_of_few_inputs_and_many_tokens(awq, lib, dev, rows, tokens, k):
    """products whose steps are few, tiles on the device at once or not, without a workspace"""
    print("few inputs", rows, tokens, k, flush=True)
    rng = np.random.default_rng(k + rows)
    block = dev.torch.zeros((rows + 255) // 256 * 256 * k, dtype=dev.torch.bfloat16, device="cuda")
    w, wv = dev.act(rng.standard_normal((rows, k)) / k ** 0.5, False)
    awq.check(lib.awq_dense_pack(w.data_ptr(), 0, rows, k, block.data_ptr(), k, 0, 0, 0, dev.stream))
    x, xv = dev.act(rng.standard_normal((tokens, k)), False)
    y = dev.empty((tokens + 1, rows), True)
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = block.data_ptr(), k, tokens, 1, awq.DENSE_F32
    a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), k, rows, 0, rows, 0, 0, 0, 0)
    awq.check(lib.awq_dense(ctypes.byref(a), 0, dev.stream))
    got = dev.host(y)
    assert np.isnan(got[tokens]).all()
    assert np.abs(got[:tokens] - xv @ wv.T).max() < 8 * k ** 0.5 * 2.0 ** -24   # as in the test above


def test_xielu_near_zero_and_far_out(awq, lib, dev):
    """the negative branch cancels near zero: small arguments keep their relative accuracy"""
    z = np.concatenate([-np.geomspace(1e-6, 60, 200), np.geomspace(1e-6, 60, 56)]).astype(np.float32)
    w = dev.torch.zeros(256 * 64, dtype=dev.torch.float32, device="cuda")
    d = dev.f(z.reshape(256, 1))
    awq.check(lib.awq_dense_pack(d.data_ptr(), 1, 256, 1, w.data_ptr(), 64, 0, 0, 1, dev.stream))
    x = dev.f(np.eye(1, 64))
    y = dev.empty((1, 256), True)
    a = awq.AwqDenseArgs()
    a.w, a.k, a.tokens, a.n_segments, a.out = w.data_ptr(), 64, 1, 1, awq.DENSE_STORE
    sp = lambda v: float(plain.softplus(np.float64(v)))
    a.segment[0] = awq.AwqDenseSegment(x.data_ptr(), y.data_ptr(), 64, 256, 0, 256, awq.ACT_XIELU, 0, sp(0.2), 0.5 + sp(1.3))
    awq.check(lib.awq_dense(ctypes.byref(a), 1, dev.stream))
    want = plain.xielu(z.astype(np.float64), 0.2, 1.3)
    # (the function has a zero near -1 / act_neg: there the parts it is the sum of set the scale)
    assert np.all(np.abs(dev.host(y)[0] - want) <= 5e-7 * np.maximum(np.abs(want), np.abs(z)))


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
def test_embedding_with_positions(awq, lib, dev, f32):
    rng = np.random.default_rng(0)
    for width, pos0 in ((7, 0), (96, 3), (130, 70000)):
        table, vals = dev.act(rng.standard_normal((19, width)), f32)
        tokens = rng.integers(0, 19, 33).astype(np.int32)
        freq = dev.torch.tensor([10000.0 ** (-2.0 * i / width) for i in range((width + 1) // 2)], dtype=dev.torch.float64).cuda()
        ids = dev.torch.from_numpy(tokens).cuda()
        x = dev.empty((33, width), True)
        awq.check(lib.awq_embed_sinusoid(table.data_ptr(), f32, ids.data_ptr(), pos0, 33, width, 1.7, freq.data_ptr(),
                                         x.data_ptr(), dev.stream))
        want = plain.embed(tokens, vals, np.float32(1.7), pos0)
        assert np.abs(dev.host(x) - want).max() < 2e-6


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("width,groups,taps", [(96, 4, 4), (90, 5, 3), (64, 1, 1), (64, 2, 2), (1280, 2, 8), (48, 3, 11), (2048, 1, 4)])
def test_norm_and_convolution_in_portions(awq, lib, dev, f32, width, groups, taps):
    print("norm_conv", width, groups, taps, f32, flush=True)
    rng = np.random.default_rng(width)
    T, eps = 75, 0.03
    x = rng.standard_normal((T, width)).astype(np.float32) * np.linspace(0.1, 3, T, dtype=np.float32)[:, None]
    w1, w2 = 1 + 0.5 * rng.standard_normal(width), rng.standard_normal(width)
    conv = rng.standard_normal((width, taps))
    h = plain.grouped_norm(x.astype(np.float64), w1.astype(np.float32), groups, eps)
    want1, want2 = plain.causal_conv(h, conv.astype(np.float32)), plain.grouped_norm(x.astype(np.float64), w2, groups, eps)
    d_w1, d_w2, d_c = dev.f(w1), dev.f(w2), dev.f(conv)
    ld = width + 8 - width % 8
    for sizes in ([75], [1], [2], [5, 1, 3], [taps, 1], [64, 2]):
        state = [dev.empty((max(1, taps - 1), width), True) for _ in range(2)]  # NaN: nothing ahead of 0 is read
        at, i = 0, 0
        while at < T:
            n = min(sizes[i % len(sizes)], T - at)
            xs = dev.f(x[at:at + n])
            y1, y2 = dev.empty((n, ld), f32), dev.empty((n, ld), f32)
            awq.check(lib.awq_norm_conv(xs.data_ptr(), n, width, groups, eps, d_w1.data_ptr(), d_c.data_ptr(), taps,
                                        state[i & 1].data_ptr(), state[i & 1 ^ 1].data_ptr(), y1.data_ptr(), d_w2.data_ptr(),
                                        y2.data_ptr(), ld, at, f32, dev.stream))
            assert np.abs(dev.host(y1)[:, :width] - want1[at:at + n]).max() <= (1e-5 if f32 else 0.01) * np.abs(want1).max()
            assert np.abs(dev.host(y2)[:, :width] - want2[at:at + n]).max() <= (1e-5 if f32 else 0.01) * np.abs(want2).max()
            at, i = at + n, i + 1


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("n", [37, 96, 4096, 5000])
def test_gated_norm(awq, lib, dev, f32, n):
    rng = np.random.default_rng(n)
    for T in (1, 9):
        o, w = 4 * rng.standard_normal((T, n)), rng.standard_normal(n)
        ldg = n + 8 - n % 8
        g, gv = dev.act(5 * rng.standard_normal((T, ldg)), f32)
        y = dev.empty((T, ldg), f32)
        d_o, d_w = dev.f(o), dev.f(w)
        awq.check(lib.awq_gated_norm(d_o.data_ptr(), n, g.data_ptr(), ldg, d_w.data_ptr(), y.data_ptr(), ldg, n, T, 1e-3, f32,
                                     dev.stream))
        want = plain.rms(o.astype(np.float32).astype(np.float64), 1e-3) * w * plain.sigmoid(gv[:, :n])
        assert km.rms_error(dev.host(y)[:, :n], want) < (2e-6 if f32 else 0.004)


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("heads,dim,vdim", [(3, 20, 12), (2, 64, 64), (2, 128, 96), (1, 256, 40), (2, 100, 36), (1, 512, 16),
                                            (4, 9, 31), (1, 200, 8)])
def test_linear_attention(awq, lib, dev, f32, heads, dim, vdim):
    """portions of every form: token by token, chunks that are full, ragged and of one token, several chunks"""
    print("linear attention", heads, dim, vdim, f32, flush=True)
    rng = np.random.default_rng(dim)
    T = 300
    n = heads * (2 * dim + vdim)
    ldp = (n + 7) // 8 * 8
    proj, pv = dev.act(np.pad(rng.standard_normal((T, n)) * 0.5 + 0.2, ((0, 0), (0, ldp - n))), f32)
    q = pv[:, :heads * dim].reshape(T, heads, dim)
    k = pv[:, heads * dim:2 * heads * dim].reshape(T, heads, dim)
    v = pv[:, 2 * heads * dim:n].reshape(T, heads, vdim)
    decay = np.array([0.999, 0.3, 0.9, 1e-6][:heads], np.float32)
    want, S = plain.linear_attention(q, k, v, decay.astype(np.float64))
    d_decay, d_lg = dev.f(decay), dev.f(np.log2(decay.astype(np.float64)))
    dimp = (dim + 63) // 64 * 64
    for sizes in ([300], [1], [2, 15], [16], [129, 1, 2], [128], [130, 31]):
        if f32 and sizes not in ([300], [1], [2, 15]):
            continue
        state = dev.empty((heads, vdim, dimp), True)  # NaN: position 0 starts from nothing
        out, at, i = [], 0, 0
        while at < T:
            m = min(sizes[i % len(sizes)], T - at)
            o = dev.empty((m, heads * vdim), True)
            awq.check(lib.awq_linear_attention(proj[at:].data_ptr(), ldp, heads, dim, vdim, d_decay.data_ptr(), d_lg.data_ptr(),
                                               state.data_ptr(), o.data_ptr(), m, at, f32, dev.stream))
            out.append(o)
            at, i = at + m, i + 1
        got = dev.host(dev.torch.cat(out)).reshape(T, heads, vdim)
        for h in range(heads):  # per head: a head that forgets at once is small beside one that remembers
            # the operands are exact, so both forms carry (nearly) binary32
            assert km.rms_error(got[:, h], want[:, h]) < 3e-5, (sizes, h)
        s = dev.host(state)[:, :, :dim].transpose(0, 2, 1)
        for h in range(heads):
            assert np.abs(s[h] - S[h]).max() <= 3e-5 * np.abs(S[h]).max(), (sizes, h)


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("heads,dim,vdim", [(3, 9, 5), (4, 64, 40), (2, 130, 33), (1, 256, 72), (2, 300, 16), (1, 512, 17)])
def test_several_tokens_of_linear_attention_are_those_of_single_ones(awq, lib, dev, f32, heads, dim, vdim):
    """few tokens at a time, and any number where a decay of zero or a wide head leaves no chunks: the same bits.  A value that
    is infinite reaches its own column from its own token on and nothing else"""
    print("linear attention, several tokens", heads, dim, vdim, f32, flush=True)
    rng = np.random.default_rng(dim)
    T, at, n = 47, 20, heads * (2 * dim + vdim)
    x = np.pad(rng.standard_normal((T, n)) * 0.5 + 0.2, ((0, 0), (0, -n % 8)))
    x[at, 2 * heads * dim + 1] = np.inf
    proj, _ = dev.act(x, f32)
    decay = np.array([0.999, 0.3, 0.9, 1e-6][:heads], np.float32)
    d_lg = dev.f(np.log2(decay.astype(np.float64)))

    def run(sizes, decay, lg):
        state, o = dev.empty((heads, vdim, (dim + 63) // 64 * 64), True), dev.empty((T, heads * vdim), True)
        d_decay = dev.f(decay)
        t = i = 0
        while t < T:
            m = min(sizes[i % len(sizes)], T - t)
            awq.check(lib.awq_linear_attention(proj[t:].data_ptr(), proj.shape[1], heads, dim, vdim, d_decay.data_ptr(), lg, state.data_ptr(),
                                               o[t:].data_ptr(), m, t, f32, dev.stream))
            t, i = t + m, i + 1
        return dev.host(o), dev.host(state)
    for zero in (False, True):
        d, lg = (np.where(decay < 0.1, 0, decay).astype(np.float32), None) if zero else (decay, d_lg.data_ptr())
        want = run([1], d, lg)
        column = np.arange(heads * vdim) == 1
        assert np.isfinite(want[0][:at]).all() and np.isfinite(want[0][:, ~column]).all() and not np.isfinite(want[0][at:, 1]).any()
        for sizes in ([2], [3, 1, 15], [15], [9, 4]) + (([40], [47]) if zero or dim > 256 else ()):
            got = run(sizes, d, lg)
            assert np.array_equal(got[0], want[0], equal_nan=True) and np.array_equal(got[1], want[1], equal_nan=True), sizes
        if f32 and not zero:  # the chunks: inside a block, behind it, in the next pass
            for sizes in ([47], [16, 31], [30, 1]):
                got = run(sizes, d, lg)
                for x, y in ((got[0], want[0]), (got[1][:, :, :dim], want[1][:, :, :dim])):
                    fine = np.isfinite(y)
                    assert np.array_equal(np.isfinite(x), fine), sizes
                    assert np.abs(x[fine] - y[fine]).max() < 1e-5 * np.abs(y[fine]).max(), sizes


@pytest.mark.parametrize("heads,dim,vdim", [(3, 63, 5), (4, 64, 40), (2, 128, 16), (2, 130, 33), (1, 256, 72)])
@pytest.mark.parametrize("sizes", [[16], [129, 1, 2], [130, 31], [15, 17, 300]], ids=str)
def test_linear_attention_in_binary32_portions(awq, lib, dev, heads, dim, vdim, sizes):
    """chunks beside single tokens on one state; decays that leave the range of a block's factors; odd widths"""
    print("linear attention, binary32", heads, dim, vdim, sizes, flush=True)
    rng = np.random.default_rng(dim + sizes[0])
    T, n = 332, heads * (2 * dim + vdim)
    ldp = (n + 7) // 8 * 8
    proj, pv = dev.act(np.pad(rng.standard_normal((T, n)) * 0.5 + 0.2, ((0, 0), (0, ldp - n))), True)
    q, k = (pv[:, i * heads * dim:(i + 1) * heads * dim].reshape(T, heads, dim) for i in (0, 1))
    v = pv[:, 2 * heads * dim:n].reshape(T, heads, vdim)
    decay = np.array([0.999, 1e-6, 0.9, 1.0][:heads], np.float32)
    want, S = plain.linear_attention(q, k, v, decay.astype(np.float64))
    d_decay, d_lg = dev.f(decay), dev.f(np.log2(decay.astype(np.float64)))
    state = dev.empty((heads, vdim, (dim + 63) // 64 * 64), True)
    o, at, i = dev.empty((T, heads * vdim), True), 0, 0
    while at < T:
        m = min(sizes[i % len(sizes)], T - at)
        awq.check(lib.awq_linear_attention(proj[at:].data_ptr(), ldp, heads, dim, vdim, d_decay.data_ptr(), d_lg.data_ptr(),
                                           state.data_ptr(), o[at:].data_ptr(), m, at, 1, dev.stream))
        at, i = at + m, i + 1
    got, s = dev.host(o).reshape(T, heads, vdim), dev.host(state)[:, :, :dim].transpose(0, 2, 1)
    for h in range(heads):  # sums of up to 332 x 256 products in binary32, as in the test above
        assert km.rms_error(got[:, h], want[:, h]) < 3e-5
        assert np.abs(s[h] - S[h]).max() <= 3e-5 * np.abs(S[h]).max()


@pytest.mark.parametrize("heads,dim,vdim", [(8, 128, 128), (8, 64, 40), (8, 256, 72)])
@pytest.mark.parametrize("f32,T,sizes", [(0, 60, [15]), (0, 60, [2]), (0, 60, [9, 1]), (1, 60, [15]), (1, 333, [333]), (1, 333, [40, 1])], ids=str)
def test_roundings_of_linear_attention(awq, lib, dev, f32, T, sizes, heads, dim, vdim):
    """Every form that carries binary32 is as close to 64 bits as the recurrence in binary32.  An output rounds its last sum, the
    products it adds and the state's decay by 2^-25 each in the mean, and a state that remembers n tokens has been rounded n
    times, the older ones decayed: 4 x 2^-25 for an output, sqrt(n) x 2^-25 for a state, n = 256 at most here."""
    rng = np.random.default_rng(dim + T)
    n = heads * (2 * dim + vdim)
    proj, pv = dev.act(plain.silu(rng.standard_normal((T, n))), f32)
    q, k = (pv[:, i * heads * dim:(i + 1) * heads * dim].reshape(T, heads, dim) for i in (0, 1))
    v = pv[:, 2 * heads * dim:n].reshape(T, heads, vdim)
    decay = (1.0 - 2.0 ** (-1.0 - 7.0 * np.arange(heads) / heads)).astype(np.float32)
    want, S = plain.linear_attention(q, k, v, decay.astype(np.float64))
    d_decay, d_lg = dev.f(decay), dev.f(np.log2(decay.astype(np.float64)))
    state, o, at, i = dev.empty((heads, vdim, (dim + 63) // 64 * 64), True), dev.empty((T, heads * vdim), True), 0, 0
    while at < T:
        m = min(sizes[i % len(sizes)], T - at)
        awq.check(lib.awq_linear_attention(proj[at:].data_ptr(), n, heads, dim, vdim, d_decay.data_ptr(), d_lg.data_ptr(), state.data_ptr(),
                                           o[at:].data_ptr(), m, at, f32, dev.stream))
        at, i = at + m, i + 1
    got, s = dev.host(o).reshape(T, heads, vdim), dev.host(state)[:, :, :dim].transpose(0, 2, 1)
    off = lambda x, y: np.linalg.norm(x - y) / np.linalg.norm(y)
    worst = max(off(got[:, h], want[:, h]) for h in range(heads)), max(off(s[h], S[h]) for h in range(heads))
    print("roundings", dim, f32, T, sizes, "%.1e %.1e" % worst, flush=True)
    assert worst[0] < 4 * 2.0 ** -25 and worst[1] < min(T, 256) ** 0.5 * 2.0 ** -25


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("heads,dim,vdim", [(3, 24, 16), (2, 128, 96), (1, 256, 40), (2, 100, 36), (4, 64, 8), (80, 16, 8)])
def test_segments_of_linear_attention(awq, lib, dev, f32, heads, dim, vdim):
    """segments side by side, by room for none, two, three and all of them: whole and ragged last ones, behind a state.  In bfloat16 rows that are not
    whole pieces have none; 80 heads leave three.  Bound: as in test_linear_attention"""
    print("segments of linear attention", heads, dim, vdim, f32, flush=True)
    rng = np.random.default_rng(dim)
    T, n = 1700, heads * (2 * dim + vdim)
    ldp = (n + 7) // 8 * 8
    proj, pv = dev.act(np.pad(rng.standard_normal((T, n)) * 0.5 + 0.2, ((0, 0), (0, ldp - n))), f32)
    q, k = (pv[:, i * heads * dim:(i + 1) * heads * dim].reshape(T, heads, dim) for i in (0, 1))
    v = pv[:, 2 * heads * dim:n].reshape(T, heads, vdim)
    decay = np.array(([0.999, 0.3, 0.9, 1e-6] * heads)[:heads], np.float32)
    want, S = plain.linear_attention(q, k, v, decay.astype(np.float64))
    d_decay, d_lg = dev.f(decay), dev.f(np.log2(decay.astype(np.float64)))
    dimp = (dim + 63) // 64 * 64
    room = heads * (vdim + 1) * dimp
    # A weight's two terms of 8 bits are 2^-17 off, and a head of 16 inputs that forgets at once cancels up to 4.2 to 1 in an output: 3.2e-5, one chunk
    # after the other.  Beside that a segment adds two roundings of binary32 to the states: 2e-7.
    for sizes, rooms in (([T], (0, 16, 3, 2, 1)), ([1, 1100, 599], (0, 16)), ([1152, 548], (0, 16))):
        for segments in rooms:
            ws, state, o = dev.empty((max(4, segments * room),), True), dev.empty((heads, vdim, dimp), True), dev.empty((T, heads * vdim), True)
            at = i = 0
            while at < T:
                m = min(sizes[i % len(sizes)], T - at)
                awq.check(lib.awq_linear_attention_segments(proj[at:].data_ptr(), ldp, heads, dim, vdim, d_decay.data_ptr(), d_lg.data_ptr(),
                                                            state.data_ptr(), o[at:].data_ptr(), m, at, f32, ws.data_ptr(), segments * room, dev.stream))
                at, i = at + m, i + 1
            got, s = dev.host(o).reshape(T, heads, vdim), dev.host(state)[:, :, :dim].transpose(0, 2, 1)
            off = [km.rms_error(got[:, h], want[:, h]) for h in range(heads)]
            alone = off if segments == 0 else alone
            assert max(off) < (3e-5 if dim > 16 else 3.3e-5), (sizes, segments)
            for h in range(heads):
                assert off[h] < alone[h] + 2e-7, (sizes, segments, h)
                assert np.abs(s[h] - S[h]).max() <= 3e-5 * np.abs(S[h]).max(), (sizes, segments, h)


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("segments", [16, 3])
def test_segments_behind_a_state_that_is_not_finite(awq, lib, dev, f32, segments):
    """Infinities and NaN are where one piece has them, whichever decay brings them along: powers that binary32 holds exactly, that it does not hold
    (0.3, and 1.5 over a state of zero), and one that leaves of 1e36 what only 64 bits have a factor for.  Bound: as in test_linear_attention"""
    print("segments behind infinities", segments, f32, flush=True)
    rng = np.random.default_rng(segments)
    decay = np.array([0.5, 0.75, 0.9995, 0.3, 1.5, 0.86, 0.9], np.float32)
    heads, dim, vdim, T, pos0 = len(decay), 64, 16, 1700, 64
    n = heads * (2 * dim + vdim)
    x = rng.standard_normal((T, n)) * 0.5 + 0.2
    k = x[:, heads * dim:2 * heads * dim].reshape(T, heads, dim).copy()
    k[:, 4:6] = 0.0
    x[:, heads * dim:2 * heads * dim] = k.reshape(T, -1)
    for t in range(500, 570, 10):  # (of the first of three segments)
        x[t, heads * dim + 5 * dim:heads * dim + 6 * dim] = 1e18 * rng.standard_normal(dim)
        x[t, 2 * heads * dim + 5 * vdim:2 * heads * dim + 6 * vdim] = 1e18 * rng.standard_normal(vdim)
    proj, pv = dev.act(x, f32)
    first = rng.standard_normal((heads, vdim, dim))
    first[:4, 1, 3], first[:4, 2, 7], first[:4, 2, 9], first[4:6] = np.inf, -np.inf, np.inf, 0.0
    d_decay, d_lg = dev.f(decay), dev.f(np.log2(decay.astype(np.float64)))
    room, out = heads * (vdim + 1) * dim, []
    for r in (0, segments):
        ws, state, o = dev.empty((max(4, r * room),), True), dev.f(first), dev.empty((T, heads * vdim), True)
        awq.check(lib.awq_linear_attention_segments(proj.data_ptr(), n, heads, dim, vdim, d_decay.data_ptr(), d_lg.data_ptr(), state.data_ptr(),
                                                    o.data_ptr(), T, pos0, f32, ws.data_ptr(), r * room, dev.stream))
        out.append((dev.host(o).reshape(T, heads, vdim).transpose(1, 2, 0), dev.host(state)))
    for one, beside in zip(*out):
        for is_so in (np.isnan, np.isposinf, np.isneginf):
            assert np.array_equal(is_so(one), is_so(beside)), is_so.__name__
        assert np.isposinf(out[0][1][1:3, 1, 3]).all() and not np.isfinite(one[:3, 1:3]).all()
        for h in range(heads):
            fine = np.isfinite(one[h])
            assert fine.any() and np.abs(one[h][fine] - beside[h][fine]).max() <= 3e-5 * np.abs(one[h][fine]).max(), h
    q, k, v = (pv[:, at:at + m].reshape(T, heads, -1)[:, 5:6] for at, m in
               ((0, heads * dim), (heads * dim, heads * dim), (2 * heads * dim, heads * vdim)))
    want = plain.linear_attention(q, k, v, decay[5:6].astype(np.float64))[0][1280:1300, 0].T  # (tokens of the third segment)
    for o, _ in out:
        assert np.abs(o[5][:, 1280:1300] - want).max() <= 3e-5 * np.abs(want).max()


def attend(awq, lib, dev, f32, proj, heads, kv, dim, vdim, window, scale, eps, temp, sizes, T, slots, max_pos):
    """the attention of T tokens in portions; proj: the tensor with all tokens' projections (kept as it is)"""
    kr, vr = lib.awq_window_row(dim), lib.awq_window_row(vdim)
    kc, vc = dev.empty((slots, kv, kr), f32, 0.0), dev.empty((slots, kv, vr), f32, 0.0)
    ws = dev.empty((max(1, lib.awq_window_workspace_floats(heads, vdim, window, max_pos)),), True)
    slope = dev.f([plain.slope(h, heads) for h in range(heads)])
    n = heads * vdim
    ldc = (n + 7) // 8 * 8
    out, at, i = [], 0, 0
    while at < T:
        m = min(sizes[i % len(sizes)], T - at)
        p = proj[at:at + m].clone()
        ctx = dev.empty((m, ldc), f32)
        a = awq.AwqWindowArgs(p.data_ptr(), p.shape[1], heads, kv, dim, vdim, window, slots, scale, eps, temp[0], 0, temp[1],
                              slope.data_ptr(), kc.data_ptr(), vc.data_ptr(), ctx.data_ptr(), ldc, m, at, max_pos, ws.data_ptr())
        awq.check(lib.awq_window_attention(ctypes.byref(a), f32, dev.stream))
        dev.torch.cuda.synchronize()
        out.append(ctx)
        at, i = at + m, i + 1
    return dev.host(dev.torch.cat(out))[:, :n].reshape(T, heads, vdim)


SHAPES = [(4, 2, 64, 64), (3, 3, 128, 128), (6, 1, 20, 12), (2, 1, 256, 96), (12, 1, 32, 200), (1, 1, 300, 72), (10, 2, 64, 36)]


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
@pytest.mark.parametrize("window", [0, 1, 33, 64, 65, 129])
def test_window_attention(awq, lib, dev, f32, shape, window):
    """random scores of some size: prompts, portions and single tokens, over several cache blocks"""
    heads, kv, dim, vdim = shape
    print("window attention", shape, window, f32, flush=True)
    rng = np.random.default_rng(dim + window)
    T, eps, scale, temp = 200, 1e-3, 3.0 / dim ** 0.5, (0.7, 13.0)
    n = heads * dim + kv * (dim + vdim)
    proj, pv = dev.act(np.pad(2 * rng.standard_normal((T, n)), ((0, 0), (0, -n % 8))), f32)
    q = plain.rms(pv[:, :heads * dim].reshape(T, heads, dim), eps)
    k = plain.rms(pv[:, heads * dim:(heads + kv) * dim].reshape(T, kv, dim), eps)
    if not f32:  # what the matrix cores are given
        q, k = km.bf16(q).astype(np.float64), km.bf16(k).astype(np.float64)
    v = pv[:, (heads + kv) * dim:n].reshape(T, kv, vdim)
    want = plain.window_attention(q, k, v, window or None, scale, temp)
    for sizes in ([200], [1], [2, 63, 1], [100, 1]):
        slots = 256 if not window else (window - 1 + max(sizes) + 63) // 64 * 64
        got = attend(awq, lib, dev, f32, proj, heads, kv, dim, vdim, window, scale, eps, temp, sizes, T, slots, T)
        assert km.rms_error(got, want) < (3e-5 if f32 else 0.01), sizes


@pytest.mark.parametrize("steep", [3.0, 16.0])
@pytest.mark.parametrize("shape", [(3, 3, 128, 128), (4, 2, 64, 128), (10, 2, 64, 36), (2, 1, 100, 60)], ids=str)
@pytest.mark.parametrize("window", [0, 160, 257])
def test_window_attention_with_the_keys_in_halves(awq, lib, dev, shape, window, steep):
    """bfloat16, more than 256 keys: every instance with halves, ragged ends, queries that see keys of one half only and, where scores are steep, maxima
    that move by more than 2^8 in either half.  Beside the output's rounding (2^-9) a component of q or k that the norm leaves
    at the edge of a rounding may fall on the other side: up to steep / sqrt(dim) x 2^-8 x 3^2 of a score, 5 % of a weight at worst, a few of them in
    a row whose other weights hold"""
    heads, kv, dim, vdim = shape
    print("window attention in halves", shape, window, steep, flush=True)
    rng = np.random.default_rng(dim + window)
    T, eps, scale = 400, 1e-3, steep / dim ** 0.5
    n = heads * dim + kv * (dim + vdim)
    proj, pv = dev.act(np.pad(2 * rng.standard_normal((T, n)), ((0, 0), (0, -n % 8))), False)
    q = km.bf16(plain.rms(pv[:, :heads * dim].reshape(T, heads, dim), eps)).astype(np.float64)
    k = km.bf16(plain.rms(pv[:, heads * dim:(heads + kv) * dim].reshape(T, kv, dim), eps)).astype(np.float64)
    v = pv[:, (heads + kv) * dim:n].reshape(T, kv, vdim)
    want = plain.window_attention(q, k, v, window or None, scale, (0.0, 1.0))
    for sizes in ([400], [300, 100], [7, 280, 113]):
        slots = ((window or T) - 1 + max(sizes) + 63) // 64 * 64
        got = attend(awq, lib, dev, 0, proj, heads, kv, dim, vdim, window, scale, eps, (0.0, 1.0), sizes, T, slots, T)
        off = km.rms_error(got, want)
        print("error %.1e" % off, flush=True)
        assert off < (0.01 if steep < 4 else 0.03), sizes


@pytest.mark.parametrize("T", [96, 400])
@pytest.mark.parametrize("window", [0, 90])
def test_a_query_among_others(awq, lib, dev, window, T):
    """bfloat16, 32 queries to a wavefront: those behind the twentieth of each 32 meet one key in every tile that they nearly equal, at scores that
    grow, and the bits of the others do not notice"""
    heads, dim = 3, 128
    print("a query among others", window, T, flush=True)
    rng = np.random.default_rng(T + window)
    q, k, v = (rng.standard_normal((T, heads, dim)) for _ in range(3))
    own = np.arange(T) % 32 < 20
    to = rng.standard_normal((heads, dim))
    others = np.where(own[:, None, None], q, to)
    for t in range(7, T, 32):
        k[t] = to + (T - t) / 100 * k[t]
    out = []
    for x in (q, others):
        proj, _ = dev.act(np.concatenate([y.reshape(T, -1) for y in (x, k, v)], axis=1), False)
        out.append(attend(awq, lib, dev, 0, proj, heads, heads, dim, dim, window, 2.0 * dim ** -0.5, 1e-6, (0.0, 1.0), [T], T,
                          ((window or T) + T + 63) // 64 * 64, T))
    assert np.array_equal(out[0][own], out[1][own]) and not np.array_equal(out[0][~own], out[1][~own])


@pytest.mark.parametrize("f32,shape", [(1, (4, 2, 64, 64)), (1, (6, 1, 20, 12)), (1, (2, 1, 300, 72)), (0, (2, 1, 300, 72)),
                                       (1, (10, 2, 64, 36)), (0, (10, 1, 300, 72)), (0, (6, 1, 300, 72))], ids=str)
@pytest.mark.parametrize("window", [0, 1, 2, 5, 250])
def test_values_that_a_query_does_not_see(awq, lib, dev, f32, shape, window):
    """several queries share a reading of the rows, two or four where there are many; a row that some of them do not see may hold
    anything.  Without a window their bits are those of queries that share none"""
    heads, kv, dim, vdim = shape
    print("rows not seen", shape, window, f32, flush=True)
    rng = np.random.default_rng(window)
    T, n = 300, heads * dim + kv * (dim + vdim)
    x = np.pad(rng.standard_normal((T, n)), ((0, 0), (0, -n % 8)))
    args = lambda p, sizes: attend(awq, lib, dev, f32, dev.act(p, f32)[0], heads, kv, dim, vdim, window, dim ** -0.5, 1e-6, (0.0, 1.0), sizes,
                                   T, ((window or T) - 1 + max(sizes) + 63) // 64 * 64, T)
    for sizes in ([T], [64, 7, 4]):
        want = args(x, sizes)
        assert np.isfinite(want).all() and (window or np.array_equal(want, args(x, [2, 70, 3])))
        for at in (0, 5, 130, 256, 258):
            y = x.copy()
            y[at, (heads + kv) * dim:n] = np.nan if at & 1 else np.inf
            got = args(y, sizes)
            sees = (np.arange(T) >= at) & (np.arange(T) < (at + window if window else T))
            assert np.array_equal(got[~sees], want[~sees]) and not np.isfinite(got[sees]).any(), (at, sizes)


@pytest.mark.parametrize("heads,kv,dim,vdim", [(4, 2, 64, 128), (6, 2, 100, 60), (2, 1, 130, 256)], ids=str)
@pytest.mark.parametrize("sizes", [[2, 14, 1], [15, 17, 33], [127, 2, 16], [129, 3]], ids=str)
@pytest.mark.parametrize("window", [0, 40])
def test_roundings_of_window_attention(awq, lib, dev, heads, kv, dim, vdim, sizes, window):
    """Portions that end beside the edges of tiles of 16 queries and 128 keys, on a ring that wraps.  A score of up to S rounds by
    S x 2^-24 (its products' sum, its bias, their difference), which its weight takes over with expf's 2^-23; a mean of values rounds
    by less: (S + 4) x 2^-24, and S is below 16 here."""
    print("roundings, window attention", heads, kv, dim, vdim, sizes, window, flush=True)
    rng = np.random.default_rng(dim + sizes[0])
    T, eps, scale, n = 300, 1e-6, 3.0 / dim ** 0.5, heads * dim + kv * (dim + vdim)
    proj, pv = dev.act(np.pad(rng.standard_normal((T, n)), ((0, 0), (0, -n % 8))), True)
    q = plain.rms(pv[:, :heads * dim].reshape(T, heads, dim), eps)
    k = plain.rms(pv[:, heads * dim:(heads + kv) * dim].reshape(T, kv, dim), eps)
    want = plain.window_attention(q, k, pv[:, (heads + kv) * dim:n].reshape(T, kv, vdim), window or None, scale, (0.0, 1.0))
    assert scale * np.abs(np.einsum("thd,shd->hts", q, np.repeat(k, heads // kv, 1))).max() < 16
    slots = ((window or T) - 1 + max(sizes) + 63) // 64 * 64
    got = attend(awq, lib, dev, True, proj, heads, kv, dim, vdim, window, scale, eps, (0.0, 1.0), sizes, T, slots, T)
    off = np.linalg.norm(got - want) / np.linalg.norm(want)
    print("error %.1e" % off, flush=True)
    assert off < 20 * 2.0 ** -24


@pytest.mark.parametrize("sizes", [[2, 47], [48, 49, 3], [50, 1, 48]], ids=str)
@pytest.mark.parametrize("window", [40, 270, 280, 300])
def test_few_queries_of_a_window_and_more(awq, lib, dev, sizes, window):
    """portions beside the line between the two forms, 384 rows and 320 keys; the bound is that of the test above"""
    test_roundings_of_window_attention(awq, lib, dev, 8, 2, 128, 100, sizes, window)


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
@pytest.mark.parametrize("window", [1, 2, 31, 32, 33, 64, 65, 96, 128, 160])
def test_window_edges(awq, lib, dev, f32, window):
    """One key outweighs every other for all queries.  At distance window - 1 it is all a query sees, at distance
    window nothing of it is left; in prompts, portions and decoding, wherever the key lies."""
    print("window edge", window, f32, flush=True)
    heads, kv, dim, vdim = 2, 1, 64, 64
    rng = np.random.default_rng(window)
    T = 330
    for far in (0, 5, 63, 64, 127):
        q = np.tile(np.eye(1, dim), (T, heads, 1)) * 8
        k = np.tile(np.eye(1, dim, 1), (T, kv, 1))
        k[far] = np.eye(1, dim)               # q . k = dim there, 0 elsewhere after the norms
        v = 0.1 * rng.standard_normal((T, kv, vdim))
        v[far] = 1.0
        proj, pv = dev.act(np.concatenate([x.reshape(T, -1) for x in (q, k, v)], axis=1), f32)
        vv = pv[:, (heads + kv) * dim:].reshape(T, kv, vdim)
        want = plain.window_attention(plain.rms(q, 1e-6), plain.rms(k, 1e-6), vv, window, 3.0)
        assert far + window >= T or (want[far + window - 1].min() > 0.9 and want[far + window].max() < 0.5)
        for sizes in ([T], [1], [37, 2, 1, 1], [128, 1]):
            slots = (window - 1 + max(sizes) + 63) // 64 * 64
            got = attend(awq, lib, dev, f32, proj, heads, kv, dim, vdim, window, 3.0, 1e-6, (0.0, 1.0), sizes, T, slots, T)
            assert np.abs(got - want).max() < (1e-4 if f32 else 0.01), (far, sizes)


@pytest.mark.parametrize("f32", FORMATS, ids=["bf16", "f32"])
def test_a_far_key_among_many_and_the_bias(awq, lib, dev, f32):
    """no window: a single key hundreds of positions back carries the answer although the distance bias pulls it down"""
    heads, kv, dim, vdim, T = 8, 4, 128, 64, 700
    q = np.tile(np.eye(1, dim), (T, heads, 1)) * 5
    k = np.tile(np.eye(1, dim, 1), (T, kv, 1))
    v = np.zeros((T, kv, vdim))
    for i, at in enumerate((3, 64, 191, 400)):
        k[at, i] = np.eye(1, dim)
        v[at, i] = 1 + i
    proj, pv = dev.act(np.concatenate([x.reshape(T, -1) for x in (q, k, v)], axis=1), f32)
    want = plain.window_attention(plain.rms(q, 1e-6), plain.rms(k, 1e-6), v, None, 0.3, (0.5, 100))
    assert want[-1].max() > 0.5 and want[-1].min() < 0.01   # heads differ: the bias decides
    for sizes in ([T], [650, 1], [127, 2]):
        got = attend(awq, lib, dev, f32, proj, heads, kv, dim, vdim, 0, 0.3, 1e-6, (0.5, 100.0), sizes, T, 704, T)
        assert np.abs(got - want).max() < (2e-3 if f32 else 0.04), sizes
