"""The fp32 convolutions on split operands (conv_split.hip, wgrad_oct.hip) against what fp32 instructions would give: the error of
their sums over the operands that networks have."""
import numpy as np
import pytest

from util import kernels_of, nl2, randn, rng, seconds

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def singa():
    from singa_amd import singa_wrap
    return singa_wrap


def operands(kind, seed, n, c, h, w, k, r):
    """x, W, dy: normal values ("normal"), x behind a ReLU ("relu"), everything of one sign ("positive")"""
    rg = rng(seed)
    x, W, dy = randn(rg, n, c, h, w), randn(rg, k, c, r, r) * np.float32((2 / (c * r * r)) ** 0.5), randn(rg, n, k, h, w)
    if kind == "relu":
        x = np.maximum(x, 0)
    if kind == "positive":
        x, W, dy = np.abs(x), np.abs(W), np.abs(dy)
    return x, W, dy


def passes(singa, dev, x, W, dy):
    """The three passes of a layer of stride 1 and "same" padding and the kernels that they ran on"""
    c, k, r = x.shape[1], W.shape[0], W.shape[2]
    xd, wd, dyd = (singa.from_numpy(a, dev) for a in (x, W, dy))
    hd = singa.CudnnConvHandle(xd, (r, r), (1, 1), (r // 2, r // 2), c, k, False)
    return [kernels_of(dev, f) for f in (lambda: singa.GpuConvForward(xd, wd, None, hd).to_numpy(),
                                         lambda: singa.GpuConvBackwardx(dyd, wd, xd, hd).to_numpy(),
                                         lambda: singa.GpuConvBackwardW(dyd, xd, wd, hd).to_numpy())]


def fma32(acc, a, b):
    """fp32 fused multiply-add (the float64 product of two fp32 values is exact, their sum with a third rounds once before the
    rounding to fp32, which does not move a statistic)"""
    return (acc.double() + a.double() * b.double()).float()


def conv64(x, W):
    """float64 convolution of stride 1 and "same" padding, and the same as one chain of fp32 multiply-adds per result"""
    import torch
    x, W = torch.from_numpy(x), torch.from_numpy(W)
    n, c, h, w = x.shape
    r = W.shape[2]
    xp = torch.nn.functional.pad(x, (r // 2,) * 4)
    want = torch.nn.functional.conv2d(x.double(), W.double(), padding=r // 2)
    chain = torch.zeros(want.shape, dtype=torch.float32)
    for ch in range(c):
        for i in range(r):
            for j in range(r):
                chain = fma32(chain, xp[:, ch:ch + 1, i:i + h, j:j + w], W[:, ch, i, j].view(1, -1, 1, 1))
    return want.numpy(), chain.numpy()


@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("n,c,h,w,k,r", [(4, 64, 12, 14, 64, 3), (2, 300, 10, 10, 64, 3), (1, 40, 9, 11, 130, 3), (2, 32, 12, 12, 64, 5)])
def test_conv_split_error_of_an_fp32_chain(singa, dev, n, c, h, w, k, r, kind):
    """Against float64, beside a chain of fp32 multiply-adds, which is what the fp32 matrix instructions form.  A chain rounds at
    its own magnitude once per product that is not zero; here that happens once per 16 products, after a dozen roundings at the
    magnitude of those 16: an error of sqrt(1 / 16 + 12 / products) of a chain's, and sqrt(2) of that where a ReLU has left half of
    the products (0.3 to 0.45; shared tiles less)."""
    x, W, dy = operands(kind, n + c + k, n, c, h, w, k, r)
    fwd, dgrad, _ = passes(singa, dev, x, W, dy)
    assert fwd[1] == {"k_conv_split"} and dgrad[1] == {"k_conv_split"}
    Wt = np.ascontiguousarray(W.transpose(1, 0, 2, 3)[:, :, ::-1, ::-1])
    for got, (want, chain) in ((fwd[0], conv64(x, W)), (dgrad[0], conv64(dy, Wt))):
        print(kind, "error %.2e, of a chain %.2e" % (nl2(got, want), nl2(chain, want)))
        assert nl2(got, want) < 0.45 * nl2(chain, want)

@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("n,c,h,w,k", [(20, 512, 7, 7, 200), (13, 256, 10, 10, 256), (20, 100, 21, 20, 260), (8, 128, 25, 29, 140), (6, 64, 48, 40, 180)])
def test_conv_wgrad_octets_error_of_fp32_chains(singa, dev, n, c, h, w, k, kind):
    """The same for the weight gradient, whose pixels are summed in twice as many stretches as there are partial images (one per
    CU): against chains of fp32 multiply-adds over as many stretches, on the first filters and channels."""
    import torch
    x, W, dy = operands(kind, n + c + k, n, c, h, w, k, 3)
    got, names = passes(singa, dev, x, W, dy)[2]
    assert names == {"k_wgrad_oct"}
    few = 16
    strips = (w + 31) // 32
    stretches = 2 * (256 // (((k + 63) // 64) * ((c + 63) // 64) * strips))
    xp = torch.nn.functional.pad(torch.from_numpy(x[:, :few]), (1, 1, 1, 1))
    taps = torch.stack([xp[:, :, i:i + h, j:j + w].permute(1, 0, 2, 3).reshape(few, -1) for i in range(3) for j in range(3)], 1)
    d = torch.from_numpy(dy[:, :few]).permute(1, 0, 2, 3).reshape(few, -1)
    want = torch.einsum("kp,ctp->kct", d.double(), taps.double()).reshape(few, few, 3, 3).numpy()
    length = -(-d.shape[1] // stretches)
    total = torch.zeros(few, few, 9, dtype=torch.float64)
    pad = stretches * length - d.shape[1]
    d, taps = (torch.nn.functional.pad(t, (0, pad)).unflatten(-1, (stretches, length)) for t in (d, taps))
    acc = torch.zeros(few, few, 9, stretches)
    for i in range(length):
        acc = fma32(acc, d[:, None, None, :, i], taps[None, :, :, :, i])
    chain = acc.double().sum(-1).float().reshape(few, few, 3, 3).numpy()
    mine = got[:few, :few]
    print(kind, "error %.2e, of chains %.2e" % (nl2(mine, want), nl2(chain, want)))
    assert nl2(mine, want) < nl2(chain, want)   # (short chains: the rounding of the result is most of either error)


@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("n,c,h,w,k", [(1, 8, 7, 7, 64), (3, 20, 9, 12, 130), (30, 64, 14, 14, 64), (2, 40, 57, 43, 60), (70, 33, 8, 8, 300), (2, 64, 30, 62, 128)])
def test_conv_split_forward_of_stride_two(singa, dev, n, c, h, w, k, kind):
    """3x3 forward passes of stride 2 and padding 1: odd and even planes, tiles over many images, every tile size, against float64, no
    further off than the fp32 chain; an infinity in x and one in a filter reach the results that they do in a zero-padded image."""
    import torch
    x, W, _ = operands(kind, n + c + h, n, c, h, w, k, 3)
    b = randn(rng(k), k)
    hd = singa.CudnnConvHandle(singa.from_numpy(x, dev), (3, 3), (2, 2), (1, 1), c, k, True)
    run = lambda x, W: kernels_of(dev, lambda: singa.GpuConvForward(*(singa.from_numpy(a, dev) for a in (x, W, b)), hd).to_numpy())
    conv = lambda x, W: (torch.nn.functional.conv2d(torch.from_numpy(x).double(), torch.from_numpy(W).double(), stride=2, padding=1)
                         + torch.from_numpy(b).double()[:, None, None]).numpy()
    got, names = run(x, W)
    assert names == {"k_conv_split"}, names
    m = min(n, 3)   # (the chain of a few images is as good as that of all)
    want, chain = conv64(x[:m], W)
    want, chain = want[:, :, ::2, ::2], chain[:, :, ::2, ::2]
    off = got - conv(x, W)
    assert nl2(got[:m] - b[:, None, None].astype(np.float64), want) <= 1.1 * nl2(chain, want) + 2.0 ** -24
    assert np.all(np.abs(off) <= 2.0 ** -24 * (9 * c + 40) * (np.abs(want).max() + np.abs(b).max()))
    x[n - 1, c - 1, h - 1, w // 2] = np.inf
    W[k - 1, 0, 0, 2] = np.inf
    got, want = run(x, W)[0], conv(x, W)
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and np.array_equal(np.isnan(got), np.isnan(want))
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= 2.0 ** -24 * (9 * c + 40) * (np.abs(want[ok]).max() + np.abs(b).max()))


@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("n,c,h,w,k", [(4, 64, 14, 14, 64), (2, 128, 9, 11, 130), (70, 33, 7, 8, 8), (1, 100, 58, 120, 72), (1, 100, 6, 256, 72),
                                       (1, 64, 8, 219, 64), (44, 64, 56, 56, 48), (300, 200, 5, 3, 16), (40, 70, 9, 1, 16), (41, 64, 11, 5, 130),
                                       (7, 300, 9, 13, 8)])   # (odd rows: single columns, tiles that begin with the last one)
def test_data_gradient_of_stride_two_on_split_operands(singa, dev, n, c, h, w, k, kind):
    """3x3 data gradients of stride 2 and padding 1: odd and even planes, tiles over many images, either tile, whole and shared, every
    slab, against float64 and no further off than the fp32 chain; onto a gradient that is there already, the sum of the two; an infinity
    in dy and one in a filter reach the results that they do where a tap outside dy does not exist."""
    import torch
    x, W, _ = operands(kind, n + c + h, n, c, h, w, k, 3)
    dy = operands(kind, n + k, n, k, (h + 1) // 2, (w + 1) // 2, 1, 1)[0]
    there = randn(rng(c), n, c, h, w)
    xd = singa.from_numpy(x, dev)
    hd = singa.CudnnConvHandle(xd, (3, 3), (2, 2), (1, 1), c, k, False)
    onto = lambda dy, W: singa.GpuConvBackwardxAccumulate(singa.from_numpy(dy, dev), singa.from_numpy(W, dev), xd, hd, singa.from_numpy(there, dev))
    run = lambda dy, W: kernels_of(dev, lambda: singa.GpuConvBackwardx(singa.from_numpy(dy, dev), singa.from_numpy(W, dev), xd, hd).to_numpy())
    grad = lambda dy, W: torch.nn.functional.conv_transpose2d(torch.from_numpy(dy).double(), torch.from_numpy(W).double(), stride=2, padding=1,
                                                              output_padding=(1 - h % 2, 1 - w % 2)).numpy()
    got, names = run(dy, W)
    assert names == {"k_dgrad_split2"}, names
    assert np.array_equal(onto(dy, W).to_numpy(), there + got)
    m = min(n, 3)   # (the chain of a few images is as good as that of all)
    apart = np.zeros((m, k, h, w), np.float32)
    apart[:, :, ::2, ::2] = dy[:m]
    want, chain = conv64(apart, np.ascontiguousarray(W.transpose(1, 0, 2, 3)[:, :, ::-1, ::-1]))
    print(kind, "error %.2e, of a chain %.2e" % (nl2(got[:m], want), nl2(chain, want)))
    assert nl2(got[:m], want) <= 1.1 * nl2(chain, want) + 2.0 ** -24   # (half an ulp of a result: one channel has one product)
    bound = lambda want: 2.0 ** -24 * (4 * k + 40) * np.abs(want).max()   # (four taps at most, a rounding each of what is no larger)
    assert np.all(np.abs(got - grad(dy, W)) <= bound(want) + 2.0 ** -24 * (4 * k + 40))
    dy[n - 1, k - 1, -1, -1] = np.inf
    W[k - 1, 0, 0, 2], W[0, c - 1, 0, 0] = np.inf, -np.inf
    got, want = run(dy, W)[0], grad(dy, W)
    assert np.array_equal(np.isfinite(got), np.isfinite(want)) and np.array_equal(np.isnan(got), np.isnan(want))
    ok = np.isfinite(want)
    assert np.all(np.abs(got[ok] - want[ok]) <= bound(want[ok]) + 2.0 ** -24 * (4 * k + 40))


def test_data_gradient_of_stride_two_by_workspace_and_size(singa, dev):
    """The split kernel runs where the workspace holds its partial tiles and where the reduction is worth the split; weights laid out for
    a call with one size of workspace are not taken by a call with another."""
    import ctypes as C

    from singa_amd import _lib
    lib = _lib.lib()
    for (n, c, h, w, k), least in (((4, 64, 20, 22, 96), "k_dgrad3x3"), ((4, 64, 21, 22, 96), "k_igemm"), ((5, 131, 9, 11, 31), None), ((2, 64, 20, 22, 40), None)):
        x, W, _ = operands("normal", 4, n, c, h, w, k, 3)
        dy = randn(rng(5), n, k, (h + 1) // 2, (w + 1) // 2)
        xd, wd, dyd, dxd = (singa.from_numpy(a, dev) for a in (x, W, dy, np.zeros_like(x)))
        hd = singa.CudnnConvHandle(xd, (3, 3), (2, 2), (1, 1), c, k, False)
        g = hd.geom
        full = lib.sgh_conv_workspace_bytes(C.byref(g), _lib.SGH_CONV_DGRAD)
        space = singa.from_numpy(np.zeros(full // 4 + 64, np.float32), dev)

        def dgrad(size):
            (rc, out), names = kernels_of(dev, lambda: (lib.sgh_conv_dgrad_f32(C.byref(g), dyd.ptr, wd.ptr, dxd.ptr, space.ptr, size, dev.stream),
                                                        dxd.to_numpy()))
            return (out, names) if rc == 0 else (None, rc)

        def prepare(size):
            item = (_lib.ConvPrepareItem * 1)()
            item[0].g, item[0].W, item[0].workspace, item[0].ws_bytes = C.pointer(g), wd.ptr, space.ptr, size
            assert lib.sgh_conv_dgrad_prepare_multi(item, 1, 0, dev.stream) == 0

        if least is None:
            assert dgrad(full)[1] in ({"k_dgrad3x3"}, {"k_igemm"})
            continue
        less = full
        while dgrad(less)[1] == {"k_dgrad_split2"}:   # (a size that is too little for it and enough for the fp32 kernel)
            less = less * 9 // 10
        want = {size: dgrad(size) for size in (full, less)}
        assert want[full][1] == {"k_dgrad_split2"} and want[less][1] == {least}, (want[less][1], least)
        assert nl2(want[full][0], want[less][0]) < 1e-6
        for prepared in (full, less):
            for called in (full, less):
                prepare(prepared)
                got, names = dgrad(called)
                assert names == want[called][1] and np.array_equal(got, want[called][0]), (prepared, called)


@pytest.mark.parametrize("what", ["inf", "one inf", "overflow", "nan", "nan weights", "inf weights"])
def test_conv_split_time_of_non_finite_operands(singa, dev, what):
    """Results that are not finite take a second pass over their tile on the fp32 instructions, 2.7 times the first one, and no search
    per result: eight times the time of ordinary operands at most (a term-by-term search took 100 to 250 times)."""
    n, c, h, w, k = 32, 256, 14, 14, 256
    x, W, dy = operands("normal", 3, n, c, h, w, k, 3)

    def times(x, W, dy):
        xd, wd, dyd = (singa.from_numpy(a, dev) for a in (x, W, dy))
        hd = singa.CudnnConvHandle(xd, (3, 3), (1, 1), (1, 1), c, k, False)
        return seconds(dev, lambda: singa.GpuConvForward(xd, wd, None, hd)), seconds(dev, lambda: singa.GpuConvBackwardx(dyd, wd, xd, hd))

    plain = times(x, W, dy)
    value = np.float32(np.nan if "nan" in what else np.inf)
    if what == "one inf":
        x[:, 0, 7, 7] = value
        dy[:, 0, 7, 7] = value
    elif what == "overflow":
        x, W, dy = x * np.float32(1e30), W * np.float32(1e10), dy * np.float32(1e30)
    elif "weights" in what:
        W[:] = value
    else:
        x[:] = value
        dy[:] = value
    for got, ordinary in zip(times(x, W, dy), plain):
        print(what, "%.1f us, ordinary operands %.1f" % (got * 1e6, ordinary * 1e6))
        assert got < 8 * ordinary


@pytest.mark.parametrize("n,c,h,w,k,r", [(2, 24, 9, 10, 40, 3), (1, 300, 6, 6, 130, 3), (30, 64, 20, 20, 64, 3), (2, 20, 9, 7, 40, 5)])
@pytest.mark.parametrize("where", ["x", "w", "both"])
def test_conv_split_infinities_and_nans(singa, dev, n, c, h, w, k, r, where):
    """+inf, -inf and NaN reach exactly the results that their products reach, with the sign that those have, and the finite
    results next to them stay what they were; an infinite weight meets the padding in the forward pass (a NaN) and not in the
    data gradient."""
    import torch
    x, W, dy = operands("normal", 11, n, c, h, w, k, r)
    if where != "w":
        for t in (x, dy):
            t[0, 1, 0, w - 1], t[-1, 2, h // 2, 1], t[0, 3, h - 1, 0] = -np.inf, np.inf, np.nan
    if where != "x":
        W[k - 1, c // 3, r // 2, 0], W[0, 0, 0, 0], W[k // 2, c - 1, r - 1, r - 1], W[1, 1, r // 2, r // 2] = -np.inf, np.inf, np.nan, -np.inf
    fwd, dgrad, _ = passes(singa, dev, x, W, dy)
    with np.errstate(all="ignore"):
        t = lambda a: torch.from_numpy(a.astype(np.float64))
        xp = torch.nn.functional.pad(t(x), (r // 2,) * 4)
        want = [sum(torch.einsum("kc,nchw->nkhw", t(W[:, :, i, j].copy()), xp[:, :, i:i + h, j:j + w]) for i in range(r) for j in range(r))]
        dx = torch.zeros(n, c, h + r - 1, w + r - 1, dtype=torch.float64)
        for i in range(r):
            for j in range(r):
                dx[:, :, i:i + h, j:j + w] += torch.einsum("kc,nkhw->nchw", t(W[:, :, i, j].copy()), t(dy))
        want.append(dx[:, :, r // 2:r // 2 + h, r // 2:r // 2 + w])
    for (got, _), ref in zip((fwd, dgrad), (a.numpy().astype(np.float32) for a in want)):
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(np.isposinf(got), np.isposinf(ref)) and np.array_equal(np.isneginf(got), np.isneginf(ref))
        fin = np.isfinite(ref)
        np.testing.assert_allclose(got[fin], ref[fin], rtol=1e-4, atol=1e-4)


# rows of one, two, four and (three) four octets, several strips, ragged channels; each takes the octet kernel
WGRAD_OCTET_LAYERS = [(20, 512, 7, 7, 200), (24, 257, 9, 8, 190), (40, 100, 13, 13, 250), (13, 130, 20, 21, 120), (14, 100, 20, 30, 140), (6, 64, 37, 41, 210)]


def wgrad64(x, dy):
    """float64 weight gradient of 3x3, stride 1, padding 1"""
    import torch
    n, c, h, w = x.shape
    xp = torch.nn.functional.pad(torch.from_numpy(x).double(), (1, 1, 1, 1))
    d = torch.from_numpy(dy).double().permute(1, 0, 2, 3).reshape(dy.shape[1], -1).contiguous()
    taps = [d @ xp[:, :, i:i + h, j:j + w].permute(0, 2, 3, 1).reshape(-1, c) for i in range(3) for j in range(3)]
    return torch.stack(taps, -1).reshape(dy.shape[1], c, 3, 3).numpy()


@pytest.mark.parametrize("n,c,h,w,k", WGRAD_OCTET_LAYERS)
def test_conv_wgrad_octets_values(singa, dev, n, c, h, w, k):
    """Against float64: within terms * 2^-23 of the sum of the terms' magnitudes, and closer than a sixteenth of the roundings of
    chains of fp32 additions (0.5 * sqrt(terms) * 2^-24, and the rounding of the result); the same bits again."""
    x, W, dy = operands("normal", n + c + k, n, c, h, w, k, 3)
    got, names = passes(singa, dev, x, W, dy)[2]
    assert names == {"k_wgrad_oct"}
    want = wgrad64(x, dy)
    assert np.all(np.abs(got - want) <= n * h * w * 2.0 ** -23 * wgrad64(np.abs(x), np.abs(dy)))
    assert nl2(got, want) < (0.5 * (n * h * w) ** 0.5 + 1) * 2.0 ** -24
    again, _ = passes(singa, dev, x, W, dy)[2]
    assert np.array_equal(again, got)


@pytest.mark.parametrize("n,c,h,w,k", WGRAD_OCTET_LAYERS)
def test_conv_wgrad_octets_infinities_and_nans(singa, dev, n, c, h, w, k):
    """+inf, -inf and NaN, also in the first and last rows and columns, reach exactly the weights that their products reach, those
    with the padding among them (zeros: NaN), with the sign that those have."""
    x, W, dy = operands("normal", 13, n, c, h, w, k, 3)
    x[n // 2, 5, h - 1, w - 1], x[1, 6, 0, 0], x[2, 7, h // 2, 1], x[0, c - 1, 0, w - 1] = -np.inf, np.inf, np.nan, np.inf
    dy[n - 1, k - 1, h - 1, 4], dy[0, 3, 1, w - 1], dy[3, 4, 2, 2] = np.inf, -np.inf, np.nan
    got, names = passes(singa, dev, x, W, dy)[2]
    assert names == {"k_wgrad_oct"}
    with np.errstate(all="ignore"):
        want = wgrad64(x, dy).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("n,c,h,w,k", [(30, 256, 14, 13, 256), (40, 150, 22, 31, 96), (20, 100, 41, 40, 260), (8, 128, 50, 57, 140), (6, 62, 97, 120, 80),
                                       (20, 520, 17, 34, 500)])   # (the last: 144 tiles and strips, split over three rounds of workgroups)
def test_weight_gradient_of_stride_two_by_octets(singa, dev, n, c, h, w, k):
    """3x3 weight gradients of stride 2 and padding 1, one strip and several, odd and even planes, against float64: within terms * 2^-23 of
    the sum of the terms' magnitudes, and closer than a sixteenth of the roundings of chains of fp32 additions (0.5 * sqrt(terms) * 2^-24, and
    the rounding of the result); infinities and NaNs reach the weights that their products reach, those with the padding among them."""
    import torch
    x, W, _ = operands("normal", n + c + k, n, c, h, w, k, 3)
    P, Q = (h + 1) // 2, (w + 1) // 2
    dy = randn(rng(n), n, k, P, Q)
    terms = n * P * Q
    hd = singa.CudnnConvHandle(singa.from_numpy(x, dev), (3, 3), (2, 2), (1, 1), c, k, False)
    run = lambda x, dy: kernels_of(dev, lambda: singa.GpuConvBackwardW(*(singa.from_numpy(a, dev) for a in (dy, x, W)), hd).to_numpy())

    def grad(x, dy):
        xp = torch.nn.functional.pad(torch.from_numpy(x).double(), (1, 2, 1, 2))
        d = torch.from_numpy(dy).double().permute(1, 0, 2, 3).reshape(k, -1).contiguous()
        taps = [d @ xp[:, :, i:i + 2 * P:2, j:j + 2 * Q:2].permute(0, 2, 3, 1).reshape(-1, c) for i in range(3) for j in range(3)]
        return torch.stack(taps, -1).reshape(k, c, 3, 3).numpy()

    got, names = run(x, dy)
    assert names == {"k_wgrad_oct"}, names
    want = grad(x, dy)
    assert np.all(np.abs(got - want) <= terms * 2.0 ** -23 * grad(np.abs(x), np.abs(dy)))
    assert nl2(got, want) < (0.5 * terms ** 0.5 + 1) * 2.0 ** -24
    assert np.array_equal(run(x, dy)[0], got)
    x[n // 2, 5, h - 1, w - 1], x[1, 6, 0, 0], x[2, 7, h // 2, 1], x[0, c - 1, 0, w - 1] = -np.inf, np.inf, np.nan, np.inf
    dy[n - 1, k - 1, P - 1, 4], dy[0, 3, 1, Q - 1], dy[3, 4, 2, 2] = np.inf, -np.inf, np.nan
    got = run(x, dy)[0]
    with np.errstate(all="ignore"):
        want = grad(x, dy).astype(np.float32)
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isposinf(got), np.isposinf(want)) and np.array_equal(np.isneginf(got), np.isneginf(want))
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("kind", ["normal", "relu", "positive"])
@pytest.mark.parametrize("n,c,h,w,k", [(64, 64, 56, 56, 128), (40, 150, 22, 31, 96)])
def test_weight_gradient_of_stride_two_leans_to_neither_side(singa, dev, n, c, h, w, k, kind):
    """The matrix instructions round towards minus infinity on average, which adds up over a sum unless half of the steps are negated.
    The mean error over the weights against their root mean square error: 1 / sqrt(weights), at most 0.004, where none leans, 0.34 and
    0.16 on these layers (a split is one image of an odd number of rows) with a sign for either half of a split alone."""
    import torch
    x, _, _ = operands(kind, n + c, n, c, h, w, 1, 1)
    dy = operands(kind, n + k, n, k, (h + 1) // 2, (w + 1) // 2, 1, 1)[0]
    if kind == "relu":
        dy = randn(rng(k), *dy.shape)
    hd = singa.CudnnConvHandle(singa.from_numpy(x, dev), (3, 3), (2, 2), (1, 1), c, k, False)
    W = np.zeros((k, c, 3, 3), np.float32)
    got, names = kernels_of(dev, lambda: singa.GpuConvBackwardW(*(singa.from_numpy(a, dev) for a in (dy, x, W)), hd).to_numpy())
    assert names == {"k_wgrad_oct"}
    xp = torch.nn.functional.pad(torch.from_numpy(x).double(), (1, 2, 1, 2))
    P, Q = dy.shape[2:]
    d = torch.from_numpy(dy).double().permute(1, 0, 2, 3).reshape(k, -1).contiguous()
    taps = [d @ xp[:, :, i:i + 2 * P:2, j:j + 2 * Q:2].permute(0, 2, 3, 1).reshape(-1, c) for i in range(3) for j in range(3)]
    off = got - torch.stack(taps, -1).reshape(k, c, 3, 3).numpy()
    print(kind, "mean error %+.4f of its root mean square" % (off.mean() / np.sqrt(np.mean(off ** 2))))
    assert abs(off.mean()) <= 0.05 * np.sqrt(np.mean(off ** 2))


@pytest.mark.parametrize("what", ["inf", "one inf", "overflow", "nan"])
def test_conv_wgrad_octets_time_of_non_finite_operands(singa, dev, what):
    """As the forward pass and the data gradient: no search per result."""
    n, c, h, w, k = 32, 256, 14, 14, 256
    x, W, dy = operands("normal", 3, n, c, h, w, k, 3)

    def time(x, dy):
        xd, wd, dyd = (singa.from_numpy(a, dev) for a in (x, W, dy))
        hd = singa.CudnnConvHandle(xd, (3, 3), (1, 1), (1, 1), c, k, False)
        assert kernels_of(dev, lambda: singa.GpuConvBackwardW(dyd, xd, wd, hd))[1] == {"k_wgrad_oct"}
        return seconds(dev, lambda: singa.GpuConvBackwardW(dyd, xd, wd, hd))

    plain = time(x, dy)
    value = np.float32(np.nan if what == "nan" else np.inf)
    if what == "one inf":
        dy[:, 0, 7, 7] = value
    elif what == "overflow":
        x, dy = x * np.float32(1e30), dy * np.float32(1e30)
    else:
        x[:] = value
        dy[:] = value
    got = time(x, dy)
    print(what, "%.1f us, ordinary operands %.1f" % (got * 1e6, plain * 1e6))
    assert got < 8 * plain


@pytest.mark.parametrize("what", ["inf", "one inf", "overflow", "nan", "inf weights"])
def test_strided_layers_time_of_non_finite_operands(singa, dev, what):
    """The three passes of a 3x3 layer of stride 2: a second pass over the tiles with results that are not finite, and no search per
    result."""
    n, c, h, w, k = 32, 128, 28, 28, 256
    x, W, _ = operands("normal", 3, n, c, h, w, k, 3)
    dy = operands("normal", 4, n, k, h // 2, w // 2, 1, 1)[0]
    kernels = ["k_conv_split", "k_dgrad_split2", "k_wgrad_oct"]

    def times(x, W, dy):
        xd, wd, dyd = (singa.from_numpy(a, dev) for a in (x, W, dy))
        hd = singa.CudnnConvHandle(xd, (3, 3), (2, 2), (1, 1), c, k, False)
        calls = [lambda: singa.GpuConvForward(xd, wd, None, hd), lambda: singa.GpuConvBackwardx(dyd, wd, xd, hd),
                 lambda: singa.GpuConvBackwardW(dyd, xd, wd, hd)]
        assert [kernels_of(dev, f)[1] for f in calls] == [{name} for name in kernels]
        return [seconds(dev, f) for f in calls]

    plain = times(x, W, dy)
    value = np.float32(np.nan if what == "nan" else np.inf)
    if what == "one inf":
        x[:, 0, 7, 7] = value
        dy[:, 0, 7, 7] = value
    elif what == "overflow":
        x, W, dy = x * np.float32(1e30), W * np.float32(1e10), dy * np.float32(1e30)
    elif what == "inf weights":
        W[:] = value
    else:
        x[:] = value
        dy[:] = value
    for name, got, ordinary in zip(kernels, times(x, W, dy), plain):
        print(name, what, "%.1f us, ordinary operands %.1f" % (got * 1e6, ordinary * 1e6))
        assert got < 8 * ordinary


@pytest.mark.parametrize("small,large", [(2.0 ** -116, 1.0), (2.0 ** -124, 2.0 ** 40), (2.0 ** -132, 2.0 ** 60), (1.0, 2.0 ** -116)])
def test_conv_split_operands_of_any_magnitude(singa, dev, small, large):
    """Inputs and gradients (or weights) of small magnitude, down to subnormal ones, at the error that ordinary magnitudes have: on
    three bfloat16 values alone the last bits of a number below 2^-110 are lost."""
    n, c, h, w, k = 14, 100, 20, 30, 140
    x, W, dy = operands("normal", 5, n, c, h, w, k, 3)
    x, W, dy = x * np.float32(small), W * np.float32(large), dy * np.float32(small)
    (y, ky), (dx, kx), _ = passes(singa, dev, x, W, dy)
    assert ky == {"k_conv_split"} and kx == {"k_conv_split"}
    import torch
    t = lambda a: torch.from_numpy(a).double()
    assert nl2(y, torch.nn.functional.conv2d(t(x), t(W), padding=1).numpy()) < 3e-7
    assert nl2(dx, torch.nn.functional.conv_transpose2d(t(dy), t(W), padding=1).numpy()) < 3e-7
    for a, b in ((x, dy / np.float32(small) * np.float32(large)), (x / np.float32(small) * np.float32(large), dy)):
        dw, kw = passes(singa, dev, a, W, b)[2]
        assert kw == {"k_wgrad_oct"}
        assert nl2(dw, wgrad64(a, b)) < 3e-7


def test_conv_split_weights_prepared_for_another_workspace(singa, dev):
    """The size of the workspace decides whether the split kernel runs: weights laid out for a call with one size are not taken by a
    call with another, and either call gives what it gives without preparation."""
    import ctypes as C

    from singa_amd import _lib
    lib = _lib.lib()
    n, c, h, w, k = 2, 64, 20, 22, 96
    x, W, dy = operands("normal", 4, n, c, h, w, k, 3)
    xd, wd, dyd, dxd = (singa.from_numpy(a, dev) for a in (x, W, dy, np.zeros_like(x)))
    hd = singa.CudnnConvHandle(xd, (3, 3), (1, 1), (1, 1), c, k, False)
    g = hd.geom
    full = lib.sgh_conv_workspace_bytes(C.byref(g), _lib.SGH_CONV_DGRAD)
    space = singa.from_numpy(np.zeros(full // 4 + 64, np.float32), dev)

    def dgrad(size):
        dxd.CopyFloatDataFromHostPtr(np.full_like(x, 7))
        (rc, out), names = kernels_of(dev, lambda: (lib.sgh_conv_dgrad_f32(C.byref(g), dyd.ptr, wd.ptr, dxd.ptr, space.ptr, size, dev.stream),
                                                    dxd.to_numpy()))
        assert rc == 0
        return out, names

    def prepare(size):
        item = (_lib.ConvPrepareItem * 1)()
        item[0].g, item[0].W, item[0].workspace, item[0].ws_bytes = C.pointer(g), wd.ptr, space.ptr, size
        assert lib.sgh_conv_dgrad_prepare_multi(item, 1, 0, dev.stream) == 0

    plain = full
    while dgrad(plain)[1] == {"k_conv_split"}:   # (a size that is too little for it and enough for the fp32 kernel)
        plain //= 2
    want = {size: dgrad(size) for size in (full, plain)}
    assert want[full][1] == {"k_conv_split"} and want[plain][1] == {"k_dgrad3x3"}
    for prepared in (full, plain):
        for called in (full, plain):
            prepare(prepared)
            got, names = dgrad(called)
            assert names == want[called][1] and np.array_equal(got, want[called][0]), (prepared, called)


def test_conv_wgrad_octets_workspace_is_an_image_per_cu(dev):
    """The partial images of the octet kernel: one for each of the card's 256 CUs at most, however many pixels there are."""
    import ctypes as C

    from singa_amd import _lib
    lib, cus = _lib.lib(), 256
    for n, c, h, w, k in WGRAD_OCTET_LAYERS + [(37, 71, 106, 112, 132), (64, 154, 37, 27, 670), (128, 64, 112, 112, 64)]:
        g = _lib.ConvGeom()
        assert lib.sgh_conv_geom_init(C.byref(g), n, c, h, w, k, 3, 3, 1, 1, 1, 1) == 0
        tiles = ((k + 63) // 64) * ((c + 63) // 64) * ((w + 31) // 32)
        assert lib.sgh_conv_workspace_bytes(C.byref(g), _lib.SGH_CONV_WGRAD) <= max(cus, tiles) * 64 * 64 * 9 * 4
