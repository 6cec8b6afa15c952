"""The fp32 convolutions on split operands (conv_split.hip, wgrad_oct.hip) against what fp32 instructions would give: the error of
their sums over the operands that networks have."""
import ctypes as C

import numpy as np
import pytest

from util import nl2, randn, rng

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def singa():
    from singa_amd import singa_wrap
    return singa_wrap


def kernels_of(dev, call):
    """(result of `call`, names of the kernels that it was timed on)"""
    from singa_amd import _lib
    lib, n, buf = _lib.lib(), C.c_int(), C.create_string_buffer(64)
    dev.Sync()
    lib.sgh_prof_clear()
    _lib.check(lib.sgh_prof_enable(1), "sgh_prof_enable")
    try:
        out = call()
        dev.Sync()
        _lib.check(lib.sgh_prof_count(C.byref(n)), "sgh_prof_count")
        names, ms, work = set(), C.c_float(), C.c_double()
        for i in range(n.value):
            _lib.check(lib.sgh_prof_get(i, buf, 64, C.byref(ms), C.byref(work)), "sgh_prof_get")
            names.update(buf.value.decode().split("/")[1:])   # ("class/kernel"; the record of a whole entry point has no kernel)
    finally:
        lib.sgh_prof_enable(0)
        lib.sgh_prof_clear()
    return out, names


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
