"""The tile convolution kernel (GPU) against fp64: channel counts around its 16- and 32-channel
steps and 64-channel tiles, ragged images, strides, dilations, depth, a fused residual, BatchNorm
and ReLU, and in fp32 (computed as bf16 plane products) non-finite values.

Bars (2-norm): fp32 sums of K products, 2^-23 sqrt(K); 16-bit results: half an ulp of the output
(2^-9 bf16, 2^-12 fp16) on each value, doubled."""

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu
DEV = "cuda"
OUT_BAR = {torch.float32: 0.0, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}


def _params(mod, dtype):
    return mod.weight.detach().to(dtype).double(), mod.bias.detach().to(dtype).double()


def _check(got, ref, k):
    assert got.shape == ref.shape
    assert not torch.isnan(got).any()
    err = ((got.double() - ref).norm() / ref.norm()).item()
    bar = 2.0 ** -23 * k ** 0.5 + OUT_BAR[got.dtype]
    assert err <= bar, (err, bar)


# n, b, ci, co, kernel, stride, padding, dilation, h, w
SHAPES = [(2, 2, 1, 1, (3, 3), 1, 1, 1, 9, 11), (1, 3, 16, 33, (3, 3), 1, 1, 1, 16, 16), (3, 1, 17, 64, (1, 1), 1, 0, 1, 13, 10),
          (2, 1, 31, 65, (3, 3), 2, 1, 1, 33, 35), (2, 2, 33, 40, (5, 5), 1, 2, 1, 12, 130), (1, 1, 64, 31, (3, 3), 1, 2, 2, 20, 20),
          (2, 1, 40, 100, (7, 7), 2, 3, 1, 31, 29), (4, 2, 96, 64, (1, 3), 1, 0, 1, 1, 70), (1, 2, 48, 16, (3, 1), (2, 1), 1, 1, 40, 5),
          (2, 1, 32, 32, (3, 3), 1, 1, 1, 1, 1), (1, 1, 8, 24, (4, 6), 3, 2, 1, 50, 64), (2, 1, 16, 16, (3, 3), 1, 0, 5, 30, 31)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,b,ci,co,kernel,stride,pad,dil,h,w", SHAPES)
def test_conv_tile_shapes(hip, n, b, ci, co, kernel, stride, pad, dil, h, w, dtype):
    import wide_compiler as wc
    torch.manual_seed(ci * 100 + co)
    mods = [nn.Conv2d(ci, co, kernel, stride=stride, padding=pad, dilation=dil) for _ in range(n)]
    wide = wc.WideConv2d.from_modules(mods).to(DEV, dtype)
    x = torch.randn(n, b, ci, h, w).to(dtype)
    with torch.no_grad():
        got = wide(x.to(DEV))
        refs = []
        for q, m in enumerate(mods):
            wt, bias = _params(m, dtype)
            refs.append(nn.functional.conv2d(x[q].double(), wt, bias, m.stride, m.padding, m.dilation))
    _check(got.cpu(), torch.stack(refs), ci * kernel[0] * kernel[1])


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
def test_conv_tile_depth(hip, dtype):
    import wide_compiler as wc
    torch.manual_seed(1)
    mods = [nn.Conv3d(20, 36, (3, 2, 3), stride=(2, 1, 1), padding=(1, 0, 1)) for _ in range(2)]
    wide = wc.WideConv3d.from_modules(mods).to(DEV, dtype)
    x = torch.randn(2, 2, 20, 7, 9, 14).to(dtype)
    with torch.no_grad():
        got = wide(x.to(DEV))
        refs = []
        for q, m in enumerate(mods):
            wt, bias = _params(m, dtype)
            refs.append(nn.functional.conv3d(x[q].double(), wt, bias, m.stride, m.padding))
    _check(got.cpu(), torch.stack(refs), 20 * 18)


@pytest.mark.parametrize("hw", [12, 13])
def test_conv_tile_fused_epilogue(hip, hw):
    """conv - BN - (+ residual) - ReLU in one launch, with 16-byte rows (12) and without (13)."""
    from wide_compiler import _hip
    torch.manual_seed(2)
    n, b, ci, co = 3, 2, 24, 40
    x, r = torch.randn(n, b, ci, hw, hw, device=DEV), torch.randn(n, b, co, hw, hw, device=DEV)
    wt = torch.randn(n * co, ci, 3, 3, device=DEV) * 0.1
    bias, g, be, mu = (torch.randn(n * co, device=DEV) for _ in range(4))
    var = torch.rand(n * co, device=DEV) + 0.5
    y = torch.full((n, b, co, hw, hw), float("nan"), device=DEV)
    _hip.conv2d(x=x, weight=wt, n=n, c_in=ci, c_out=co, kernel=(3, 3), stride=(1, 1), padding=(1, 1),
                dilation=(1, 1), y=y, bias=bias, bn=(g, be, mu, var, 1e-5), residual=r, relu=True)
    refs = []
    for q in range(n):
        s = slice(q * co, (q + 1) * co)
        v = nn.functional.conv2d(x[q].double().cpu(), wt[s].double().cpu(), bias[s].double().cpu(), padding=1)
        a = [t[s].double().cpu()[None, :, None, None] for t in (mu, var, g, be)]
        refs.append(torch.relu((v - a[0]) / (a[1] + 1e-5).sqrt() * a[2] + a[3] + r[q].double().cpu()))
    _check(y.cpu(), torch.stack(refs), ci * 9)


def test_conv_tile_fp32_special_values(hip):
    """Infinities, NaN and values above the largest bf16 reach exactly the outputs that read them."""
    import wide_compiler as wc
    torch.manual_seed(3)
    mods = [nn.Conv2d(20, 40, 3, padding=1) for _ in range(5)]
    wide = wc.WideConv2d.from_modules(mods).to(DEV)
    x = torch.randn(5, 2, 20, 17, 19)
    x[0, 0, 3, 5, 6] = float("inf")
    x[1, 1, 19, 16, 18] = float("nan")
    x[2, 0, 0, 0, 0] = torch.finfo(torch.float32).max        # an infinity as a bf16
    with torch.no_grad():
        wide.grouped_conv.weight[3 * 40 + 7, 2, 1, 1] = -float("inf")
        mods[3].weight[7, 2, 1, 1] = -float("inf")
        got = wide(x.to(DEV)).cpu()
        ref = torch.stack([nn.functional.conv2d(x[q].double(), m.weight.double(), m.bias.double(), padding=1)
                           for q, m in enumerate(mods)])
    f = ref.float()
    assert torch.equal(torch.isnan(got), torch.isnan(f))
    assert torch.equal(torch.isinf(got), torch.isinf(f))
    assert torch.equal(torch.sign(got[torch.isinf(got)]), torch.sign(f[torch.isinf(f)]))
    for q in range(5):
        ok = torch.isfinite(f[q]) & (f[q].abs() < 1e30)
        err = ((got[q][ok].double() - ref[q][ok]).norm() / ref[q][ok].norm()).item()
        assert err <= 2.0 ** -23 * 180 ** 0.5


def test_conv_tile_fp32_infinite_weight_meets_padding(hip):
    """A padding pixel is a zero like any other: times an infinite weight it is NaN, so the border
    outputs whose window holds that tap over the padding are NaN and the others infinite."""
    import wide_compiler as wc
    torch.manual_seed(4)
    mods = [nn.Conv2d(20, 40, 3, padding=1) for _ in range(2)]
    x = torch.randn(2, 2, 20, 17, 19)
    with torch.no_grad():
        mods[1].weight[7, 2, 0, 0] = float("inf")
        wide = wc.WideConv2d.from_modules(mods).to(DEV)
        got = wide(x.to(DEV)).cpu()
        refs = []
        for q, m in enumerate(mods):
            cols = nn.functional.unfold(x[q].double(), 3, padding=1)
            ref = (m.weight.double().flatten(1) @ cols + m.bias.double()[:, None]).view(2, 40, 17, 19)
            refs.append(ref)
    f = torch.stack(refs).float()
    assert torch.isnan(f[1, :, 7, 0]).all() and torch.isinf(f[1, :, 7, 1:, 1:]).all()
    assert torch.equal(torch.isnan(got), torch.isnan(f))
    assert torch.equal(torch.isinf(got), torch.isinf(f))


@pytest.mark.parametrize("ci,co,hw", [(20, 40, 17), (40, 70, 30), (16, 24, 9)])
@pytest.mark.parametrize("xs,ws", [(2.0 ** -107, 1.0), (2.0 ** -112, 1.0), (2.0 ** -120, 1.0), (2.0 ** -138, 1.0),
                                   (1.0, 2.0 ** -118), (2.0 ** -118, 2.0 ** 60), (2.0 ** -58, 2.0 ** -62)])
def test_conv_tile_fp32_small_values(hip, ci, co, hw, xs, ws):
    """Values below what three bf16 planes carry in one image or in some filters, beside ordinary ones and zeros:
    every image and filter keeps the fp32 bar.  Subnormal results have steps of 2^-149 besides: 2 K roundings of
    at most half a step each add 2^-150 sqrt(2 K) in the root mean square."""
    from wide_compiler import _hip
    torch.manual_seed(6)
    n, b = 3, 2
    x = torch.randn(n, b, ci, hw, hw, device=DEV)
    w = torch.randn(n * co, ci, 3, 3, device=DEV)
    if xs < ws:
        x[:, 1] *= xs
        w *= ws
        x[:, 1, 3] = 0.0
    else:
        w[::3] *= ws
        x *= xs
    y = torch.full((n, b, co, hw, hw), float("nan"), device=DEV)
    _hip.conv2d(x=x, weight=w, n=n, c_in=ci, c_out=co, kernel=(3, 3), stride=(1, 1), padding=(1, 1), dilation=(1, 1),
                y=y, bias=None)
    got = y.double().cpu().reshape(n, b, co, -1)
    ref = torch.stack([nn.functional.conv2d(x[q].double().cpu(), w[q * co:(q + 1) * co].double().cpu(), padding=1)
                       for q in range(n)]).reshape(n, b, co, -1)
    for image in range(b):
        for at in range(3):
            g, r = (t.reshape(n, b, co, -1)[:, image].reshape(n * co, -1)[at::3] for t in (got, ref))
            bar = 2.0 ** -23 * (9 * ci) ** 0.5 + 2.0 ** -150 * (18 * ci * r.numel()) ** 0.5 / r.norm().item()
            assert ((g - r).norm() / r.norm()).item() <= bar, (image, at)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,b,ci,co,h,w,kh,kw,stride,pad", [
    (2, 3, 3, 40, 9, 12, 3, 3, 1, 1),        # rows of 27 values; channels past a tile's first 32
    (3, 1, 17, 70, 13, 7, 3, 3, 2, 1),       # one channel past an MFMA step, two channel tiles
    (1, 2, 33, 16, 1, 132, 1, 3, 1, 1),      # one channel in the second chunk
    (4, 2, 128, 40, 8, 8, 1, 1, 1, 0),       # a tap only, four chunks
    (2, 1, 53, 24, 21, 7, 3, 1, 2, 1),       # rows of 159 values, a partial chunk
])
def test_conv_tile_reads_the_filter_bank(hip, dtype, n, b, ci, co, h, w, kh, kw, stride, pad):
    """Few tiles: the filters read in their own layout give the packed layout's result bit for bit,
    also at an address of element alignment; a packed-only size says so."""
    from wide_compiler import _hip
    torch.manual_seed(5)
    x = torch.randn(n, b, ci, h, w, device=DEV).to(dtype)
    store = (torch.randn(n * co * ci * kh * kw + 1, device=DEV) * 0.1).to(dtype)
    bias = torch.randn(n * co, device=DEV).to(dtype)
    ph, pw = (0 if kh == 1 else pad), (0 if kw == 1 else pad)
    ho, wo = (h + 2 * ph - kh) // stride + 1, (w + 2 * pw - kw) // stride + 1
    for at in (0, 1):
        wt = store[at:at + n * co * ci * kh * kw].view(n * co, ci, kh, kw)
        got = [torch.full((n, b, co, ho, wo), float("nan"), dtype=dtype, device=DEV) for _ in range(2)]
        packs = []
        real = _hip.conv_pack_weights
        try:
            _hip.conv_pack_weights = lambda *a: (packs.append(1), real(*a))[1]
            for y, packed in zip(got, (False, True)):
                _hip.conv2d(x=x, weight=wt, n=n, c_in=ci, c_out=co, kernel=(kh, kw), stride=(stride, stride),
                            padding=(ph, pw), dilation=(1, 1), y=y, bias=bias, packed=packed)
        finally:
            _hip.conv_pack_weights = real
        assert len(packs) == 1                                # the packed call only
        assert torch.equal(got[0], got[1])
        ref = torch.stack([nn.functional.conv2d(x[q].double().cpu(), wt[q * co:(q + 1) * co].double().cpu(),
                                                bias[q * co:(q + 1) * co].double().cpu(), stride, (ph, pw))
                           for q in range(n)])
        _check(got[0].cpu(), ref, ci * kh * kw)
