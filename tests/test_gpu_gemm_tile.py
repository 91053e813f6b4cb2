"""The 128x128 / 64x64 tile kernel of the grouped GEMM (GPU) against fp64, at the sizes where it can
go wrong: edges of tiles and K steps, rows at element alignment, short k, residual, ReLU, strided
rows, and for fp32 (computed as bf16 plane products) infinities, NaN and the ends of the exponent
range.

Bars (2-norm): fp32 sums of k products, each product and each of the k / 2 or fewer additions
rounded to 2^-24 of a partial sum: 2^-23 sqrt(k) covers it.  16-bit results: half an ulp of the output
(2^-9 bf16, 2^-12 fp16) on each value, doubled."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
OUT_BAR = {torch.float32: 0.0, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}


def _run(x, w, b, out_dtype=None, relu=False, residual=None, rows_inner=None):
    """x [N, M, K] (any strides with unit inner stride), w [N, O, K] contiguous."""
    from wide_compiler import _hip
    n, m, k = x.shape
    o = w.shape[1]
    c = torch.full((n, m, o), float("nan"), device=DEV, dtype=out_dtype or x.dtype)
    _hip.grouped_gemm(n=n, m=m, o=o, k=k, a=x, a_sn=x.stride(0), a_so=0, a_si=x.stride(1), a_rows_inner=m,
                      w=w, w_sn=o * k, c=c, c_sn=m * o, c_so=0, c_si=o, c_rows_inner=m, bias=b, bias_sn=o,
                      relu=relu, residual=residual, r_sn=m * o, r_so=0, r_si=o)
    return c


def _ref(x, w, b, relu=False, residual=None):
    y = torch.bmm(x.double(), w.double().transpose(1, 2).contiguous())
    if b is not None:
        y = y + b.double()[:, None, :]
    if residual is not None:
        y = y + residual.double()
    return torch.relu(y) if relu else y


def _check(got, ref, k):
    bar = 2.0 ** -23 * max(k, 1) ** 0.5 + OUT_BAR[got.dtype]
    assert not torch.isnan(got).any()
    err = ((got.double() - ref).norm() / ref.norm()).item()
    assert err <= bar, (err, bar)


# n, m, o, k: 128 x 128 tiles from 512 of them on, 64 x 64 from 192 (fp32) or 256 / k > 64 (16-bit) on
SHAPES = [(130, 129, 128, 33), (512, 127, 128, 7), (70, 256, 255, 65), (600, 128, 128, 1), (20, 800, 1000, 300),
          (200, 64, 63, 64), (100, 65, 64, 31), (48, 64, 256, 100), (49, 33, 255, 129), (192, 33, 33, 16)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,m,o,k", SHAPES)
def test_tile_gemm_edges(hip, n, m, o, k, dtype):
    torch.manual_seed(n + m + o + k)
    x = torch.randn(n, m, k, device=DEV).to(dtype)
    w = torch.randn(n, o, k, device=DEV).to(dtype)
    b = torch.randn(n, o, device=DEV).to(dtype)
    r = torch.randn(n, m, o, device=DEV).to(dtype)
    _check(_run(x, w, b), _ref(x, w, b), k)
    _check(_run(x, w, None, relu=True, residual=r), _ref(x, w, None, True, r), k)
    if dtype != torch.float32:
        _check(_run(x, w, b.float(), out_dtype=torch.float32), _ref(x, w, b), k)
    # rows at element alignment: x starts one element into a wider, odd-pitched buffer
    wide = torch.randn(n, m, k + 3, device=DEV).to(dtype)
    _check(_run(wide[:, :, 1:k + 1], w, b), _ref(wide[:, :, 1:k + 1], w, b), k)


def test_tile_gemm_packed_rows(hip):
    """The channel-packed input view [N, B, T, K] (rows in two strides) through WideLinear."""
    import wide_compiler as wc
    torch.manual_seed(3)
    n, b, t, i, o = 24, 40, 9, 40, 200
    mods = [torch.nn.Linear(i, o) for _ in range(n)]
    wide = wc.WideLinear.from_modules(mods).to(DEV)
    x = torch.randn(b, t, n, i, device=DEV).permute(2, 0, 1, 3)
    with torch.no_grad():
        y = wide(x)
    ref = torch.stack([m.to(DEV).double()(x[q].double()) for q, m in enumerate(mods)])
    _check(y, ref, i)


@pytest.mark.parametrize("n,m,o,k", [(130, 128, 128, 64), (200, 64, 64, 40), (520, 128, 128, 64)])
def test_tile_gemm_fp32_special_values(hip, n, m, o, k):
    """Infinities, NaN, values above the largest bf16 and overflowing sums give what fp32 arithmetic gives;
    rows without them keep their values to the fp32 bar."""
    torch.manual_seed(5)
    x = torch.randn(n, m, k, device=DEV)
    w = torch.randn(n, o, k, device=DEV)
    top = torch.finfo(torch.float32).max
    x[0, 3, 5] = float("inf")
    x[1, 7, k - 1] = float("-inf")
    x[2, 0, 0] = float("nan")
    w[3, 4, 1] = float("inf")
    x[4, 1] = 0.0
    x[4, 1, 2] = top                               # rounds up to infinity as a bf16
    w[4, :, 2] = 0.5
    x[5, 2] = top / 2                              # sums overflow
    w[5, 6] = 1.0
    got = _run(x, w, None)
    ref = torch.bmm(x.double(), w.double().transpose(1, 2).contiguous())
    ref32 = ref.float()                            # overflows to infinity where fp32 does
    for q in range(6):
        a, e = got[q], ref32[q]
        if q == 5:
            assert torch.isinf(a[2, 6]) and a[2, 6] > 0
            a, e = torch.cat([a[:2], a[3:]]), torch.cat([e[:2], e[3:]])
        assert torch.equal(torch.isnan(a), torch.isnan(e)), q
        assert torch.equal(torch.isinf(a), torch.isinf(e)), q
        assert torch.equal(torch.sign(a[torch.isinf(a)]), torch.sign(e[torch.isinf(e)])), q
        ok = torch.isfinite(e)
        err = ((a[ok] - e[ok]).double().norm() / e[ok].double().norm()).item()
        assert err <= 2.0 ** -23 * k ** 0.5, (q, err)
    _check(got[6:], ref[6:], k)


@pytest.mark.parametrize("scale", [2.0 ** -60, 2.0 ** 60])
def test_tile_gemm_fp32_range(hip, scale):
    torch.manual_seed(6)
    x = torch.randn(130, 128, 48, device=DEV) * scale
    w = torch.randn(130, 128, 48, device=DEV)
    _check(_run(x, w, None), _ref(x, w, None), 48)


@pytest.mark.parametrize("n,m,o,k", [(520, 128, 128, 72), (200, 64, 64, 40)])
@pytest.mark.parametrize("xs,ws", [(2.0 ** -107, 1.0), (2.0 ** -112, 1.0), (2.0 ** -120, 1.0), (2.0 ** -126, 1.0),
                                   (2.0 ** -138, 1.0), (1.0, 2.0 ** -118), (2.0 ** -118, 2.0 ** 60),
                                   (2.0 ** -118, 2.0 ** 100), (2.0 ** 30, 2.0 ** -118), (2.0 ** -58, 2.0 ** -62)])
def test_tile_gemm_fp32_small_values(hip, n, m, o, k, xs, ws):
    """Values below what three bf16 planes carry, alone and beside ordinary ones and zeros: every row and column
    keeps the fp32 bar.  Subnormal results have steps of 2^-149 besides: 2 k roundings (products and sums) of at most
    half a step each add 2^-150 sqrt(2 k) in the root mean square."""
    torch.manual_seed(7)
    x = torch.randn(n, m, k, device=DEV)
    w = torch.randn(n, o, k, device=DEV)
    if xs < ws:
        x[:, 1::2] *= xs                               # every other row
        w *= ws
        x[:, 5] = 0.0
    else:
        w[:, ::3] *= ws
        x *= xs
        x[:, :, :4] = 0.0
    got, ref = _run(x, w, None).double(), _ref(x, w, None)
    for rows, cols in ((slice(1, None, 2), slice(None)), (slice(0, None, 2), slice(None)),
                       (slice(None), slice(0, None, 3)), (slice(None), slice(1, None, 3))):
        g, r = got[:, rows, cols], ref[:, rows, cols]
        bar = 2.0 ** -23 * k ** 0.5 + 2.0 ** -150 * (2 * k * r.numel()) ** 0.5 / r.norm().item()
        assert ((g - r).norm() / r.norm()).item() <= bar, (rows, cols)
    assert (got[:, 5] == 0.0).all() or xs >= ws


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,m,k,o1,o2", [(40, 200, 96, 128, 256), (100, 65, 40, 64, 128), (3, 20, 64, 32, 64),
                                         (2, 33, 48, 50, 100), (5, 1, 16, 96, 7), (64, 260, 64, 192, 384),
                                         (32, 1024, 64, 256, 512)])
def test_gemm_pair(hip, n, m, k, o1, o2, dtype):
    """Two weights and one output: splits on a tile of every kernel and off them, with and without bias,
    equal to two separate calls to the bar and to fp64."""
    from wide_compiler import _hip
    torch.manual_seed(n + m + o1)
    x = torch.randn(n, m, k, device=DEV).to(dtype)
    w1, w2 = torch.randn(n, o1, k, device=DEV).to(dtype), torch.randn(n, o2, k, device=DEV).to(dtype)
    b1, b2 = torch.randn(n, o1, device=DEV).to(dtype), torch.randn(n, o2, device=DEV).to(dtype)
    for p1, p2 in ((b1, b2), (None, None), (b1, None), (None, b2)):
        c = torch.full((n, m, o1 + o2), float("nan"), device=DEV, dtype=dtype)
        _hip.grouped_gemm_pair(n=n, m=m, k=k, o1=o1, o2=o2, a=x, a_sn=m * k, a_so=0, a_si=k, a_rows_inner=m,
                               w1=w1, bias1=p1, w2=w2, bias2=p2, c=c)
        _check(c, torch.cat([_ref(x, w1, p1), _ref(x, w2, p2)], -1), k)
