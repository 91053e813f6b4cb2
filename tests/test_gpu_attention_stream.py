"""The streaming 16-bit attention kernel (GPU) against fp64 and against the general kernel, which a
mask of zeros selects: head dims on both sides of its padded widths, ragged numbers of queries
and keys around its 32-key blocks and 64-key tiles, causal and full, cross lengths, non-finite
values.

Bar: P and the output are each rounded to the operand type (half an ulp, 2^-9 bf16 / 2^-12 fp16
relative, on every value), Q K^T is exact products in fp32; the 2-norm error against fp64 stays
under twice the sum of the two, and under 1.1 times the general kernel's."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
BAR = {torch.bfloat16: 4 * 2.0 ** -9, torch.float16: 4 * 2.0 ** -12}


def _attend(q, k, v, heads, causal, masked):
    """q [nb, sq, d], k / v [nb, skv, d] views with unit inner stride."""
    from wide_compiler import _hip
    nb, sq, d = q.shape
    skv = k.shape[1]
    o = torch.full((nb, sq, d), float("nan"), device=DEV, dtype=q.dtype)
    mask = None
    if masked:
        mask = torch.zeros(1, 1, sq, skv, device=DEV)
        if causal:
            mask = mask.masked_fill(torch.ones(sq, skv, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
        mask = mask.expand(nb, heads, sq, skv)
    _hip.attention(q=q, k=k, v=v, o=o, nb=nb, heads=heads, sq=sq, skv=skv, head_dim=d // heads,
                   q_strides=q.stride()[:2], k_strides=k.stride()[:2], v_strides=v.stride()[:2],
                   o_strides=(sq * d, d), scale=(d // heads) ** -0.5, causal=causal and not masked, mask=mask)
    return o


def _ref(q, k, v, heads, causal):
    nb, sq, d = q.shape
    skv = k.shape[1]
    split = lambda t, s: t.double().reshape(nb, s, heads, d // heads).transpose(1, 2).contiguous()  # noqa: E731
    a = split(q, sq) @ split(k, skv).transpose(2, 3).contiguous() * (d // heads) ** -0.5
    if causal:
        a = a.masked_fill(torch.ones(sq, skv, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    return (torch.softmax(a, -1) @ split(v, skv)).transpose(1, 2).reshape(nb, sq, d)


def _err(a, b):
    return ((a.double() - b).norm() / b.norm()).item()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nb,heads,dh,s", [
    (3, 2, 8, 31), (2, 3, 16, 64), (1, 2, 24, 65), (2, 8, 32, 128), (4, 4, 32, 129), (1, 5, 40, 33),
    (2, 2, 48, 257), (3, 2, 64, 1), (1, 1, 64, 63), (5, 8, 64, 96), (2, 8, 64, 300), (3, 1, 72, 127), (2, 2, 96, 66),
    (1, 3, 120, 190), (2, 4, 128, 255), (64, 8, 64, 256), (32, 8, 32, 250), (40, 8, 96, 512)])
def test_stream_attention(hip, nb, heads, dh, s, causal, dtype):
    torch.manual_seed(nb * 1000 + dh + s)
    d = heads * dh
    qkv = torch.randn(nb, s, 3 * d, device=DEV).to(dtype)
    q, k, v = qkv[..., :d], qkv[..., d:2 * d], qkv[..., 2 * d:]
    ref = _ref(q, k, v, heads, causal)
    got = _attend(q, k, v, heads, causal, False)
    assert not torch.isnan(got).any()
    e, general = _err(got, ref), _err(_attend(q, k, v, heads, causal, True), ref)
    assert e <= BAR[dtype], (e, general)
    assert e <= 1.1 * general + 2.0 ** -16, (e, general)


@pytest.mark.parametrize("sq,skv,causal", [(1, 300, False), (37, 1000, False), (300, 37, False), (70, 200, True),
                                           (200, 70, True), (130, 1, False)])
def test_stream_cross_lengths(hip, sq, skv, causal):
    torch.manual_seed(sq + skv)
    heads, dh = 4, 64
    q = torch.randn(3, sq, heads * dh, device=DEV).to(torch.bfloat16)
    kv = torch.randn(3, skv, 2 * heads * dh, device=DEV).to(torch.bfloat16)
    k, v = kv[..., :heads * dh], kv[..., heads * dh:]
    ref = _ref(q, k, v, heads, causal)
    got = _attend(q, k, v, heads, causal, False)
    assert _err(got, ref) <= BAR[torch.bfloat16]


def test_stream_growing_scores(hip):
    """Scores that grow along the keys move the running maximum in every tile; large ones leave
    one key with all the weight."""
    torch.manual_seed(9)
    heads, dh, s = 2, 64, 333
    q = torch.randn(2, s, heads * dh, device=DEV)
    k = torch.randn(2, s, heads * dh, device=DEV) * torch.linspace(0.1, 12, s, device=DEV)[None, :, None]
    v = torch.randn(2, s, heads * dh, device=DEV)
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    for causal in (False, True):
        assert _err(_attend(q, k, v, heads, causal, False), _ref(q, k, v, heads, causal)) <= BAR[torch.bfloat16]


def test_stream_non_finite_values(hip):
    """A NaN or infinity in one key, query or value reaches the rows that attend to it, and no row of
    another head or batch entry."""
    torch.manual_seed(10)
    heads, dh, s = 2, 48, 100
    q, k, v = (torch.randn(4, s, heads * dh, device=DEV).to(torch.bfloat16) for _ in range(3))
    clean = _attend(q, k, v, heads, False, False)
    q[0, 5, 3] = float("nan")
    k[1, 7, 50] = float("nan")
    v[2, 99, 1] = float("inf")
    got = _attend(q, k, v, heads, False, False)
    nan = torch.isnan(got)
    assert nan[0, 5, :dh].all() and not nan[0, :5].any() and not nan[0, 6:].any() and not nan[0, 5, dh:].any()
    assert nan[1, :, dh:].all() and not nan[1, :, :dh].any()
    assert torch.isinf(got[2, :, 1]).all() and torch.equal(got[2, :, 2:], clean[2, :, 2:])
    assert torch.equal(got[3], clean[3])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dh,skv,causal", [(64, 2047, False), (64, 2048, True), (40, 1000, False), (128, 513, False)])
def test_stream_row_sum_is_32_bit(hip, dh, skv, causal, dtype):
    """The row sum takes P before it is rounded for P V.  One key holds the row's largest score and the
    only non-zero value, so P V is exactly 1 and the output 1 / l; the other keys of a row all have
    the same P, whose rounding, were it in l, would not average out.  Bar: half an ulp of the output
    type, and 2^-18 for fp32's share (the exponential, its argument, 2,048 additions in two chains)."""
    torch.manual_seed(dh + skv)
    nb, sq = 2, 256 if not causal else skv
    q = torch.zeros(nb, sq, dh, device=DEV)
    q[:, :, 0] = torch.rand(nb, sq, device=DEV) * 4.0 + 0.5
    k = torch.zeros(nb, skv, dh, device=DEV)
    k[:, 0, 0] = dh ** 0.5
    v = torch.zeros(nb, skv, dh, device=DEV)
    v[:, 0] = 1.0
    q, k, v = (t.to(dtype) for t in (q, k, v))
    got = _attend(q, k, v, 1, causal, False).double()
    d = q[:, :, 0].double() * k[0, 0, 0].double() * dh ** -0.5
    others = torch.arange(sq, device=DEV).double() if causal else float(skv - 1)
    ref = (1.0 / (1.0 + others * torch.exp(-d)))[:, :, None]
    half_ulp = torch.exp2(torch.floor(torch.log2(ref))) * (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11)
    assert ((got - ref).abs() <= half_ulp + 2.0 ** -18 * ref).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,blocked", [(torch.bfloat16, 64), (torch.bfloat16, 150), (torch.float16, 128)])
def test_stream_first_scores_are_minus_infinity(hip, dtype, blocked, causal):
    """Keys whose score is -infinity (an overflow in bf16, an infinite key in fp16) weigh nothing, also when they
    come first and the scores after them lie far below zero: the row's maximum is the largest of the
    finite ones.  Every score is the same but theirs, so the output is the mean of the other values."""
    heads, dh, s = 2, 64, 260
    torch.manual_seed(blocked)
    q = torch.zeros(2, s, heads, dh, device=DEV)
    k = torch.zeros(2, s, heads, dh, device=DEV)
    if dtype == torch.bfloat16:
        q[..., 0] = 1e20
        k[..., 0] = -2e-17                                  # scores of -250
        k[:, :blocked, :, 0] = -1e20
    else:
        q[..., 0] = 100.0
        k[..., 0] = -20.0
        k[:, :blocked, :, 0] = -float("inf")
    q, k = (t.view(2, s, heads * dh).to(dtype) for t in (q, k))
    v = torch.randn(2, s, heads * dh, device=DEV).to(dtype)
    got = _attend(q, k, v, heads, causal, False).double()
    sums = v.double()[:, blocked:].cumsum(1)
    if causal:
        ref = sums / torch.arange(1, s - blocked + 1, device=DEV).double()[:, None]
        got = got[:, blocked:]                              # rows that see no other key have no defined value
    else:
        ref = (sums[:, -1:] / (s - blocked)).expand(2, s, heads * dh)
    assert _err(got, ref) <= BAR[dtype]


@pytest.mark.parametrize("s,heads,fewer", [
    (1000, 128, 125),             # K and V of one workgroup fill a CU's LDS: a full round, and all but 6 of its places
    (1000, 256, 230),             # two rounds
    (512, 256, 200),              # two workgroups share a CU's LDS
])
def test_resident_and_streaming_kernels_share_a_range(hip, s, heads, fewer):
    """bf16, head dim 32: the choice between the resident and the streaming kernel follows how full the chip is, not one
    number of workgroups: a few heads less take the same kernel (the same bits), and either keeps the bar."""
    torch.manual_seed(s)
    q, k, v = (torch.randn(heads, s, 32, device=DEV).to(torch.bfloat16) for _ in range(3))
    full = _attend(q, k, v, 1, False, False)
    part = _attend(q[:fewer], k[:fewer], v[:fewer], 1, False, False)
    few = _attend(q[:20], k[:20], v[:20], 1, False, False)
    assert torch.equal(part, full[:fewer])
    ref = _ref(q[:20], k[:20], v[:20], 1, False)
    for got in (full[:20], few):
        assert _err(got, ref) <= BAR[torch.bfloat16]
