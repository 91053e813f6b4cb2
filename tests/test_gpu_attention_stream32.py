"""The streaming fp32 attention kernel (GPU; bf16 plane products) against fp64 and against the
general kernel, which a mask of zeros selects: head dims up to 64, ragged numbers of queries and
keys around its 64-key tiles and 128-query workgroups, causal and full, cross lengths, non-finite
values.

Bar: at most the general kernel's 2-norm error (plus 2^-24, the rounding of the result), which
sums the same products in fp32."""

import pytest
import torch

from tests.test_gpu_attention_stream import _attend, _err, _ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nb,heads,dh,s", [
    (3, 2, 4, 31), (2, 3, 12, 64), (1, 2, 16, 65), (2, 8, 32, 128), (4, 4, 32, 129), (1, 5, 36, 33), (2, 2, 48, 257),
    (3, 2, 64, 1), (1, 1, 64, 63), (5, 8, 64, 96), (2, 8, 60, 300), (40, 8, 32, 250)])
def test_stream32_attention(hip, nb, heads, dh, s, causal):
    torch.manual_seed(nb * 1000 + dh + s)
    d = heads * dh
    qkv = torch.randn(nb, s, 3 * d, device=DEV)
    q, k, v = qkv[..., :d], qkv[..., d:2 * d], qkv[..., 2 * d:]
    ref = _ref(q, k, v, heads, causal)
    got = _attend(q, k, v, heads, causal, False)
    assert not torch.isnan(got).any()
    e, general = _err(got, ref), _err(_attend(q, k, v, heads, causal, True), ref)
    assert e <= general + 2.0 ** -24, (e, general)


@pytest.mark.parametrize("sq,skv,causal", [(1, 300, False), (37, 1000, False), (300, 37, False), (70, 200, True),
                                           (200, 70, True), (130, 1, False)])
def test_stream32_cross_lengths(hip, sq, skv, causal):
    torch.manual_seed(sq + skv)
    heads, dh = 4, 64
    q = torch.randn(3, sq, heads * dh, device=DEV)
    kv = torch.randn(3, skv, 2 * heads * dh, device=DEV)
    k, v = kv[..., :heads * dh], kv[..., heads * dh:]
    ref = _ref(q, k, v, heads, causal)
    e, general = _err(_attend(q, k, v, heads, causal, False), ref), _err(_attend(q, k, v, heads, causal, True), ref)
    assert e <= general + 2.0 ** -24, (e, general)


def test_stream32_growing_scores(hip):
    """Scores that grow along the keys move the running maximum in every tile."""
    torch.manual_seed(9)
    heads, dh, s = 2, 64, 333
    q, k, v = (torch.randn(2, s, heads * dh, device=DEV) for _ in range(3))
    k = k * torch.linspace(0.1, 12, s, device=DEV)[None, :, None]
    for causal in (False, True):
        ref = _ref(q, k, v, heads, causal)
        e, general = _err(_attend(q, k, v, heads, causal, False), ref), _err(_attend(q, k, v, heads, causal, True), ref)
        assert e <= general + 2.0 ** -24, (e, general)


@pytest.mark.parametrize("causal", [False, True])
def test_stream32_non_finite_values(hip, causal):
    """A NaN or infinity in one query, key or value gives what the general kernel gives wherever no
    other key of the row is involved, and leaves other heads and batch entries as they were."""
    torch.manual_seed(10)
    heads, dh, s = 2, 48, 150
    q, k, v = (torch.randn(6, s, heads * dh, device=DEV) for _ in range(3))
    clean = _attend(q, k, v, heads, causal, False)
    q[0, 5, 3] = float("nan")
    k[1, 7, 50] = float("nan")
    v[2, s - 1, 1] = float("inf")
    v[3, 0, 60] = -float("inf")
    q[4, 9, 50] = 3.4e38                            # an infinity as a bf16; scores overflow
    got, general = _attend(q, k, v, heads, causal, False), _attend(q, k, v, heads, causal, True)
    assert torch.isnan(got[0, 5, :dh]).all() and torch.equal(got[0, 6:], clean[0, 6:])
    assert torch.isnan(got[1, 7:, dh:]).all() and not torch.isnan(got[1, :, :dh]).any()
    for b, col in ((2, 1), (3, 60)):
        last = s - 1 if causal and b == 2 else 0     # rows that attend to the infinite value
        assert torch.isinf(got[b, last:, col]).all()
        assert torch.equal(torch.sign(got[b, last:, col]), torch.sign(general[b, last:, col]))
        rest = [c for c in range(heads * dh) if c != col]
        assert torch.isfinite(got[b][:, rest]).all()
        assert (got[b][:, rest] - clean[b][:, rest]).abs().max().item() <= 1e-5
    assert torch.equal(torch.isnan(got[4, 9]), torch.isnan(general[4, 9]))
    assert torch.equal(got[5], clean[5])


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("qv,kv", [(1.003e3, -3e38), (3.01e20, -3.01e20), (-2.0 ** 90, 2.0 ** 60)])
def test_stream32_scores_that_overflow(hip, qv, kv, causal):
    """Finite operands whose product overflows to -infinity: the key weighs nothing, as in fp32
    arithmetic, and the row's other keys share the weight."""
    torch.manual_seed(11)
    heads, dh, s = 2, 64, 200
    q = torch.full((2, s, heads * dh), qv, device=DEV)
    k = torch.randn(2, s, heads * dh, device=DEV) / abs(qv)
    v = torch.randn(2, s, heads * dh, device=DEV)
    k[:, 5::7] = kv
    ref = _ref(q, k, v, heads, causal)
    got, general = _attend(q, k, v, heads, causal, False), _attend(q, k, v, heads, causal, True)
    assert not torch.isnan(general).any() and not torch.isnan(got).any()
    assert _err(got, ref) <= _err(general, ref) + 2.0 ** -24


def test_stream32_values_that_overflow(hip):
    """Values whose unnormalised sum exceeds fp32: infinite, as in the general kernel.  (1.4965 x 2^127 rounds up
    as a bf16, and enough keys take the sum of those roundings to the other infinity.)"""
    heads, dh, s = 1, 32, 4000
    q, k = (torch.zeros(1, s, heads * dh, device=DEV) for _ in range(2))
    v = torch.full((1, s, heads * dh), 1.4965 * 2.0 ** 127, device=DEV)
    v[:, :, 1] *= -1.0
    v[:, :, 2] = 1.0
    got, general = _attend(q, k, v, heads, False, False), _attend(q, k, v, heads, False, True)
    assert torch.isinf(general[:, :, :2]).all()
    assert torch.equal(got[:, :, :2], general[:, :, :2])
    assert ((got[:, :, 2] - 1.0).abs() <= 2.0 ** -20).all()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("vs", [2.0 ** -112, 2.0 ** -120, 2.0 ** -126, 2.0 ** -138])
def test_stream32_small_values(hip, vs, causal):
    """Values below what three bf16 planes carry, in some columns of one head: those columns' outputs keep the
    general kernel's error, and 2^-148 for the steps of subnormal numbers."""
    torch.manual_seed(12)
    heads, dh, s = 2, 40, 150
    q, k, v = (torch.randn(2, s, heads * dh, device=DEV) for _ in range(3))
    v[0, :, 3:9] *= vs
    v[1, :, dh:] *= vs
    ref = _ref(q, k, v, heads, causal)
    got, general = (_attend(q, k, v, heads, causal, m).double() for m in (False, True))
    for cols in ((0, slice(3, 9)), (1, slice(dh, 2 * dh)), (0, slice(9, 2 * dh))):
        g, e, r = (t[cols[0], :, cols[1]] for t in (got, general, ref))
        slack = 2.0 ** -24 + 2.0 ** -148 * r.numel() ** 0.5 / r.norm().item()
        assert _err(g, r) <= _err(e, r) + slack, cols


@pytest.mark.parametrize("qs", [2.0 ** -115, 2.0 ** -122, 2.0 ** 100])
def test_stream32_queries_and_keys_far_apart(hip, qs):
    """Queries and keys of opposite scales, ordinary scores."""
    torch.manual_seed(13)
    heads, dh, s = 2, 64, 140
    q, k, v = (torch.randn(2, s, heads * dh, device=DEV) for _ in range(3))
    q, k = q * qs, k / qs
    ref = _ref(q, k, v, heads, False)
    e, general = _err(_attend(q, k, v, heads, False, False), ref), _err(_attend(q, k, v, heads, False, True), ref)
    assert e <= general + 2.0 ** -24, (e, general)
