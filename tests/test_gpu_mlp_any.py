"""wc_mlp2_any (two chained Linear layers of any widths in one launch) through traced models,
against the same forward in fp64, at the edges of its tiles; and the rule that picks it."""

import pytest
import torch
import torch.nn as nn

from wide_compiler import _hip

DEV = "cuda"
# fp32: at most 512 products a layer, |error| of a sum about sqrt(k) roundings of 2^-24 of its size,
# two layers: 512^0.5 * 2^-24 * 2 = 2.7e-6 of the result's 2-norm at most.  16 bits: inputs are
# exact, h and y round once each (2^-9 and 2^-12 relative), 2-norm below one full rounding each.
REL = {torch.float32: 2.7e-6, torch.bfloat16: 2 * 2.0 ** -9, torch.float16: 2 * 2.0 ** -12}


class _Chain(nn.Module):
    def __init__(self, i, h, o, relu1, relu2, bias):
        super().__init__()
        self.fc1, self.fc2 = nn.Linear(i, h, bias=bias), nn.Linear(h, o, bias=bias)
        self.relu1, self.relu2 = relu1, relu2

    def forward(self, x):
        h = self.fc1(x)
        y = self.fc2(torch.relu(h) if self.relu1 else h)
        return torch.relu(y) if self.relu2 else y


def _run(dtype, n, b, i, h, o, relu1=True, relu2=False, bias=True):
    import wide_compiler as wc
    torch.manual_seed(n * 1000 + b + i + h + o)
    models = [_Chain(i, h, o, relu1, relu2, bias).to(DEV).to(dtype) for _ in range(n)]
    x = torch.randn(b, n * i, device=DEV).to(dtype)
    wide = wc.compile(models, x[:, :i].contiguous()).eval()
    with torch.no_grad():
        y = wide(x)
        y2 = wide(x)                                          # the kept launch arguments
    xd = x.double().view(b, n, i)
    want = []
    with torch.no_grad():
        for k, m in enumerate(models):
            w = [t.detach().double() for t in (m.fc1.weight, m.fc2.weight)]
            bb = [m.fc1.bias.double(), m.fc2.bias.double()] if bias else [0.0, 0.0]
            t = (xd[:, k, None, :] * w[0]).sum(-1) + bb[0]
            t = torch.relu(t) if relu1 else t
            t = (t[:, None, :] * w[1]).sum(-1) + bb[1]
            want.append(torch.relu(t) if relu2 else t)
    want = torch.cat(want, 1)
    assert torch.equal(y, y2)
    rel = ((y.double() - want).norm() / want.norm()).item()
    assert rel <= REL[dtype], rel
    return wide


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,b,i,h,o", [
    (4, 1, 16, 16, 16),           # one row, one tile a layer
    (3, 17, 33, 31, 19),          # odd rows, widths and alignments
    (5, 16, 128, 129, 384),       # one column past a tile; the last wave's second and third tiles
    (2, 5, 257, 500, 511),        # k past a block of 128 and 256, seven eighths of a k-step left over
    (9, 250, 128, 19, 74),        # many row blocks
    (1, 3, 7, 9, 3),              # weights smaller than a k-step: units moved back to the tensor's end
    (2, 20, 130, 3, 5),           # one k value pair past a block, two-column tiles
    (128, 80, 40, 72, 24),        # 32-row workgroups, the last half empty
])
def test_any_widths(monkeypatch, dtype, n, b, i, h, o):
    monkeypatch.setattr(_hip, "mlp2_entry", lambda *a: "wc_mlp2_any")     # also where two GEMMs are faster
    wide = _run(dtype, n, b, i, h, o)
    assert "one two-layer launch" in wide.summary()


@pytest.mark.gpu
@pytest.mark.parametrize("relu1,relu2,bias", [(False, False, True), (True, True, True), (False, True, False)])
def test_any_activations(relu1, relu2, bias):
    _run(torch.float32, 6, 21, 50, 70, 30, relu1, relu2, bias)


@pytest.mark.gpu
def test_rows_beyond_the_rule_run_two_gemms():
    """The chain is fused for few rows; a later call with many rows takes the two GEMMs."""
    assert _hip.mlp2_entry(torch.float32, 16, 4096, 200, 500, 300) is None
    assert _hip.mlp2_entry(torch.float32, 16, 4, 100, 200, 60) == "wc_mlp2_any"
    _run(torch.float32, 16, 4096, 200, 500, 300)
    _run(torch.float32, 16, 1024, 100, 200, 60)


@pytest.mark.gpu
def test_any_infinities_stay_in_their_row_and_column():
    import wide_compiler as wc
    torch.manual_seed(7)
    models = [_Chain(20, 40, 12, False, False, True).to(DEV) for _ in range(3)]
    x = torch.randn(5, 60, device=DEV)
    x[2, 25] = float("inf")
    x[4, 3] = float("nan")
    wide = wc.compile(models, x[:, :20].contiguous()).eval()
    with torch.no_grad():
        y = wide(x)
        want = torch.cat([m.double()(x.double()[:, 20 * k:20 * k + 20]) for k, m in enumerate(models)], 1)
    assert torch.equal(torch.isfinite(y), torch.isfinite(want))


def test_rule():
    e = _hip.mlp2_entry
    assert e(torch.float32, 100, 32, 64, 128, 64) == "wc_mlp2"
    assert e(torch.float16, 100, 32, 64, 128, 64) == "wc_mlp2_any"
    assert e(torch.float32, 8, 4, 176, 48, 16) == "wc_mlp2_any"
    assert e(torch.float32, 1, 1, 2000, 2000, 8) is None          # 16 rows of x and h exceed LDS
    assert e(torch.float32, 1, 1, 4097, 8, 8) is None
    assert e(torch.float32, 1, 1, 3, 2, 8) is None                # fewer than 8 weights
    assert e(torch.float32, 128, 16, 256, 256, 250) == "wc_mlp2_any"
    assert e(torch.float32, 32, 64, 256, 512, 250) is None
    assert e(torch.float64, 1, 1, 16, 16, 16) is None
    assert e(torch.float32, 0, 1, 20, 16, 16) is None
