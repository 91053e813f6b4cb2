"""The partitioned fp32 recurrence (GPU): LSTM and GRU at hidden sizes above 128 up to 384, against
fp64 modules per timestep and against the one-launch-per-step kernel (which a captured stream
takes), at the edges of its splits: row chunks of 16, more units than fit one launch, both widths
of workgroup.  Bar per timestep: 1e-5 normwise, the suite's fp32 bar (sums of at most 640 products
in fp32, through sigmoid / tanh of slope at most 1)."""

import pytest
import torch
import torch.nn as nn

from tests._util import TOL_F32, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _mods(kind, n, i, h, bias=True):
    cls = nn.LSTM if kind == "lstm" else nn.GRU
    return [cls(i, h, batch_first=True, bias=bias) for _ in range(n)]


def _wide(kind, mods):
    import wide_compiler as wc
    return (wc.WideLSTM if kind == "lstm" else wc.WideGRU).from_modules(mods).to(DEV)


def _ref(mods, x, states):
    with torch.no_grad():
        res = [m.double()(x[q].double(), None if states is None else
                          (tuple(s[q][None].double() for s in states) if len(states) == 2
                           else states[0][q][None].double())) for q, m in enumerate(mods)]
    for m in mods:
        m.float()
    outs = torch.stack([r[0] for r in res])
    fin = [torch.stack([(r[1][k] if isinstance(r[1], tuple) else r[1])[0] for r in res])
           for k in range(2 if isinstance(res[0][1], tuple) else 1)]
    return outs, fin


def _run(wide, x, states):
    from wide_compiler import _hip
    import ctypes
    a, _ = _hip.rnn_args(cell=_hip.CELL_LSTM if "LSTM" in type(wide).__name__ else _hip.CELL_GRU, x=x.to(DEV),
                         w_ih=wide.weight_ih, w_hh=wide.weight_hh, b_ih=None, b_hh=None, h0=None, c0=None,
                         out=torch.empty(*x.shape[:3], wide.hidden_size, device=DEV), h_n=None, c_n=None,
                         allocate=False)
    assert _hip.lib().wc_rnn_status_offset(ctypes.byref(a)) >= 0      # the partitioned kernel runs
    with torch.no_grad():
        if states is None:
            out, fin = wide(x.to(DEV))
        else:
            s = tuple(t.to(DEV) for t in states)
            out, fin = wide(x.to(DEV), s if len(s) == 2 else s[0])
    return out, list(fin) if isinstance(fin, tuple) else [fin]


@pytest.mark.parametrize("kind", ["lstm", "gru"])
@pytest.mark.parametrize("n,b,t,i,h,given", [
    (1, 1, 12, 8, 160, False), (2, 3, 16, 16, 192, True), (3, 16, 20, 32, 256, True), (2, 17, 13, 24, 256, False),
    (16, 16, 12, 64, 256, False), (33, 5, 24, 20, 256, True), (3, 33, 16, 12, 224, True), (2, 20, 12, 40, 320, True),
    (12, 4, 30, 8, 384, False), (20, 2, 40, 8, 384, True), (40, 2, 40, 8, 288, True)])
def test_part32_against_fp64(hip, kind, n, b, t, i, h, given):
    torch.manual_seed(n + b + h)
    mods = _mods(kind, n, i, h, bias=given or n > 2)
    wide = _wide(kind, mods)
    x = torch.randn(n, b, t, i)
    states = None
    if given:
        states = [torch.randn(n, b, h) * 1.5 for _ in range(2 if kind == "lstm" else 1)]
    out, fin = _run(wide, x, states)
    hip.rnn_sync_check(block=True)
    ref, rfin = _ref(mods, x, states)
    for s in range(t):
        assert rel_err(out[:, :, s], ref[:, :, s]) <= TOL_F32, s
    for a, r in zip(fin, rfin):
        assert rel_err(a, r) <= TOL_F32


@pytest.mark.parametrize("kind", ["lstm", "gru"])
def test_part32_equals_streamed_kernel_under_capture(hip, kind):
    """A captured forward takes the one-launch-per-step kernel: replays agree with it to the fp32 bar
    and with each other bit for bit, between eager (partitioned) forwards, themselves repeatable."""
    torch.manual_seed(5)
    n, b, t, i, h = 4, 18, 14, 32, 256
    wide = _wide(kind, _mods(kind, n, i, h))
    x = torch.randn(n, b, t, i, device=DEV)
    with torch.no_grad():
        first = wide(x)[0].clone()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            held = wide(x)[0]
        replays = []
        for _ in range(3):
            graph.replay()
            replays.append(held.clone())
            again = wide(x)[0]
            torch.cuda.synchronize()
            assert torch.equal(again, first)
    hip.rnn_sync_check(block=True)
    assert torch.equal(replays[0], replays[1]) and torch.equal(replays[0], replays[2])
    assert rel_err(replays[0], first) <= TOL_F32


def test_part32_recurrence_repeats_and_noalloc(hip):
    """The recurrence launched again on the same gates, and through the static scratch: bit-identical."""
    torch.manual_seed(6)
    n, b, t, i, h = 20, 16, 20, 16, 256
    wide = _wide("lstm", _mods("lstm", n, i, h))
    x = torch.randn(n, b, t, i, device=DEV)
    w = dict(cell=hip.CELL_LSTM, x=x, w_ih=wide.weight_ih.detach(), w_hh=wide.weight_hh.detach(),
             b_ih=wide.bias_ih.detach(), b_hh=wide.bias_hh.detach(), h0=None, c0=None, h_n=None, c_n=None)
    with torch.no_grad():
        ref = wide(x)[0].clone()
    out = torch.empty_like(ref)
    a, ws = hip.rnn_args(out=out, status=hip.rnn_status_word(x.device), **w)
    hip.rnn_phase(a, "input_projection", x)
    for _ in range(4):
        out.fill_(float("nan"))
        hip.rnn_phase(a, "recurrence", x)
        hip.rnn_sync_check(block=True)
        assert torch.equal(out, ref)
    out.fill_(float("nan"))
    hip.rnn_forward_noalloc(out=out, **w)
    hip.rnn_sync_check(block=True)
    assert torch.equal(out, ref)


def test_part32_give_up_is_raised(hip):
    torch.manual_seed(7)
    wide = _wide("gru", _mods("gru", 3, 8, 256))
    x = torch.randn(3, 4, 16, 8, device=DEV)
    with torch.no_grad():
        ref = wide(x)[0].clone()
        hip.rnn_sync_check(block=True)
        hip.rnn_set_spin_limit(0)
        try:
            wide(x)
            with pytest.raises(hip.WideKernelError, match="gave up"):
                hip.rnn_sync_check(block=True)
        finally:
            hip.rnn_set_spin_limit(-1)
        again = wide(x)[0]
    hip.rnn_sync_check(block=True)
    assert torch.equal(again, ref)


@pytest.mark.parametrize("kind", ["lstm", "gru"])
def test_part32_infinite_weights_and_states(hip, kind):
    """An infinite weight saturates its gate and an infinite or NaN h0 stays in its own row, as in fp32."""
    torch.manual_seed(8)
    n, b, t, i, h = 3, 5, 12, 8, 256
    mods = _mods(kind, n, i, h)
    with torch.no_grad():
        mods[0].weight_hh_l0[3, 200] = float("inf")            # first gate of unit 3
        mods[1].weight_hh_l0[h + 70, 5] = -float("inf")        # second gate of unit 70
    states = [torch.randn(n, b, h) * 0.5 for _ in range(2 if kind == "lstm" else 1)]
    states[0][2, 1, 9] = float("nan")
    wide = _wide(kind, mods)
    x = torch.randn(n, b, t, i)
    out, _ = _run(wide, x, states)
    hip.rnn_sync_check(block=True)
    ref, _ = _ref(mods, x, states)
    assert torch.equal(torch.isnan(out.cpu()), torch.isnan(ref))
    keep = ~torch.isnan(ref)
    assert (out.cpu().double()[keep] - ref[keep]).abs().max().item() <= 1e-5


@pytest.mark.parametrize("kind", ["lstm", "gru"])
@pytest.mark.parametrize("hv,wv", [(3.01e20, 3.01e20), (1.003e3, 3e38), (2.0 ** 90, 2.0 ** 60)])
def test_part32_gate_sums_that_overflow(hip, kind, hv, wv):
    """A finite h0 and finite weights whose gate sums overflow saturate the gate, as in fp32: the LSTM's first gate
    of every fourth unit (0) and its third (-1), and the GRU's update gate of every unit (h_1 = n)."""
    torch.manual_seed(9)
    n, b, t, i, h = 2, 3, 12, 8, 256
    mods = _mods(kind, n, i, h)
    with torch.no_grad():
        for m in mods:
            m.weight_hh_l0 /= hv
            if kind == "lstm":
                m.weight_hh_l0[0:h:4] = -wv
                m.weight_hh_l0[2 * h:3 * h:3] = -wv
            else:
                m.weight_hh_l0[h:2 * h] = -wv
    states = [torch.randn(n, b, h) * 0.5 for _ in range(2 if kind == "lstm" else 1)]
    states[0][:] = hv
    wide = _wide(kind, mods)
    x = torch.randn(n, b, t, i)
    out, _ = _run(wide, x, states)
    hip.rnn_sync_check(block=True)
    ref, _ = _ref(mods, x, states)
    assert not torch.isnan(out).any()
    assert rel_err(out[:, :, 0], ref[:, :, 0]) <= TOL_F32


@pytest.mark.parametrize("kind", ["lstm", "gru"])
def test_part32_states_and_weights_far_apart(hip, kind):
    """Subnormal-range states on weights near the top of the range: gates of order one keep the fp32 bar."""
    torch.manual_seed(10)
    n, b, t, i, h = 2, 3, 12, 8, 256
    mods = _mods(kind, n, i, h)
    with torch.no_grad():
        for m in mods:
            m.weight_hh_l0[:, 17] = torch.randn(m.weight_hh_l0.shape[0]) * 2.0 ** 122
    states = [torch.randn(n, b, h) * 0.5 for _ in range(2 if kind == "lstm" else 1)]
    states[0][:, :, 17] = torch.randn(n, b) * 2.0 ** -122
    wide = _wide(kind, mods)
    x = torch.randn(n, b, t, i)
    out, _ = _run(wide, x, states)
    hip.rnn_sync_check(block=True)
    ref, _ = _ref(mods, x, states)
    assert rel_err(out[:, :, 0], ref[:, :, 0]) <= TOL_F32


@pytest.mark.parametrize("kind", ["lstm", "gru"])
def test_part32_status_word_after_replays(hip, kind):
    """Without a status word of the caller's the workspace's own one reads 0 after a clean forward, also a
    captured one, which runs another kernel and finds the workspace in any state."""
    import ctypes
    torch.manual_seed(11)
    n, b, t, i, h = 4, 18, 14, 32, 256
    wide = _wide(kind, _mods(kind, n, i, h))
    x = torch.randn(n, b, t, i, device=DEV)
    out = torch.empty(n, b, t, h, device=DEV)
    a, ws = hip.rnn_args(cell=hip.CELL_LSTM if kind == "lstm" else hip.CELL_GRU, x=x, w_ih=wide.weight_ih.detach(),
                         w_hh=wide.weight_hh.detach(), b_ih=wide.bias_ih.detach(), b_hh=wide.bias_hh.detach(),
                         h0=None, c0=None, out=out, h_n=None, c_n=None)
    at = hip.lib().wc_rnn_status_offset(ctypes.byref(a))
    assert 0 <= at <= ws.numel() - 4
    word = ws[at:at + 4].view(torch.int32)

    def both():
        hip.rnn_phase(a, "input_projection", x)
        hip.rnn_phase(a, "recurrence", x)

    ws.fill_(255)
    both()
    torch.cuda.synchronize()
    assert word.item() == 0
    with torch.no_grad():
        ref = wide(x)[0]
    assert rel_err(out, ref) <= TOL_F32
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        both()
    for _ in range(3):
        ws.fill_(255)
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert word.item() == 0
        assert rel_err(out, ref) <= TOL_F32
