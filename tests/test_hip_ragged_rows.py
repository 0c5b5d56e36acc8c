"""Rows that the vector width does not divide (``whole_group`` of ``csrc/sjhip_common.h``): the last work-item of a row
takes the row's last V neurons, some of which its neighbour has too.  The same neurons inside rows padded to a whole number
of vectors are the reference: every output must have the same bits, and a neuron held twice must count once in dL/dk."""

import pytest
import torch

from spikingjelly_amd import configure
from spikingjelly_amd.activation_based import neuron, surrogate

pytestmark = pytest.mark.gpu

MODES = [(torch.float32, "torch"), (torch.float16, "torch"), (torch.bfloat16, "torch"), (torch.float16, "fp32_state"),
         (torch.bfloat16, "fp32_state")]


def _node(kind, v_seq):
    kw = dict(surrogate_function=surrogate.ATan(2.0), step_mode="m", backend="hip", store_v_seq=v_seq)
    if kind == "if":
        return neuron.IFNode(v_reset=None, **kw).cuda()
    if kind == "plif":
        return neuron.ParametricLIFNode(init_tau=2.0, v_reset=None, **kw).cuda()
    return neuron.LIFNode(tau=3.0, **kw).cuda()


def _run(kind, x, gs, gv):
    node = _node(kind, gv is not None)
    x = x.clone().requires_grad_()
    s = node(x)
    if gv is None:
        s.backward(gs)
    else:
        torch.autograd.backward([s, node.v_seq], [gs, gv])
    return (s.detach(), node.v.detach(), None if gv is None else node.v_seq.detach(), x.grad,
            node.w.grad if kind == "plif" else None)


# (one vector, one neuron more, one less than two; the last work-item at the edges of a wavefront and of blocks of 64,
# 128 and 256; T on both sides of the short-sequence kernels' limit and in pieces)
@pytest.mark.parametrize("T", [8, 9, 45])
@pytest.mark.parametrize("N", [8, 9, 15, 257, 1025, 4099])
@pytest.mark.parametrize("dtype,mode", MODES)
@pytest.mark.parametrize("kind", ["lif", "plif", "if"])
def test_ragged_rows_equal_padded_rows(kind, dtype, mode, N, T, monkeypatch):
    monkeypatch.setattr(configure, "hip_half_precision_mode", mode)
    g = torch.Generator().manual_seed(N * 100 + T)
    pad = (N + 7) // 8 * 8
    x = torch.zeros(T, pad)
    gs, gv = torch.zeros(T, pad), torch.zeros(T, pad)
    x[:, :N] = torch.randn(T, N, generator=g) * 0.8 + 0.4
    gs[:, :N] = torch.randn(T, N, generator=g)
    gv[:, :N] = torch.randn(T, N, generator=g) * 0.1
    x, gs, gv = (t.to(dtype).cuda() for t in (x, gs, gv))
    cut = lambda t: t[..., :N].contiguous()
    gv = gv if N % 2 else None
    # 16-bit storage with fp32 state: a saved h_seq is rounded, a replayed one is not; ragged rows keep the saved route
    with monkeypatch.context() as m:
        m.setattr(configure, "hip_backward_recompute", mode != "fp32_state" or N % 8 == 0)
        want = _run(kind, x, gs, gv)
    got = _run(kind, cut(x), cut(gs), None if gv is None else cut(gv))
    for name, a, b in zip(("spikes", "v", "v_seq", "grad_x"), got[:4], want[:4]):
        if b is not None:
            assert torch.equal(a, b[..., :N]), (name, N, T)
    if kind == "plif":
        # fp32 sums of T N terms below 2 (|G| < 2, |h - v| < 2 for these inputs, times dk/dw = 1/4 and 1/k = 2), at most T + 60
        # additions behind each other; the padding adds zeros
        assert abs(float(got[4]) - float(want[4])) <= (T + 60) * 2.0 ** -24 * 2.0 * T * N, (float(got[4]), float(want[4]))


@pytest.mark.parametrize("T", [8, 45])
@pytest.mark.parametrize("N", [9, 15, 1025, 1027, 4099])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("saved_h", [False, True])
def test_a_neuron_held_twice_counts_once_in_the_time_constant(dtype, N, T, saved_h, monkeypatch):
    """Only the last vector of a row has an upstream gradient: dL/dk is then a sum of few terms, most of them of the neurons that
    two work-items hold."""
    monkeypatch.setattr(configure, "hip_backward_recompute", not saved_h)
    g = torch.Generator().manual_seed(N * 100 + T)
    pad, V = (N + 7) // 8 * 8, 16 // dtype.itemsize
    x, gs = torch.zeros(T, pad), torch.zeros(T, pad)
    x[:, :N] = torch.randn(T, N, generator=g) * 0.8 + 0.4
    gs[:, N - V:N] = torch.rand(T, V, generator=g) + 0.5
    x, gs = x.to(dtype).cuda(), gs.to(dtype).cuda()
    got = float(_run("plif", x[:, :N].contiguous(), gs[:, :N].contiguous(), None)[4])
    want = float(_run("plif", x, gs, None)[4])
    # (fp32 sums of T V terms below 8: the carried gradient reaches 1.5 / (1 - 1/2) and more through the reset, times |h - v| < 2)
    assert abs(got - want) <= (T + 60) * 2.0 ** -24 * 8.0 * T * V, (got, want)
    assert abs(want) > 0.05  # a shared neuron counted twice would show


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("offset", [1, 3])
def test_rows_that_begin_off_the_vector_alignment(dtype, offset):
    """The forward of a view into a longer buffer, with one element's alignment only."""
    T, N = 5, 1031
    buf = (torch.randn(T * N + offset, generator=torch.Generator().manual_seed(3)) * 0.8 + 0.4).to(dtype).cuda()
    x = buf[offset:].view(T, N)
    assert x.data_ptr() % 16 != 0
    with torch.no_grad():
        got, want = _node("lif", True), _node("lif", True)
        assert torch.equal(got(x), want(x.clone())) and torch.equal(got.v_seq, want.v_seq) and torch.equal(got.v, want.v)


def test_short_rows_keep_the_saved_route():
    """Fewer neurons than one vector: nothing to overlap with, the element-wise kernels and the saved h run."""
    for N in (1, 3, 7):
        x = torch.randn(6, N, generator=torch.Generator().manual_seed(N)).half().cuda()
        gs = torch.ones_like(x)
        pad = torch.zeros(6, 8, dtype=torch.float16, device="cuda")
        xp, gp = pad.clone(), pad.clone()
        xp[:, :N], gp[:, :N] = x, gs
        got, want = _run("lif", x, gs, None), _run("lif", xp, gp, None)
        assert all(torch.equal(got[i], want[i][..., :N]) for i in (0, 1, 3))
