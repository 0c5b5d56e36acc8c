"""C ABI calls whose outputs lie in the place of their inputs.  Rows that the vector width does not divide would have two
work-items share neurons (``whole_group`` of ``csrc/sjhip_common.h``): such calls run the element-wise kernels or are refused."""

import ctypes

import pytest
import torch

from spikingjelly_amd.activation_based.hip_kernel import library as L


def _params(flags=0, sg=1):
    return L.NeuronParams(2.0, 1.0, 0.0, 2.0, sg, flags, 0.0, 0.0, 0.0, 4.0, 0.0, 4.0)


X, V, GS, GX, GV, CK = (0x1000000 * i for i in range(1, 7))


@pytest.mark.parametrize("N", [5, 9, 1027])
def test_replaying_backward_refuses_shared_memory_in_ragged_rows(N):
    lib, p, T = L.load(), _params(1), 20
    for gx, gv0, grads in ((GS, None, (GS, None, None)), (GX, GV, (GS, None, GV)), (X, None, (GS, None, None)),
                           (GS + 4 * (T * N - 1) // 16 * 16, None, (GS, None, None)), (GX, V, (GS, None, None))):
        rc = lib.sjhip_neuron_backward_recompute(L.NEURON_LIF, L.DTYPE_F32, ctypes.byref(p), T, N, X, V, None, *grads, gx, gv0, None, None, None)
        assert rc == -2 and b"overlap" in lib.sjhip_last_error(), (gx, gv0)
        rc = lib.sjhip_neuron_backward_recompute_pieces(L.NEURON_LIF, L.DTYPE_F32, ctypes.byref(p), T, N, 16, X, V, None, CK, *grads, gx, gv0,
                                                        None, None, None)
        assert rc == -2 and b"overlap" in lib.sjhip_last_error(), (gx, gv0)


@pytest.mark.parametrize("N", [5, 9, 1027])
def test_forward_in_pieces_refuses_shared_memory_in_ragged_rows(N):
    lib, p, T = L.load(), _params(1), 20
    for s, v_seq, v_last in ((X, None, GV), (GS, X, GV), (GS, None, V)):
        rc = lib.sjhip_neuron_forward_pieces(L.NEURON_LIF, L.DTYPE_F32, ctypes.byref(p), T, N, 16, X, V, None, s, v_seq, v_last, CK, None)
        assert rc == -2 and b"overlap" in lib.sjhip_last_error(), (s, v_seq, v_last)


@pytest.mark.parametrize("T", [4, 20])
def test_batch_norm_backward_refuses_shared_memory_in_ragged_rows(T):
    lib, p = L.load(), _params(1)
    for g, gv0, gl in ((GS, None, None), (X, None, None), (GX, V, None), (GX, GV, GV)):
        rc = lib.sjhip_bn_lif_backward(L.NEURON_LIF, ctypes.byref(p), T, 2, 4, 9, X, CK, CK, V, GS, gl, g, gv0, CK, None)
        assert rc == -2 and b"overlap" in lib.sjhip_last_error(), (g, gv0)


@pytest.mark.gpu
@pytest.mark.parametrize("T", [4, 20])
def test_batch_norm_backward_of_whole_rows_in_place(T):
    lib, p, B, C, Lp = L.load(), ctypes.byref(_params(1)), 2, 4, 12
    g = torch.Generator().manual_seed(T)
    y, gs = (torch.randn(T, B, C, Lp, generator=g).cuda() for _ in range(2))
    one, zero, v0 = torch.ones(C).cuda(), torch.zeros(C).cuda(), torch.zeros(B, C, Lp).cuda()
    sums, sums2, dz = torch.empty(B * C, 2).cuda(), torch.empty(B * C, 2).cuda(), torch.empty_like(y)
    st, ptr = L.current_stream_ptr(y.device), lambda t: t.data_ptr()
    call = lambda grad, out, part: lib.sjhip_bn_lif_backward(L.NEURON_LIF, p, T, B, C, Lp, ptr(y), ptr(one), ptr(zero), ptr(v0), ptr(grad), None,
                                                             ptr(out), None, ptr(part), st)
    assert call(gs, dz, sums) == 0 and call(gs, gs, sums2) == 0
    assert torch.equal(dz, gs) and torch.equal(sums, sums2)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("N", [3, 8, 9, 1027, 262147])
def test_in_place_calls_equal_calls_with_buffers_of_their_own(N, dtype):
    lib, T, d = L.load(), 9, L.dtype_id(dtype)
    g = torch.Generator().manual_seed(N)
    x, gs = ((torch.randn(T, N, generator=g) + 0.4).to(dtype).cuda() for _ in range(2))
    v0, gl = ((torch.randn(N, generator=g) * 0.2).to(dtype).cuda() for _ in range(2))
    p, st = ctypes.byref(_params(1)), L.current_stream_ptr(x.device)
    s, h, v1 = torch.empty_like(x), torch.empty_like(x), torch.empty_like(v0)
    ptr = lambda t: t.data_ptr()
    assert lib.sjhip_neuron_forward(L.NEURON_LIF, d, p, T, N, ptr(x), ptr(v0), None, ptr(s), None, ptr(v1), ptr(h), st) == 0
    for share in ("x", "v", "both"):
        x2, v2 = x.clone(), v0.clone()
        s2, v3, h2 = x2 if share != "v" else torch.empty_like(x), v2 if share != "x" else torch.empty_like(v0), torch.empty_like(x)
        assert lib.sjhip_neuron_forward(L.NEURON_LIF, d, p, T, N, ptr(x2), ptr(v2), None, ptr(s2), None, ptr(v3), ptr(h2), st) == 0
        assert torch.equal(s2, s) and torch.equal(v3, v1) and torch.equal(h2, h), share
    gx, gv = torch.empty_like(x), torch.empty_like(v0)
    assert lib.sjhip_neuron_backward(L.NEURON_LIF, d, p, T, N, ptr(gs), None, ptr(gl), ptr(h), None, None, ptr(gx), ptr(gv), None, None, st) == 0
    for share in ("gs", "h", "gl"):
        gs2, h2, gl2 = gs.clone(), h.clone(), gl.clone()
        gx2 = gs2 if share == "gs" else (h2 if share == "h" else torch.empty_like(x))
        gv2 = gl2 if share == "gl" else torch.empty_like(v0)
        assert lib.sjhip_neuron_backward(L.NEURON_LIF, d, p, T, N, ptr(gs2), None, ptr(gl2), ptr(h2), None, None, ptr(gx2), ptr(gv2), None, None,
                                         st) == 0
        assert torch.equal(gx2, gx) and torch.equal(gv2, gv), share
