"""Convolution, batch norm and neuron over samples whose number of positions four does not divide.

Every kernel is compared with itself on the same rows padded with zeros to a multiple of four (the layout the other tests
pin against the oracle): element-wise results, sums in the same order and exact sums have the same bits, sums in another
order the rounding of fp32 sums of their length."""

import pytest
import torch

from helpers import seeded_randn
from oracle import neuron_oracle as no

pytestmark = pytest.mark.gpu

LENGTHS = [4, 5, 6, 7, 9, 31, 33, 49, 81, 127, 129, 198, 257, 259, 1025]


@pytest.fixture(scope="module")
def C():
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif

    return conv_bn_lif


def _padded(x):
    return torch.nn.functional.pad(x, (0, -x.shape[-1] % 4)).contiguous()


def _spec(T):
    from spikingjelly_amd.activation_based.hip_kernel import neuron_kernel as K

    return (2.0, 1.0, 0.0, K._flags(False, False, True, 0), no.SG_IDS["atan"], no.SG_DEFAULT_ALPHA["atan"])


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("S, M, K", [(1, 5, 3), (5, 130, 70), (2, 256, 96)])
@pytest.mark.parametrize("spikes", [False, True])
def test_gemms(C, L, S, M, K, spikes):
    F = C.F16 | 2
    terms = C.F16 | 1 if spikes else F
    x = (seeded_randn((S, K, L), 1) > 0.3).float().cuda() if spikes else seeded_randn((S, K, L), 1).cuda()
    dy, w = seeded_randn((S, M, L), 2).cuda(), seeded_randn((M, K), 3).cuda()
    xp, dyp = _padded(x), _padded(dy)
    planes = C.split_weight(w, False, F)
    got, sums = C.pw_gemm(planes, F, M, K, x, terms, True)
    want, want_sums = C.pw_gemm(planes, F, M, K, xp, terms, True)
    assert torch.equal(C.pw_grad_weight(dy, F, x, terms), C.pw_grad_weight(dyp, F, xp, terms))
    # (against 64 bits: what the split drops, 2^-22, and 2^-24 per fp32 addition of K terms)
    exact = w.double() @ x.double()
    bound = (2.0 ** -22 + K * 2.0 ** -24) * (w.double().abs() @ x.double().abs())
    for c in (got, want[..., :L]):
        assert ((c.double() - exact).abs() <= bound).all()
    # The rows of other lengths add their K steps in another order than rows of a multiple of four: the same bits where
    # every sum is exact (integers, sums below 2^24)
    xi, wi = (x * 4.0).round().clamp(-8, 8), (w * 4.0).round().clamp(-8, 8)
    planes = C.split_weight(wi, False, F)
    got_i, sums_i = C.pw_gemm(planes, F, M, K, xi, terms, True)
    want_i, want_sums_i = C.pw_gemm(planes, F, M, K, _padded(xi), terms, True)
    assert torch.equal(got_i, want_i[..., :L]) and torch.equal(got_i.double(), wi.double() @ xi.double())
    assert torch.equal(sums_i[..., 0], want_sums_i[..., 0])
    # (sums and sums of squares of 64 columns, 2^-24 per addition; squares with the product's own rounding; on 2^-22 + K 2^-24
    # of the terms from either order of the sums inside a column)
    for i, power in ((0, 1), (1, 2)):
        a, b = sums[..., i].double().sum(0), want_sums[..., i].double().sum(0)
        scale = (w.double().abs() @ x.double().abs()).pow(power).sum((0, 2))
        assert ((a - b).abs() <= power * 2 * (2.0 ** -22 + K * 2.0 ** -24 + 64 * 2.0 ** -24) * scale).all()


# Relative 2-norm errors against 64 bits, in 1e-7, of torch's fp32 convolution (y, dx, dw) on the inputs of the test below: the smallest of
# four processes, which differ in the last digits of dw only.
LIBRARY_ERRORS = {
    (6, 8, 512, 128): {False: (2.065, 2.033, 2.321), True: (1.149, 2.033, 2.264)},
    (4, 1, 512, 1536): {False: (2.880, 3.540, 1.333), True: (1.478, 3.540, 0.8018)},
    (4, 16, 256, 256): {False: (1.498, 2.049, 2.065), True: (0.8767, 2.049, 1.901)},
    (2, 32, 512, 96): {False: (2.068, 1.760, 1.939), True: (1.144, 1.760, 1.477)},
}


@pytest.mark.parametrize("T, B, Cin, Cout", LIBRARY_ERRORS)
@pytest.mark.parametrize("spikes", [False, True])
def test_no_further_from_64_bits_than_the_library(C, T, B, Cin, Cout, spikes):
    """Position counts that four does not divide ran on the library's fp32 convolution before they ran on the fp16 split: the
    split's sums (the K steps of a column, and the sample groups of a weight gradient in 64 bits) are no further from 64 bits.
    The kernels add in a fixed order, so the errors are the same on every run: 0.35 to 0.92 of the library's (with one chain over
    all of K and fp32 sums over the groups up to 1.34)."""
    F, S, L = C.F16 | 2, T * B, 49
    x = (seeded_randn((S, Cin, L), 30) > 0.7).float().cuda() if spikes else seeded_randn((S, Cin, L), 30).cuda()
    w, dy = (seeded_randn((Cout, Cin), 31) * Cin ** -0.5).cuda(), seeded_randn((S, Cout, L), 32).cuda()
    terms = C.F16 | 1 if spikes else F
    split = (C.pw_gemm(C.split_weight(w, False, F), F, Cout, Cin, x, terms), C.pw_gemm(C.split_weight(w, True, F), F, Cin, Cout, dy, F),
             C.pw_grad_weight(dy, F, x, terms))
    x64, w64, dy64 = x.double(), w.double(), dy.double()
    exact = (w64 @ x64, w64.t().contiguous() @ dy64,
             dy64.transpose(0, 1).reshape(Cout, -1) @ x64.transpose(0, 1).reshape(Cin, -1).t().contiguous())
    for name, a, r, library in zip(("y", "dx", "dw"), split, exact, LIBRARY_ERRORS[T, B, Cin, Cout][spikes]):
        assert float((a.double() - r).norm() / r.norm()) <= library * 1e-7, name


@pytest.mark.parametrize("L", LENGTHS)
@pytest.mark.parametrize("T", [1, 4, 9, 35])
def test_normalise_and_neuron(C, L, T):
    B, Ch = 3, 8
    y = seeded_randn((T, B, Ch, L), 4, 0.4, 1.2).cuda()
    gs = seeded_randn((T, B, Ch, L), 5).cuda()
    gamma = seeded_randn((Ch,), 6, 1.0, 0.2).cuda()
    stats = C._bn_map(y.flatten(0, 1), gamma, None, None, None, True, 0.1, 1e-5)
    y64 = y.double().transpose(0, 2).reshape(Ch, -1)
    torch.testing.assert_close(stats[2].double(), y64.mean(1), rtol=1e-5, atol=1e-6)
    torch.testing.assert_close(stats[3].double(), (y64.var(1, unbiased=False) + 1e-5).rsqrt(), rtol=1e-5, atol=0)
    v0 = seeded_randn((B, Ch, L), 7, 0.0, 0.3).cuda()
    spec = _spec(T)
    yp, gp, vp = _padded(y), _padded(gs), _padded(v0)
    spikes, v = C._bn_lif_forward(y, stats, v0, spec, False)
    want, want_v = C._bn_lif_forward(yp, stats, vp, spec, False)
    assert torch.equal(spikes, want[..., :L]) and torch.equal(v, want_v[..., :L])
    bits, _ = C._bn_lif_forward(y, stats, v0, spec, True) if B * Ch * L % 8 == 0 else (None, None)
    if bits is not None:
        unpacked = (bits[:, None] >> torch.arange(8, device="cuda", dtype=torch.uint8)) & 1
        assert torch.equal(unpacked.flatten().float(), spikes.flatten())
    for batch_stats in (False, True):
        dy, dgamma, dbeta, gvi, dy_amax = C._bn_lif_backward(y, stats, gamma, v0, spec, batch_stats, gs, None, True, True)
        pdy, pdgamma, pdbeta, pgvi, _ = C._bn_lif_backward(yp, stats, gamma, vp, spec, False, gp, None, True, True)
        assert torch.equal(gvi, pgvi[..., :L])
        torch.testing.assert_close(dgamma, pdgamma, rtol=1e-5, atol=1e-4)  # sums of up to T B L = 1e5 terms of order one, in another order
        torch.testing.assert_close(dbeta, pdbeta, rtol=1e-5, atol=1e-4)
        assert torch.equal(C.sample_amax(dy_amax), dy.abs().amax(dim=(2, 3)).flatten())
        if not batch_stats:
            assert torch.equal(dy, pdy[..., :L])
        else:   # dy = a (g - mean(g) - yhat mean(g yhat)), a g being the gradient without batch statistics
            yhat = (y - stats[2].view(-1, 1)) * stats[3].view(-1, 1)
            n, a = T * B * L, (gamma * stats[3]).view(-1, 1)
            ref = pdy[..., :L].double() - (a * (dbeta.view(-1, 1) + yhat * dgamma.view(-1, 1)) / n).double()
            torch.testing.assert_close(dy.double(), ref, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("T", [3, 20])
@pytest.mark.parametrize("L", [5, 49, 257])  # (a wavefront per row, rows packed into blocks, several rounds of a wavefront per row)
@pytest.mark.parametrize("last", [False, True])
def test_parametric_time_constant(C, T, L, last):
    B, Ch = 2, 20
    y, gs = seeded_randn((T, B, Ch, L), 8, 0.4, 1.2).cuda(), seeded_randn((T, B, Ch, L), 9).cuda()
    if last:  # only the row's last four positions, most of which two groups hold, have an upstream gradient
        gs[..., :-4] = 0.0
    stats = C._bn_map(y.flatten(0, 1), None, None, None, None, True, 0.1, 1e-5)
    v0 = torch.zeros((B, Ch, L), device="cuda")
    k = torch.tensor([0.4], device="cuda")
    spec = (0.0, *_spec(T)[1:])
    out = C._bn_lif_backward(y, stats, None, v0, spec, False, gs, None, False, False, k)
    ref = C._bn_lif_backward(_padded(y), stats, None, _padded(v0), spec, False, _padded(gs), None, False, False, k)
    # padded positions have no upstream gradient, hence no share in dL/dk
    assert torch.equal(out[0], ref[0][..., :L])
    torch.testing.assert_close(out[-1], ref[-1], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("train", [False, True])
def test_modules_take_the_fused_chain(train):
    """The attention block over 7 x 7 positions and a convolution block over 5 x 5: the fused chain runs, and equals the
    chain run module by module up to spikes at their threshold (another order of the convolution's sums)."""
    from spikingjelly_amd import configure
    from spikingjelly_amd.activation_based import functional, layer
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif
    from spikingjelly_amd.activation_based.model.spikformer import SpikformerConv2dBNLIF

    for make, shape in ((lambda: layer.SpikingSelfAttention(64, 2, backend="hip"), (4, 3, 64, 49)),
                        (lambda: SpikformerConv2dBNLIF(24, 40, 1, backend="hip"), (3, 2, 24, 5, 5))):
        torch.manual_seed(11)
        block = make().cuda().train(train)
        for m in block.modules():   # (scales and offsets that make the neurons fire)
            if isinstance(m, (torch.nn.BatchNorm1d, torch.nn.BatchNorm2d)):
                torch.nn.init.constant_(m.weight, 1.5), torch.nn.init.constant_(m.bias, 0.4), m.running_var.fill_(0.1)
        x = seeded_randn(shape, 12).cuda()
        results = []
        for fuse in (True, False):
            configure.hip_fuse_conv_bn_lif = fuse
            calls = []
            run = conv_bn_lif._chain_forward
            conv_bn_lif._chain_forward = lambda *a, **k: (calls.append(1), run(*a, **k))[1]
            try:
                xd = x.clone().requires_grad_()
                out = block(xd)
                out.backward(seeded_randn(tuple(out.shape), 13).cuda())
            finally:
                conv_bn_lif._chain_forward = run
                configure.hip_fuse_conv_bn_lif = True
            assert bool(calls) == fuse
            states = [m.v.clone() for m in block.modules() if hasattr(m, "v") and isinstance(m.v, torch.Tensor)]
            functional.reset_net(block)
            results.append((out.detach(), xd.grad, states, [p.grad.clone() for p in block.parameters()]))
            block.zero_grad()
        (a, ga, sa, pa), (b, gb, sb, pb) = results
        assert a.shape == b.shape and [s.shape for s in sa] == [s.shape for s in sb]
        assert 0.0 < float(b.mean()) < 1.0 and float((a != b).float().mean()) < 1e-3
        for p, q in zip([ga, *pa], [gb, *pb]):
            assert float((p - q).norm()) < 2e-2 * float(q.norm())


def test_evaluation_map_made_with_the_weights(C):
    """Without batch statistics the chain's first launch makes the batch norm's map: the bits of the finalizing launch."""
    T, B, Cin, Cout, L = 2, 3, 20, 133, 8
    x, w = seeded_randn((T, B, Cin, L), 20).cuda(), seeded_randn((Cout, Cin), 21).cuda()
    gamma, beta = seeded_randn((Cout,), 22, 1.0, 0.2).cuda(), seeded_randn((Cout,), 23, 0.2, 0.2).cuda()
    mean, var = seeded_randn((Cout,), 24).cuda(), seeded_randn((Cout,), 25).square().cuda()
    v0 = torch.zeros((B, Cout, L), device="cuda")
    for g, b in ((gamma, beta), (None, None)):
        for before in (mean.clone(),):
            _, _, y, bn_map, _ = C._chain_forward(x, None, x.shape, w, g, b, v0, (mean, var, False, 0.1, 1e-5), _spec(T), False, False, None)
            assert torch.equal(bn_map, C._bn_map(y.flatten(0, 1), g, b, mean, var, False, 0.1, 1e-5)) and torch.equal(mean, before)
