"""The weight gradient over rows of at least eight groups of four positions: tile widths of one to three times 128 columns, chunks of the
contraction that end inside a sample, several partial tiles per chunk, a short last chunk, rows and columns beyond the tiles.

Against float64.  The 2-norm of the error, relative to the result's, stays below that of the kernel with one sum of 32 bits per chunk of
whole samples (``pw_dw_kernel``), measured on the same inputs and written beside each shape; an element's below 2e-6 of the sum of its
terms' magnitudes, as for the shorter rows."""

import pytest
import torch

from helpers import seeded_randn

pytestmark = pytest.mark.gpu


FORMER = [  # S, M, N, L; error of the former kernel in 1e-8: fp32 x (two terms), bfloat16 values and spikes (one term)
    # a step or two, edges of the tiles
    (2, 128, 384, 29, 10.14, 7.37, 6.80), (5, 130, 390, 36, 10.64, 7.82, 7.17),
    (3, 129, 127, 31, 9.95, 7.38, 6.76),
    # few samples or short rows: sums of a few steps
    (4, 1152, 512, 32, 9.90, 7.21, 6.72), (4, 1376, 224, 30, 10.06, 7.32, 6.82),
    (31, 1536, 160, 29, 10.73, 8.16, 7.55), (38, 1152, 384, 30, 12.02, 9.13, 8.09),
    (60, 1536, 512, 32, 13.50, 10.41, 8.92), (58, 416, 416, 36, 11.84, 9.25, 8.44),
    (20, 1376, 480, 49, 11.92, 8.90, 7.80), (36, 1152, 384, 49, 12.20, 9.22, 8.17),
    (44, 512, 512, 49, 12.42, 9.42, 8.22), (192, 64, 64, 49, 14.94, 12.03, 10.90),
    (128, 512, 512, 49, 14.75, 11.50, 9.83), (32, 1152, 384, 64, 12.18, 9.32, 8.21),
    (41, 1472, 480, 64, 14.82, 11.56, 9.68),
    # widths of one to three
    (300, 260, 257, 64, 24.43, 19.22, 14.52), (96, 512, 256, 400, 34.82, 27.10, 19.53),
    (1000, 256, 768, 33, 35.98, 28.10, 20.07),
    # long sums: two partial tiles per chunk
    (256, 1152, 384, 196, 46.01, 35.36, 24.80), (128, 1536, 384, 196, 37.34, 29.46, 21.28),
]


def _error(S, M, N, L, x, x_terms):
    """``(dw, dy, x, largest error of an element over the sum of its terms' magnitudes, 2-norm of the error over the result's)``"""
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C

    g = torch.Generator(device="cuda").manual_seed(S + M)
    dy = torch.randn((S, M, L), generator=g, device="cuda")
    x = x(torch.randn((S, N, L), generator=g, device="cuda"))
    got = C.pw_grad_weight(dy, C.F16 | 2, x, C.F16 | x_terms)
    want, bound = (torch.zeros((M, N), dtype=torch.float64, device="cuda") for _ in range(2))
    for s in range(0, S, 32):  # [M, 32 L] x [32 L, N], both contiguous
        a = dy[s:s + 32].transpose(0, 1).reshape(M, -1).double()
        b = x[s:s + 32].transpose(1, 2).reshape(-1, N).double().contiguous()
        want += a @ b
        bound += a.abs() @ b.abs()
    error = got.double() - want
    return got, dy, x, float((error.abs() / bound.clamp_min(1e-300)).max()), float(error.norm() / want.norm())


@pytest.mark.parametrize("S, M, N, L, fp32, bf16, spikes", FORMER)
def test_no_further_from_float64_than_one_sum_per_chunk(S, M, N, L, fp32, bf16, spikes):
    """(2 %: sums in another order; the results have at least 4096 elements)"""
    for former, x, terms in ((fp32, lambda v: v, 2), (bf16, lambda v: v.bfloat16().float(), 1), (spikes, lambda v: (v > 0.5).float(), 1)):
        assert _error(S, M, N, L, x, terms)[4] < 1.02e-8 * former


@pytest.mark.parametrize("S, M, N, L", [(1, 1, 1, 32)] + [case[:4] for case in FORMER])
@pytest.mark.parametrize("spikes", [False, True])
def test_against_float64(S, M, N, L, spikes):
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C
    from spikingjelly_amd.activation_based.hip_kernel.compress import bit_spike_compress

    got, dy, x, largest, norm = _error(S, M, N, L, (lambda v: (v > 0.5).float()) if spikes else (lambda v: v), 1 if spikes else 2)
    assert norm < 4.6e-7 and largest < 2e-6
    if spikes and L % 4 == 0 and N * L % 8 == 0:
        assert torch.equal(C.pw_grad_weight_bits(dy, bit_spike_compress(x), N), got)


def test_positions_beyond_the_last_chunk_do_not_count():
    """A last K step with less than eight groups: what lies behind the tensors in memory takes no part."""
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C

    for S, L in ((1, 36), (3, 44), (7, 100), (5, 49)):
        room_dy = torch.full((S * 40 * L + 4096,), float("nan"), device="cuda")
        room_x = torch.full((S * 24 * L + 4096,), float("nan"), device="cuda")
        dy, x = room_dy[:S * 40 * L].view(S, 40, L), room_x[:S * 24 * L].view(S, 24, L)
        dy.copy_(seeded_randn((S, 40, L), 1))
        x.copy_(seeded_randn((S, 24, L), 2))
        amax = [C.amax(t.clone()) for t in (dy, x)]
        got = C.pw_grad_weight(dy, C.F16 | 2, x, C.F16 | 2, *amax)
        want = torch.einsum("sml,snl->mn", dy.double().cpu(), x.double().cpu())
        torch.testing.assert_close(got.double().cpu(), want, rtol=1e-5, atol=1e-5)


def _longest_sum(S, M, N, L, x_terms):
    """K steps (32 positions) that a sum of 32 bits may hold.  A chunk of whole samples that one block of the former kernel took, in
    quads of positions; on tiles where the products of small terms have sums of their own 5 / 2 of it if it is longer than a step, with
    one term of x twice its length less a step and a half, and from three steps on only (below, the former kernel runs)."""
    tiles = -(-M // 128) * -(-N // 128)
    samples = -(-S // min(S, max(1, (1024 if tiles >= 16 else 512) // tiles)))
    quads = samples * -(-L // 4)
    if x_terms == 1:
        return (quads - 6) // 4 if quads >= 24 else -(-quads // 8)
    return 5 * quads // 16 if quads > 8 else 1


@pytest.mark.parametrize("S, M, N, L", [
    (32, 1152, 384, 64), (20, 1376, 480, 49), (20, 1408, 448, 49),  # chunks whose last pieces are the tail of the loop
    (36, 1248, 160, 49), (128, 512, 512, 49), (100, 1152, 384, 36), (58, 416, 416, 36), (41, 1472, 480, 64), (60, 1536, 512, 32), (38, 1152, 384, 30),
])
@pytest.mark.parametrize("x_terms", [1, 2])
def test_no_sum_is_longer_than_its_limit(S, M, N, L, x_terms):
    """A term of 1/2 that is a whole limit of K steps away from 2^25 and from -2^25 is in neither's sum: the products are exact, the
    partial tiles are added in 64 bits, so the result is 1/2 exactly; added to 2^25 in 32 bits it would be lost."""
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C

    limit, quads = _longest_sum(S, M, N, L, x_terms), -(-L // 4)
    last = S * quads // 8 - 1
    assert last >= 2 * limit
    first = torch.arange(M, device="cuda") % (last - 2 * limit + 1)
    dy = torch.zeros((S, M, L), device="cuda")
    for distance, value in ((0, 2.0 ** 25), (limit, 0.5), (2 * limit, -2.0 ** 25)):
        quad = (first + distance) * 8
        dy[quad // quads, torch.arange(M, device="cuda"), quad % quads * 4] = value
    got = C.pw_grad_weight(dy, C.F16 | 2, torch.ones((S, N, L), device="cuda"), C.F16 | x_terms)
    assert torch.equal(got, torch.full((M, N), 0.5, device="cuda"))


@pytest.mark.parametrize("S, M, N, L", [(1, 128, 128, 196), (4, 384, 384, 196), (20, 1376, 480, 49), (3, 129, 127, 31), (128, 512, 512, 49), (5, 40, 24, 20)])
@pytest.mark.parametrize("x_terms", [1, 2])
def test_workspace_of_the_stated_size_is_enough(S, M, N, L, x_terms):
    """(a buffer for any length, of which the part beyond the stated size keeps its contents)"""
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C

    lib = C.L.load()
    size = lib.sjhip_pwconv_grad_weight_workspace_floats_for(M, N, S, L, C.F16 | 2, x_terms)
    room = torch.full((lib.sjhip_pwconv_grad_weight_workspace_floats(M, N, S),), 7.0, device="cuda")
    dy, x = seeded_randn((S, M, L), 1).cuda(), (seeded_randn((S, N, L), 2) > 0.5).float().cuda()
    amax, dw = [C.amax(t) for t in (dy, x)], torch.empty((M, N), device="cuda")
    assert lib.sjhip_pwconv_grad_weight_f16(dy.data_ptr(), amax[0].data_ptr(), x.data_ptr(), x_terms, amax[1].data_ptr(), S, M, N, L,
                                            dw.data_ptr(), room.data_ptr(), C._stream(dy)) == 0
    assert bool((room[size:] == 7.0).all()) and torch.equal(dw, C.pw_grad_weight(dy, C.F16 | 2, x, C.F16 | x_terms))
