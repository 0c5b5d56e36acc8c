"""The weight gradient over rows of at least eight groups of four positions: tile widths of one to three times 128 columns, chunks of the
contraction that end inside a sample, several partial tiles per chunk, a short last chunk, rows and columns beyond the tiles.

Against float64.  The 2-norm of the error stays below what sums of 32 bits over up to 42 steps of 32 positions, rounded as often as the
matrix cores round them, showed on the largest of these shapes (4.6e-7 of the result's); an element's below 2e-6 of the sum of its terms'
magnitudes, as for the shorter rows."""

import pytest
import torch

from helpers import seeded_randn

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S, M, N, L", [
    (2, 128, 384, 29), (1, 1, 1, 32), (5, 130, 390, 36), (3, 129, 127, 31),   # a step or two, edges of the tiles
    (128, 512, 512, 49), (192, 64, 64, 49),                                    # short chains: several sums per chunk
    (300, 260, 257, 64), (96, 512, 256, 400), (1000, 256, 768, 33),            # widths of one to three
    (256, 1152, 384, 196), (128, 1536, 384, 196),                              # long chains: two partial tiles per chunk
])
@pytest.mark.parametrize("spikes", [False, True])
def test_against_float64(S, M, N, L, spikes):
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C
    from spikingjelly_amd.activation_based.hip_kernel.compress import bit_spike_compress

    g = torch.Generator(device="cuda").manual_seed(S + M)
    dy = torch.randn((S, M, L), generator=g, device="cuda")
    x = torch.randn((S, N, L), generator=g, device="cuda")
    if spikes:
        x = (x > 0.5).float()
    got = C.pw_grad_weight(dy, C.F16 | 2, x, C.F16 | 1 if spikes else C.F16 | 2)
    want, bound = (torch.zeros((M, N), dtype=torch.float64, device="cuda") for _ in range(2))
    for s in range(0, S, 32):  # [M, 32 L] x [32 L, N], both contiguous
        a = dy[s:s + 32].transpose(0, 1).reshape(M, -1).double()
        b = x[s:s + 32].transpose(1, 2).reshape(-1, N).double().contiguous()
        want += a @ b
        bound += a.abs() @ b.abs()
    error = got.double() - want
    assert float(error.norm() / want.norm()) < 4.6e-7
    assert float((error.abs() / bound.clamp_min(1e-300)).max()) < 2e-6
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


def _longest_sum(S, M, N, L):
    """K steps (32 positions) that a sum of 32 bits may hold: the chunk of whole samples that one block took when every product went
    into one sum (n), and 5 / 2 of it, at most 3 n - 2, on tiles where the products of small terms have sums of their own."""
    tiles = -(-M // 128) * -(-N // 128)
    samples = -(-S // min(S, max(1, (1024 if tiles >= 16 else 512) // tiles)))
    n = -(-samples * (-(-L // 4) * 4) // 32)
    return max(n, min(5 * n // 2, 3 * n - 2))


@pytest.mark.parametrize("S, M, N, L", [
    (32, 1152, 384, 64), (20, 1376, 480, 49), (20, 1408, 448, 49),  # chunks whose last pieces are the tail of the loop
    (36, 1248, 160, 49), (128, 512, 512, 49), (100, 1152, 384, 36),
])
def test_no_sum_is_longer_than_its_limit(S, M, N, L):
    """A term of 1/2 that is a whole limit of K steps away from 2^25 and from -2^25 is in neither's sum: the products are exact, the
    partial tiles are added in 64 bits, so the result is 1/2 exactly; added to 2^25 in 32 bits it would be lost."""
    from spikingjelly_amd.activation_based.hip_kernel import conv_bn_lif as C

    limit, quads = _longest_sum(S, M, N, L), -(-L // 4)
    last = S * quads // 8 - 1
    assert last >= 2 * limit
    first = torch.arange(M, device="cuda") % (last - 2 * limit + 1)
    dy = torch.zeros((S, M, L), device="cuda")
    for distance, value in ((0, 2.0 ** 25), (limit, 0.5), (2 * limit, -2.0 ** 25)):
        quad = (first + distance) * 8
        dy[quad // quads, torch.arange(M, device="cuda"), quad % quads * 4] = value
    got = C.pw_grad_weight(dy, C.F16 | 2, torch.ones((S, N, L), device="cuda"), C.F16 | 2)
    assert torch.equal(got, torch.full((M, N), 0.5, device="cuda"))
