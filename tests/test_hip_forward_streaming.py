"""Forward calls whose tensors exceed the cache in front of the memory stream one side of their accesses
(``beyond_cache`` in ``csrc/neuron_fwd.hip``).  Neurons are independent columns, so the same columns computed in
slices small enough for the default policy have to give the same bits: spikes, states and gradients."""
import pytest
import torch

from spikingjelly_amd import configure
from spikingjelly_amd.activation_based import neuron, surrogate

pytestmark = pytest.mark.gpu

BOUND = 256 * 1024 * 1024 * 4 // 3  # bytes of the [T, N] tensors together


def run(x, v_seq, grad):
    node = neuron.LIFNode(tau=2.0, surrogate_function=surrogate.ATan(), step_mode="m", backend="hip", store_v_seq=v_seq).cuda()
    x = x.detach().requires_grad_(True)
    s = node(x)
    s.backward(grad)
    out = [s.detach(), node.v.detach().reshape(1, -1)] + ([node.v_seq.detach()] if v_seq else [])
    # (16-bit rows with fp32 state have one backward for whole 16-byte groups and one for ragged rows, which round differently)
    return out + ([x.grad] if configure.hip_half_precision_mode == "torch" or x.dtype == torch.float32 else [])


@pytest.mark.parametrize("dtype,mode,T,v_seq,beside", [
    (torch.float32, "torch", 2, False, 1),      # just beyond the bound, no whole number of 16-byte groups
    (torch.float32, "torch", 9, True, 3),
    (torch.float32, "torch", 70, False, 4),     # a long sequence: checkpoints beside the streamed spikes
    (torch.float32, "torch", 70, True, 2),
    (torch.float32, "torch", 3, False, 0),      # at the bound: the default policy
    (torch.float16, "torch", 3, False, 5),
    (torch.float16, "fp32_state", 2, False, 8),
    (torch.bfloat16, "torch", 6, False, 7),
    (torch.float16, "torch", 39, False, 3),     # the longest sequence that does not run in pieces
    (torch.bfloat16, "torch", 64, False, 7),    # in pieces: 16 bit keeps the default policy at any size
])
def test_streamed_calls_equal_their_slices(dtype, mode, T, v_seq, beside, monkeypatch):
    monkeypatch.setattr(configure, "hip_half_precision_mode", mode)
    size = torch.empty(0, dtype=dtype).element_size()
    N = BOUND // (size * (3 if v_seq else 2)) // T + beside
    g = torch.Generator(device="cuda").manual_seed(T + beside)
    x = torch.randn(T, N, generator=g, device="cuda").mul_(0.8).add_(0.6).to(dtype)
    grad = torch.randn(T, N, generator=g, device="cuda").to(dtype)
    whole = run(x, v_seq, grad)
    assert 0 < whole[0].float().mean().item() < 1
    step = (N // 3 + 8) // 8 * 8
    for c in range(0, N, step):
        part = run(x[:, c:c + step].contiguous(), v_seq, grad[:, c:c + step].contiguous())
        for a, b in zip(whole, part):
            assert torch.equal(a[:, c:c + step], b)
