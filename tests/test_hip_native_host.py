"""The native host path (``csrc/torch_binding.cpp``) against the general Python path: same kernels, so the same bits, for the
states, layouts and gradients where the two could part; and the calls it must leave to the general path."""

import pytest
import torch

from spikingjelly_amd import configure
from spikingjelly_amd.activation_based import functional, neuron, surrogate
from spikingjelly_amd.activation_based.functional import neuron as F
from spikingjelly_amd.activation_based.hip_kernel import native
from spikingjelly_amd.activation_based.hip_kernel.surrogate_registry import resolve_sg_hip_id_and_alpha

pytestmark = pytest.mark.gpu

EXTRA = (0.0,) * 6


def _both(monkeypatch, fn):
    served = []
    module = native.load()

    class Spy:
        def __getattr__(self, name):
            def call(*a):
                out = getattr(module, name)(*a)
                served.append(out is not None)
                return out

            return call

    monkeypatch.setattr(F, "_native", (Spy(), resolve_sg_hip_id_and_alpha))
    got = fn()
    monkeypatch.setattr(F, "_native_sequence", lambda *a, **k: None)
    return got, fn(), served


def _equal(a, b):
    assert len(a) == len(b)
    for x, y in zip(a, b):
        assert (x is None) == (y is None) and (x is None or (x.dtype == y.dtype and x.shape == y.shape and torch.equal(x, y)))


@pytest.mark.parametrize("shape", [(4, 8, 16, 1, 1), (3, 1, 40), (2, 5, 1), (1, 64)])
@pytest.mark.parametrize("kind", ["if", "lif", "plif"])
@pytest.mark.parametrize("state", ["fresh", "dense", "needs_grad"])
def test_native_and_general_path_give_the_same_bits(kind, shape, state, monkeypatch):
    g = torch.Generator().manual_seed(sum(shape))
    x0 = (torch.randn(shape, generator=g) + 0.4).cuda()
    gs = torch.randn(shape, generator=g).cuda()
    v0 = (torch.randn(shape[1:], generator=g) * 0.2).cuda()
    cls = {"if": neuron.IFNode, "lif": neuron.LIFNode, "plif": neuron.ParametricLIFNode}[kind]

    def run():
        node = cls(step_mode="m", backend="hip", surrogate_function=surrogate.ATan(), store_v_seq=True).cuda()
        x = x0.clone().requires_grad_()
        v = v0.clone().requires_grad_(state == "needs_grad")
        if state != "fresh":
            node.v = v
        s = node(x)
        (s * gs).sum().backward(retain_graph=True)
        (node.v_seq.sum() + 2.0 * node.v.sum()).backward()  # a second backward through the same node: gradients add up
        return [s.detach(), node.v.detach(), node.v_seq.detach(), x.grad, v.grad] + [p.grad for p in node.parameters()]

    got, want, served = _both(monkeypatch, run)
    N = x0.numel() // shape[0]
    assert served == [N >= 4]  # shorter rows than a vector save h: the general path's business
    _equal(got, want)


def test_truncated_backpropagation_crosses_calls(monkeypatch):
    x0 = (torch.randn(2, 3, 64, generator=torch.Generator().manual_seed(5)) + 0.4).cuda()

    def run():
        node = neuron.LIFNode(step_mode="m", backend="hip", surrogate_function=surrogate.ATan()).cuda()
        x = x0.clone().requires_grad_()
        first = node(x)
        second = node(x * 0.5)  # its state is the first call's
        (second.sum() + 0.1 * first.sum()).backward()
        return [second.detach(), x.grad]

    got, want, served = _both(monkeypatch, run)
    assert served == [True, True]
    _equal(got, want)


def test_single_steps(monkeypatch):
    x0 = (torch.randn(5, 7, 33, generator=torch.Generator().manual_seed(6)) + 0.4).cuda()

    def run():
        node = neuron.LIFNode(step_mode="s", backend="hip", surrogate_function=surrogate.ATan()).cuda()
        x = x0.clone().requires_grad_()
        out = torch.stack([node(x[t]) for t in range(5)])
        (out * torch.arange(5, device="cuda").view(5, 1, 1)).sum().backward()
        return [out.detach(), x.grad, node.v.detach()]

    got, want, served = _both(monkeypatch, run)
    assert served == [True] * 5
    _equal(got, want)


def test_what_the_native_path_leaves_alone(monkeypatch):
    m = native.load()
    call = lambda x, v, steps=39: m.neuron_sequence(x, v, None, False, 1, 2.0, 1.0, 0.0, 1, 1, 2.0, False, steps, EXTRA)
    x = torch.randn(4, 64, device="cuda")
    v = torch.zeros(64, device="cuda")
    assert call(x, v) is not None
    assert call(x.double(), v.double()) is None                          # a dtype without kernels: the general path raises
    assert call(torch.randn(64, 4, device="cuda").t(), v) is None        # a layout that needs a copy
    assert call(x, v[:32]) is None and call(x, v.half()) is None
    assert call(x.cpu(), v.cpu()) is None
    xg = x.clone().requires_grad_()
    assert call(xg, v, steps=3) is None                                  # too long to replay in one piece
    assert call(xg, v, steps=4) is not None
    with torch.no_grad():
        assert call(xg, v, steps=0) is not None                          # inference replays nothing
    seen = []
    torch.func.vmap(lambda t: (seen.append(call(t, v) is None), t)[1])(torch.randn(2, 4, 64, device="cuda"))
    assert seen == [True]


@pytest.mark.parametrize("dual", ["x", "v", "w"])
def test_forward_mode_derivatives_are_refused_not_dropped(dual):
    """The kernels carry no tangents: a call that would have to produce one raises, whichever argument brings it."""
    import torch.autograd.forward_ad as fwAD

    t = {"x": torch.randn(4, 64, device="cuda"), "v": torch.zeros(64, device="cuda"), "w": torch.tensor(0.2, device="cuda")}
    with fwAD.dual_level():
        t[dual] = fwAD.make_dual(t[dual].requires_grad_(), torch.ones_like(t[dual]))
        with pytest.raises(NotImplementedError, match="jvp"):
            functional.plif_multi_step_hip(t["x"], t["v"], t["w"], True, 1.0, 0.0, surrogate.ATan())


def test_traced_call_follows_its_input():
    """``torch.jit.trace`` records the autograd function; an untraced call would leave its result in the trace as a constant."""
    x, v = torch.randn(4, 64, device="cuda").requires_grad_(), torch.zeros(64, device="cuda")
    fn = lambda t: functional.lif_multi_step_hip(t, v, 2.0, True, 1.0, 0.0, surrogate.ATan())[0]
    traced = torch.jit.trace(fn, (x,), check_trace=False)
    for shift in (0.0, 1.0, 3.0):
        y = (x.detach() + shift).requires_grad_()
        assert torch.equal(traced(y), fn(y))


def test_training_call_without_a_surrogate_function_is_refused():
    x, v, w = torch.randn(4, 64, device="cuda").requires_grad_(), torch.zeros(64, device="cuda"), torch.zeros((), device="cuda")
    for call in (lambda: functional.if_multi_step_hip(x, v, 1.0, 0.0, None),
                 lambda: functional.lif_multi_step_hip(x, v, 2.0, True, 1.0, 0.0, None),
                 lambda: functional.plif_multi_step_hip(x, v, w, True, 1.0, 0.0, None),
                 lambda: functional.lif_step_hip(x[0], v, 2.0, True, 1.0, 0.0, None)):
        with pytest.raises(NotImplementedError, match="surrogate"):
            call()
        with torch.no_grad():
            call()


def test_sequences_without_a_neuron_dimension_are_refused():
    x = torch.randn(4, device="cuda")
    for call in (lambda: functional.lif_multi_step_hip(x, x[0], 2.0, True, 1.0, 0.0, surrogate.ATan()),
                 lambda: functional.lif_step_hip(x[0], x[1], 2.0, True, 1.0, 0.0, surrogate.ATan()),
                 lambda: functional.lif_multi_step_hip_packed(torch.randn(8, device="cuda"), x[0], 2.0, True, 1.0, 0.0)):
        with pytest.raises(IndexError):
            call()


class _Tagged(torch.Tensor):
    pass


@pytest.mark.parametrize("grad", [False, True])
def test_results_keep_the_type_of_a_tensor_subclass(grad):
    x, v = torch.randn(4, 64, device="cuda").as_subclass(_Tagged).requires_grad_(grad), torch.zeros(64, device="cuda")
    out = functional.lif_multi_step_hip(x, v, 2.0, True, 1.0, 0.0, surrogate.ATan(), store_v_seq=True)
    assert [type(t) for t in out] == [_Tagged] * 3
    step = functional.lif_step_hip(x[0], v, 2.0, True, 1.0, 0.0, surrogate.ATan())
    assert [type(t) for t in step] == [_Tagged] * 2
    if not grad:
        _, v_last, v_seq = functional.lif_multi_step_hip_packed(x, v, 2.0, True, 1.0, 0.0, True)
        assert type(v_last) is _Tagged and type(v_seq) is _Tagged


def test_saved_tensors_go_through_hooks_and_are_freed():
    packed = []
    x = torch.randn(4, 64, device="cuda").requires_grad_()
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (packed.append(t.shape), t.cpu())[1], lambda t: t.cuda()):
        s, _, _ = functional.lif_multi_step_hip(x, torch.zeros(64, device="cuda"), 2.0, True, 1.0, 0.0, surrogate.ATan())
    s.sum().backward()
    assert torch.Size((4, 64)) in packed
    with pytest.raises(RuntimeError, match="backward through the graph a second time"):
        s.sum().backward()
    x2 = torch.randn(4, 64, device="cuda").requires_grad_()
    y = x2 * 1.0
    s, _, _ = functional.lif_multi_step_hip(y, torch.zeros(64, device="cuda"), 2.0, True, 1.0, 0.0, surrogate.ATan())
    y.add_(1.0)
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        s.sum().backward()


def _calls(x, v, w):
    sg = surrogate.ATan()
    levels = surrogate.MultiLevelSpikeCount(4)
    return {
        "if": lambda: functional.if_multi_step_hip(x, v, 1.0, None, sg, True),
        "lif": lambda: functional.lif_multi_step_hip(x, v, 2.0, True, 1.0, 0.0, sg, store_v_seq=True),
        "plif": lambda: functional.plif_multi_step_hip(x, v, w, False, 1.0, 0.0, sg),
        "qif": lambda: functional.qif_multi_step_hip(x, v, 2.0, 1.0, 0.0, 0.0, 0.8, 1.0, False, sg),
        "eif": lambda: functional.eif_multi_step_hip(x, v, 2.0, 1.0, 0.0, 0.0, 0.8, 1.0, False, sg),
        "ilif": lambda: functional.ilif_multi_step_hip(x, v, 2.0, 1.0, levels),
        "step": lambda: functional.lif_step_hip(x[0], v, 2.0, True, 1.0, 0.0, sg),
    }


@pytest.mark.parametrize("compiler", ["graph module", "eager", "aot_eager"])
@pytest.mark.parametrize("kind", ["if", "lif", "plif", "qif", "eif", "ilif", "step"])
def test_compiled_autograd_records_the_operators(kind, compiler):
    """Compiled autograd asks a C++ node for its arguments and for its backward on recorded tensors."""
    from torch._dynamo import compiled_autograd

    torch._dynamo.reset()
    enable = (lambda gm: gm) if compiler == "graph module" else torch.compile(backend=compiler)
    g = torch.Generator().manual_seed(8)
    for T, v_th in ((4, 1.0), (3, 1.0)):
        x0, v0 = (torch.randn(T, 8, 5, generator=g) + 0.4).cuda(), (torch.randn(8, 5, generator=g) * 0.2).cuda()
        results = []
        for compiled in (False, True):
            x, v, w = x0.clone().requires_grad_(), v0.clone().requires_grad_(), torch.tensor(0.2, device="cuda").requires_grad_()
            s, v_last, *rest = _calls(x * 1.5, v, w)[kind]()
            loss = (s * torch.arange(5.0, device="cuda")).sum() + v_last.sum() + sum(r.square().sum() for r in rest if r is not None)
            if compiled:
                with compiled_autograd._enable(enable):
                    loss.backward()
            else:
                loss.backward()
            results.append([x.grad, v.grad, w.grad])
        _equal(*results)


def _reversed_strides(t):
    out = torch.empty(t.shape[::-1], dtype=t.dtype, device=t.device).permute(*range(t.dim() - 1, -1, -1))
    return out.copy_(t)


@pytest.mark.parametrize("unpack", [_reversed_strides, lambda t: t.clone(memory_format=torch.contiguous_format), lambda t: t.double(),
                                    lambda t: t[..., :1].clone().expand(t.shape) if t.dim() == 2 and bool((t == t.flatten()[0]).all()) else t,
                                    lambda t: torch.cat([t.flatten()[:1], t.flatten()])[1:].view(t.shape)],
                         ids=["strided", "dense", "double", "expanded", "off 16 bytes"])
@pytest.mark.parametrize("state", ["one element", "constant", "dense"])
def test_saved_tensors_come_back_in_any_layout(unpack, state):
    g = torch.Generator().manual_seed(7)
    x0, gs = (torch.randn(3, 8, 5, generator=g) + 0.4).cuda(), torch.randn(3, 8, 5, generator=g).cuda()
    v0 = {"one element": torch.full((1, 1), 0.25).cuda().expand(8, 5), "constant": torch.full((8, 5), 0.25).cuda(),
          "dense": (torch.randn(8, 5, generator=g) * 0.2).cuda()}[state]
    results = []
    for hook in (lambda t: t, lambda t: unpack(t) if t.dim() else t):  # (sigmoid(w), which sigmoid saves as well, stays as it is)
        x, w = x0.clone().requires_grad_(), torch.tensor(0.2, device="cuda").requires_grad_()
        v = v0 if state == "one element" else v0.clone().requires_grad_()
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, hook):
            s = functional.plif_multi_step_hip(x, v, w, True, 1.0, 0.0, surrogate.ATan())[0]
        s.backward(gs)
        results.append([x.grad, v.grad, w.grad])
    _equal(*results)


@pytest.mark.parametrize("what", ["device", "size"])
@pytest.mark.parametrize("which", ["x_seq", "v_init", "k"])
def test_saved_tensors_that_are_not_the_saved_ones_are_refused(what, which):
    x, v = torch.randn(4, 64, device="cuda").requires_grad_(), torch.zeros(64, device="cuda")
    k = torch.tensor(0.4, device="cuda").requires_grad_()
    other = (lambda t: t.cpu()) if what == "device" else (lambda t: t[..., :32].contiguous() if t.dim() else t.expand(2).contiguous())
    dim = {"x_seq": 2, "v_init": 1, "k": 0}[which]
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: other(t) if t.dim() == dim else t):
        s = native.load().neuron_sequence(x, v, k, False, 2, 0.0, 1.0, 0.0, 1, 1, 2.0, False, 39, EXTRA)[0]
    with pytest.raises(RuntimeError, match=f"saved {which}"):
        s.sum().backward()


def test_calls_on_a_side_stream():
    """Forward on a stream of its own, backward asked for from the main stream: kernels and memory stay with the forward's
    stream, also while the main stream allocates and works."""
    g = torch.Generator().manual_seed(9)
    x0, gs = (torch.randn(6, 1 << 16, generator=g) + 0.4).cuda(), torch.randn(6, 1 << 16, generator=g).cuda()
    v = torch.zeros(1 << 16, device="cuda")

    def run(stream):
        x = x0.clone().requires_grad_()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            out = functional.lif_multi_step_hip(x * 1.25, v, 2.0, True, 1.0, 0.0, surrogate.ATan(), store_v_seq=True)
        noise = [torch.randn(6, 1 << 16, device="cuda") for _ in range(4)]
        torch.cuda.current_stream().wait_stream(stream)
        (out[0] * gs + out[2]).sum().backward()
        return [t.detach() for t in out] + [x.grad, sum(noise)]

    want = run(torch.cuda.current_stream())[:4]
    side = torch.cuda.Stream()
    for _ in range(5):
        got = run(side)[:4]
        torch.cuda.synchronize()
        _equal(got, want)


def test_packed_inference_equals_the_operator():
    x = (torch.rand(6, 5, 16, device="cuda") * 0.6).half()
    v = torch.zeros(5, 16, dtype=torch.float16, device="cuda")
    bits, v1, v_seq = functional.if_multi_step_hip_packed(x, v, 1.0, None, True)
    want = torch.ops.sj.hip_multistep_if_inference_packed(x.flatten(1), v.flatten(), 1.0, 0.0, True, True, F._hip_mode_flags(x))
    assert torch.equal(bits, want[0]) and torch.equal(v_seq.flatten(1), want[1]) and torch.equal(v1.flatten(), want[2])
    assert configure.hip_half_precision_mode == "torch"
