"""The graph that `causal_conv1d_fn` records from C++ against the one of `CausalConv1dFn`, the Python function:
which of the two a call takes, that hooks and checkpoints see the same tensors in both, that every input gets its
gradient whatever happens to the saved tensors in between, and that the gradients are the same bits, also for inputs
without gradients, outputs without one and a second pass."""
import contextlib

import pytest
import torch
from torch._dynamo import compiled_autograd
from torch.utils.checkpoint import checkpoint

from helpers import gen, make_states, make_wb, make_x, random_seq_idx, to_dev_like


def _meta(*shape, grad=False):
    return torch.zeros(*shape, device="meta", requires_grad=grad)


def _native(t):
    return "CppNode" in t.grad_fn.name()


def test_which_graph_a_call_takes(pkg, monkeypatch):
    """On meta tensors, without a GPU."""
    from causal_conv1d import cpp_functions
    x, w, b, init = _meta(2, 8, 9, grad=True), _meta(8, 4), _meta(8), _meta(2, 8, 3)
    assert _native(pkg.causal_conv1d_fn(x, w, b)) and _native(pkg.causal_conv1d_fn(x.detach(), w, b.requires_grad_()))
    assert all(_native(t) for t in pkg.causal_conv1d_fn(x, w, b, initial_states=init, return_final_states=True))
    assert pkg.causal_conv1d_fn(x.detach(), w, b.detach()).grad_fn is None
    with torch.no_grad():
        assert pkg.causal_conv1d_fn(x, w, b).grad_fn is None
    # left to the Python function: the caller's final_states, return_final_states that is no bool, x that needs a copy, a
    # subclass, a forward-mode gradient, a replaced backward
    out, fin = pkg.causal_conv1d_fn(x, w, b, return_final_states=True, final_states_out=_meta(2, 3, 8).transpose(1, 2))
    assert not _native(out)
    assert not _native(pkg.causal_conv1d_fn(x, w, b, return_final_states=1)[0])
    assert not _native(pkg.causal_conv1d_fn(_meta(2, 16, 18, grad=True)[:, ::2, ::2], w, b))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(w, _meta(8, 4))
        with pytest.raises(RuntimeError, match="jvp"):
            pkg.causal_conv1d_fn(x, dual, b)
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.func.grad(lambda q: pkg.causal_conv1d_fn(x, q, b).sum())(w)
    with pytest.raises(RuntimeError, match="setup_context"):
        torch.vmap(lambda q: pkg.causal_conv1d_fn(q, w, b))(_meta(3, 2, 8, 9, grad=True))
    with pytest.raises(NotImplementedError, match="activation"):
        pkg.causal_conv1d_fn(x, w, b, activation="relu")
    monkeypatch.setattr(cpp_functions, "_direct_backward", lambda *a: NotImplemented)
    assert not _native(pkg.causal_conv1d_fn(x, w, b))


def _both(monkeypatch, f):
    from causal_conv1d import causal_conv1d_interface as interface
    native = f()
    monkeypatch.setattr(interface, "_direct_forward", lambda *a: NotImplemented)
    return native, f()


def test_hooks_and_second_order(pkg, monkeypatch):
    """On meta tensors, without a GPU."""
    def saved():
        seen = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(tuple(t.shape)), t)[1], lambda t: (seen.append("unpacked"), t)[1]):
            leaves = [_meta(2, 8, 9, grad=True), _meta(8, 4, grad=True), _meta(2, 8, 3, grad=True)]
            pkg.causal_conv1d_fn(leaves[0], leaves[1], initial_states=leaves[2]).sum().backward()
        return seen

    def second():
        leaves = [_meta(2, 8, 9, grad=True), _meta(8, 4, grad=True)]
        out = pkg.causal_conv1d_fn(*leaves)
        grads = torch.autograd.grad(out, leaves, _meta(2, 8, 9), create_graph=True)
        return [g.requires_grad for g in grads]

    def twice():
        out = pkg.causal_conv1d_fn(_meta(2, 8, 9, grad=True), _meta(8, 4))
        out.sum().backward()
        with pytest.raises(RuntimeError, match="second time"):
            out.sum().backward()

    native, python = _both(monkeypatch, lambda: (saved(), second(), twice()))
    assert native == python and len(native[0]) == 6


@pytest.mark.parametrize("compiled", [False, True], ids=["engine", "compiled_autograd"])
@pytest.mark.parametrize("between", ["nothing", "hooks", "checkpoint", "reentrant", "detached"])
def test_every_gradient_arrives(pkg, monkeypatch, between, compiled):
    """On meta tensors, without a GPU: what happens to initial_states between forward and backward (saved-tensor hooks
    that hand back another tensor, a checkpoint's second forward, an in-place detach) takes no gradient away.
    initial_states are a leaf, or in front of one."""
    if between == "reentrant" and compiled:
        pytest.skip("a reentrant checkpoint runs the engine inside of the engine")

    def run(leaf):
        leaves = [_meta(2, 8, 9, grad=True), _meta(8, 4, grad=True), _meta(8, grad=True), _meta(2, 8, 3, grad=True)]
        init = leaves[3] if leaf else leaves[3] * 2
        f = lambda x, w, b, i: pkg.causal_conv1d_fn(x, w, b, initial_states=i, return_final_states=True, activation="silu")
        hooks = torch.autograd.graph.saved_tensors_hooks(lambda t: t.detach(), lambda t: t) if between == "hooks" else contextlib.nullcontext()
        with hooks:
            if between in ("checkpoint", "reentrant"):
                out, fin = checkpoint(f, *leaves[:3], init, use_reentrant=between == "reentrant")
            else:
                out, fin = f(*leaves[:3], init)
        if between == "detached" and not leaf:
            init.detach_()
        with compiled_autograd._enable(torch.compile(backend="eager")) if compiled else contextlib.nullcontext():
            (out.sum() + fin.sum()).backward()
        return [None if t.grad is None else tuple(t.grad.shape) for t in leaves]

    native, python = _both(monkeypatch, lambda: (run(True), run(False)))
    assert native == python == ([(2, 8, 9), (8, 4), (8,), (2, 8, 3)],) * 2


def test_saved_tensors_of_the_node(pkg, monkeypatch):
    """On meta tensors, without a GPU: grad_fn.saved_tensors in every combination of activation, final states and states."""
    def run():
        seen = []
        for activation in (None, "silu"):
            for final in (False, True):
                for init in (None, _meta(2, 8, 3), _meta(2, 8, 3, grad=True)):
                    x, w = _meta(2, 8, 9, grad=True), _meta(8, 4)
                    out = pkg.causal_conv1d_fn(x, w, initial_states=init, return_final_states=final, activation=activation)
                    out = out[0] if final else out
                    saved = out.grad_fn.saved_tensors
                    assert len(saved) == 5 and saved[0] is x and saved[1] is w and saved[4] is init
                    seen.append((type(out.grad_fn).__name__, [t if t is None else tuple(t.shape) for t in saved]))
                    out.sum().backward()
                    with pytest.raises(RuntimeError, match="second time"):
                        out.grad_fn.saved_tensors
        return seen

    native, python = _both(monkeypatch, run)
    assert native == python


def test_gradient_of_states_that_need_a_copy(pkg):
    """On meta tensors, without a GPU: initial_states with no unit stride are copied first, and keep their gradient."""
    x, w, init = _meta(2, 8, 9, grad=True), _meta(8, 4), _meta(2, 16, 6, grad=True)
    pkg.causal_conv1d_fn(x, w, initial_states=init[:, ::2, ::2]).sum().backward()
    assert x.grad.shape == x.shape and init.grad is not None and init.grad.shape == init.shape


@pytest.mark.gpu
@pytest.mark.parametrize("channel_last", [False, True], ids=["cf", "cl"])
@pytest.mark.parametrize("extra", ["none", "states", "seq_idx", "no_bias"])
def test_both_graphs_give_the_same(pkg, gpu_device, monkeypatch, channel_last, extra):
    if extra == "seq_idx" and not channel_last:
        pytest.skip("seq_idx needs channel-last x")
    g = gen(77)
    B, D, L, W, dtype = 2, 40, 77, 4, torch.bfloat16
    x = to_dev_like(make_x(B, D, L, dtype, channel_last, g), gpu_device)
    w, b = (t.to(gpu_device) for t in make_wb(D, W, True, g, w_dtype=dtype))
    dout = torch.randn(B, D, L, generator=g).to(dtype).to(gpu_device)               # channel-first, for both layouts of x
    init = make_states(B, D, W - 1, dtype, g).to(gpu_device) if extra == "states" else None
    seq = random_seq_idx(B, L, g).to(gpu_device) if extra == "seq_idx" else None
    kw = dict(seq_idx=seq, return_final_states=init is not None, activation="silu")

    def run(wanted=(True, True, True, True), final_only=False, through=None):
        leaves = [t.detach().requires_grad_(on) if t is not None else None for t, on in zip((x, w, None if extra == "no_bias" else b, init), wanted)]
        f = lambda *a: pkg.causal_conv1d_fn(a[0], a[1], a[2], initial_states=a[3], **kw)
        res = f(*leaves) if through is None else through(f, *leaves)
        outs = list(res) if isinstance(res, tuple) else [res]
        used = outs[1:] if final_only else outs[:1]
        given = [torch.ones_like(t) if final_only else dout for t in used]
        asked = [t for t in leaves if t is not None and t.requires_grad]
        grads = torch.autograd.grad(used, asked, given, retain_graph=True)
        again = torch.autograd.grad(used, asked, given)
        assert all(torch.equal(p, q) for p, q in zip(grads, again))
        return [o.detach() for o in outs] + list(grads)

    def everything():
        res = run() + run((True, False, False, False)) + run((False, True, False, False))
        res += run(through=lambda f, *a: checkpoint(f, *a, use_reentrant=False))
        if init is not None:
            res += run((False, False, False, True)) + run(final_only=True)
            res += run(final_only=True, through=lambda f, *a: checkpoint(f, *a, use_reentrant=False))
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            res += run()
        torch.cuda.current_stream().wait_stream(side)
        return res

    native, python = _both(monkeypatch, everything)
    assert len(native) == len(python)
    for n, p in zip(native, python):
        assert n.dtype == p.dtype and n.stride() == p.stride() and torch.equal(n, p)
