"""The functions' direct way to the dispatcher (`_update_call`, `_forward_call`, `_backward_call` of the
extension module): what it must leave to the generic path, and that both see and give the same."""
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from helpers import DTYPES, gen, make_states, make_wb, make_x, random_seq_idx, to_dev_like


class _Subclass(torch.Tensor):
    pass


class _Functions(TorchFunctionMode):
    def __torch_function__(self, func, types, args=(), kwargs=None):
        return func(*args, **(kwargs or {}))


class _Ops(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.names = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        self.names.append(func._schema.name)
        return func(*args, **(kwargs or {}))


def _update_args():
    return [torch.zeros(2, 8), torch.zeros(2, 8, 4), torch.zeros(8, 4), torch.zeros(8), True, None, None]


def test_left_to_the_generic_path(pkg):
    import causal_conv1d_cuda as ext
    for i in (0, 1, 2, 3):
        a = _update_args()
        a[i] = a[i].as_subclass(_Subclass)
        assert ext._update_call(*a) is NotImplemented
        a[i] = 5
        assert ext._update_call(*a) is NotImplemented
    assert ext._update_call(*_update_args()[:-1]) is NotImplemented
    with _Functions():
        assert ext._update_call(*_update_args()) is NotImplemented
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        ext._update_call(*_update_args())
    x, w = torch.zeros(2, 8, 9), torch.zeros(8, 4)
    forward = lambda x=x, bias=None, seq=None, init=None, final=False, out=None: ext._forward_call(x, w, bias, seq, init, final, out, True)
    wide = torch.zeros(2, 16, 18)[:, ::2, ::2]
    assert forward(x=wide) is NotImplemented                        # neither stride is 1: needs a copy
    assert forward(bias=torch.zeros(16)[::2]) is NotImplemented
    assert forward(seq=torch.zeros(2, 18, dtype=torch.int32)[:, ::2]) is NotImplemented
    assert forward(init=torch.zeros(2, 16, 6)[:, ::2, ::2]) is NotImplemented
    assert forward(seq=torch.zeros(2, 9, dtype=torch.int32), final=True) is NotImplemented   # refused by the layer above
    assert forward(final=True, out=torch.zeros(2, 16, 6)[:, ::2, ::2]) is NotImplemented
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        forward()
    assert pkg.causal_conv1d_fn(x.to("meta"), w.to("meta")).shape == x.shape


def _backward_args():
    return [torch.zeros(2, 8, 9), torch.zeros(8, 4), torch.zeros(8), torch.zeros(2, 8, 9), torch.zeros(2, 9, dtype=torch.int32),
            torch.zeros(2, 8, 3), torch.zeros(2, 8, 3), True, True]


def test_backward_left_to_the_generic_path(pkg):
    import causal_conv1d_cuda as ext
    for i in range(9):
        a = _backward_args()
        if i < 7:
            a[i] = a[i].as_subclass(_Subclass)
            assert ext._backward_call(*a) is NotImplemented
        for other in ((5,) if i in (2, 4, 5, 6) else (5, None)):
            a[i] = other
            assert ext._backward_call(*a) is NotImplemented
    assert ext._backward_call(*_backward_args()[:-1]) is NotImplemented
    for i, t in ((0, torch.zeros(8, 9)), (1, torch.zeros(8, 1, 4)), (3, torch.zeros(2, 16, 18)[:, ::2, ::2])):
        a = _backward_args()
        a[i] = t                                                    # x not (batch, dim, seqlen), weight not (dim, width), dout needs a copy
        assert ext._backward_call(*a) is NotImplemented
    with _Functions():
        assert ext._backward_call(*_backward_args()) is NotImplemented
    with pytest.raises(RuntimeError, match="must be on the GPU"):
        ext._backward_call(*_backward_args())


@pytest.mark.filterwarnings("ignore:.*torch.jit.trace")
def test_tracing_sees_the_ops(pkg):
    """On meta tensors: the direct calls step aside while torch.jit.trace records."""
    import causal_conv1d_cuda as ext
    answers = []

    def step(x, st):
        answers.append(ext._update_call(x, st, w, None, True, None, None))
        answers.append(ext._forward_call(st, w, None, None, None, False, None, True))
        answers.append(ext._backward_call(st, w, None, st, None, None, None, False, True))
        return pkg.causal_conv1d_update(x, st, w)

    w = torch.zeros(8, 4, device="meta")
    traced = torch.jit.trace(step, (torch.zeros(2, 8, device="meta"), torch.zeros(2, 8, 4, device="meta")), check_trace=False)
    assert len(answers) == 3 and all(a is NotImplemented for a in answers)
    assert "DaoAILab::_causal_conv1d_update_out_cpp" in str(traced.graph)


def test_vmap_is_refused_by_both_ways(pkg, monkeypatch):
    """The ops have no batching rule; the direct calls reach the dispatcher with the same batched tensors."""
    from causal_conv1d import causal_conv1d_interface as interface
    x, w, st = torch.zeros(3, 2, 8, device="meta"), torch.zeros(8, 4, device="meta"), torch.zeros(3, 2, 8, 4, device="meta")
    for _ in range(2):
        with pytest.raises(RuntimeError, match="Batching rule not implemented for DaoAILab::_causal_conv1d_update_out_cpp"):
            torch.vmap(lambda q, s: pkg.causal_conv1d_update(q, s, w))(x, st)
        with pytest.raises(RuntimeError, match="Batching rule not implemented for DaoAILab::_causal_conv1d_fwd_out_cpp"):
            torch.vmap(lambda q: pkg.causal_conv1d_fn(q, w))(st)
        monkeypatch.setattr(interface, "_direct_update", lambda *a: NotImplemented)
        monkeypatch.setattr(interface, "_direct_forward", lambda *a: NotImplemented)


def test_dispatch_modes_see_the_ops(pkg):
    """On meta tensors, without a GPU."""
    x, w, st = torch.zeros(2, 8, device="meta"), torch.zeros(8, 4, device="meta"), torch.zeros(2, 8, 4, device="meta")
    with _Ops() as ops:
        pkg.causal_conv1d_update(x, st, w)
        pkg.causal_conv1d_fn(torch.zeros(2, 8, 9, device="meta"), w, return_final_states=True)
    assert "DaoAILab::_causal_conv1d_update_out_cpp" in ops.names and "DaoAILab::_causal_conv1d_fwd_out_cpp" in ops.names


@pytest.mark.gpu
@pytest.mark.parametrize("wide_weights", [False, True], ids=["w16", "w32"])
@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("channel_last", [False, True], ids=["cf", "cl"])
@pytest.mark.parametrize("extra", ["none", "states", "seq_idx", "no_bias"])
def test_both_paths_give_the_same(pkg, gpu_device, monkeypatch, channel_last, dtype, extra, wide_weights):
    if extra == "seq_idx" and not channel_last:
        pytest.skip("seq_idx needs channel-last x")
    from causal_conv1d import causal_conv1d_interface as interface, cpp_functions
    answers = {}

    def watched(module, name):
        call = getattr(module, name)

        def wrapper(*args):
            res = call(*args)
            answers.setdefault(name, []).append(res is not NotImplemented)
            return res
        monkeypatch.setattr(module, name, wrapper)

    watched(interface, "_direct_forward")
    watched(interface, "_direct_update")
    watched(cpp_functions, "_direct_backward")
    g = gen(31)
    B, D, L, W = 2, 40, 77, 4
    wtype = torch.float32 if wide_weights else dtype
    x = to_dev_like(make_x(B, D, L, dtype, channel_last, g), gpu_device)
    w, b = (t.to(gpu_device) for t in make_wb(D, W, True, g, w_dtype=wtype))
    dout = to_dev_like(make_x(B, D, L, dtype, channel_last, g, sliced=False), gpu_device)
    init = make_states(B, D, W - 1, dtype, g).to(gpu_device) if extra == "states" else None
    seq = random_seq_idx(B, L, g).to(gpu_device) if extra == "seq_idx" else None
    state = torch.randn(B, W, D, generator=g).to(dtype).to(gpu_device).transpose(1, 2)
    bias = None if extra == "no_bias" else b

    def everything():
        leaves = [t.detach().requires_grad_() for t in (x, w, bias, init) if t is not None]
        it = iter(leaves)
        x_, w_ = next(it), next(it)
        b_ = None if bias is None else next(it)
        i_ = None if init is None else next(it)
        res = pkg.causal_conv1d_fn(x_, w_, b_, seq_idx=seq, initial_states=i_, return_final_states=init is not None, activation="silu")
        outs = list(res) if isinstance(res, tuple) else [res]
        grads = torch.autograd.grad(outs[0], leaves, dout)
        with torch.no_grad():
            quiet = pkg.causal_conv1d_fn(x, w, bias, seq_idx=seq, initial_states=init, return_final_states=init is not None)
        st = state.clone()
        step = pkg.causal_conv1d_update(x[..., 0].contiguous(), st, w, bias, "silu")
        return outs + list(grads) + (list(quiet) if isinstance(quiet, tuple) else [quiet]) + [st, step]

    direct = everything()
    calls = {"_direct_forward": 2, "_direct_backward": 1, "_direct_update": 1}
    assert answers == {name: [True] * n for name, n in calls.items()}
    answers.clear()
    # torch.autograd.grad is a function that modes see: its body, the backward included, runs outside of the mode.
    monkeypatch.setattr(cpp_functions, "_direct_backward", lambda *a: answers.setdefault("_direct_backward", []).append(False) or NotImplemented)
    with _Functions():                                              # every call takes torch.ops
        generic = everything()
    assert answers == {name: [False] * n for name, n in calls.items()}
    assert len(direct) == len(generic)
    for d, r in zip(direct, generic):
        assert d.dtype == r.dtype and d.stride() == r.stride() and torch.equal(d, r)
