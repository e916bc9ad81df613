"""Decode steps on ring buffers and slots at the edges of the position arithmetic: rings whose length is a
power of two (a mask in the kernels of a few tokens) and others (a division), no longer than the window and longer,
positions that wrap inside the window, are negative or near the end of int32, a batch that is no whole number of
a workgroup's rows, padding slots.  Outputs against the plain PyTorch step, the cache bit for bit."""
import pytest
import torch

from causal_conv1d.causal_conv1d_interface import causal_conv1d_update_ref
from helpers import assert_close, gen, make_wb

pytestmark = pytest.mark.gpu


RINGS = [(2, 1), (2, 2), (3, 2), (3, 5), (4, 3), (4, 4), (4, 7), (4, 8), (4, 16)]


@pytest.mark.parametrize("slots", [False, True], ids=["rows", "slots"])
@pytest.mark.parametrize("width,state_len,tokens", [r + (1,) for r in RINGS] + [r + (3,) for r in RINGS if r[1] >= 3])
def test_ring_positions(pkg, gpu_device, width, state_len, slots, tokens):
    _check(pkg, gpu_device, width, state_len, slots, tokens, 264)   # two column blocks, the second a partial one


# dim 264: vectors along dim, more tokens than the kernels of a few take; dim 33: elements
@pytest.mark.parametrize("slots", [False, True], ids=["rows", "slots"])
@pytest.mark.parametrize("width,state_len,tokens,dim", [r + (1, 33) for r in RINGS] + [(4, 7, 3, 33), (2, 9, 9, 264), (3, 13, 9, 264), (4, 16, 9, 264), (4, 16, 16, 264)])
def test_ring_positions_general(pkg, gpu_device, width, state_len, slots, tokens, dim):
    """The same in the kernels for many tokens and for any strides, where every lane has a position of its own."""
    _check(pkg, gpu_device, width, state_len, slots, tokens, dim)


def _check(pkg, gpu_device, width, state_len, slots, tokens, D):
    g = gen(100 * width + 10 * state_len + tokens)
    B = 11
    rows = 2 * B if slots else B
    state = torch.randn(rows, state_len, D, generator=g).to(torch.bfloat16).transpose(1, 2)
    x = torch.randn(B, tokens, D, generator=g).to(torch.bfloat16).transpose(1, 2)
    w, b = make_wb(D, width, True, g)
    lengths = torch.tensor([0, 1, 2, 3, 7, 8, 1000, 2**31 - 9, -1, -2, -13], dtype=torch.int32)
    index = torch.randperm(rows, generator=g)[:B].to(torch.int32) if slots else None
    if slots:
        index[[2, 9]] = -1
    on_gpu = state.to(gpu_device)
    assert on_gpu.stride(1) == 1
    out = pkg.causal_conv1d_update(x.to(gpu_device), on_gpu, w.to(gpu_device), b.to(gpu_device), "silu",
                                   lengths.to(gpu_device), None if index is None else index.to(gpu_device))
    live = torch.ones(B, dtype=torch.bool) if index is None else index >= 0
    at = torch.arange(B) if index is None else index.long()
    # the plain step on the live rows; it moves bits unchanged, so fp32 holds the cache exactly
    stepped = state[at[live]].float()
    ref = causal_conv1d_update_ref(x[live].float(), stepped, w, b, "silu", lengths[live])
    want = state.clone()
    want[at[live]] = stepped.to(torch.bfloat16)
    assert torch.equal(on_gpu.cpu(), want)
    assert_close(out[live.to(gpu_device)], ref, torch.bfloat16, "out")
    assert not out[~live.to(gpu_device)].any()
