"""The decode step with one and with two batch rows a lane: batches at the edges of the rule that chooses (two
rows where they come to 449 .. 512 or 657 .. 768 workgroups of eight batch rows and 64 column groups each and at
most one row lies in front of the window), and batches that are no whole number of a workgroup's rows.  Outputs against the plain PyTorch step, the cache bit for bit."""
import pytest
import torch

from causal_conv1d.causal_conv1d_interface import causal_conv1d_update_ref
from helpers import assert_close, gen, make_wb

pytestmark = pytest.mark.gpu


# column blocks of 64 x 8 bytes, batch: workgroups with two rows a lane
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("ring", [False, True], ids=["shift", "ring"])
@pytest.mark.parametrize("blocks,batch", [(1, 1), (3, 5), (1, 3584), (1, 3585), (1, 4093), (1, 4096), (1, 4097), (7, 511), (7, 513), (8, 505)])
def test_step_rows(pkg, gpu_device, blocks, batch, ring, dtype):
    _check(pkg, gpu_device, blocks, batch, ring, dtype, 8 if ring else 3)


@pytest.mark.parametrize("ring", [False, True], ids=["shift", "ring"])
@pytest.mark.parametrize("blocks,batch,state_len", [(1, 5248, 3), (1, 5249, 4), (3, 1755, 5), (3, 2041, 4), (1, 6144, 3), (1, 6145, 3), (1, 3585, 4), (1, 4096, 5)])
def test_step_rows_in_front_of_the_window(pkg, gpu_device, blocks, batch, ring, state_len):
    _check(pkg, gpu_device, blocks, batch, ring, torch.bfloat16, state_len)


def _check(pkg, gpu_device, blocks, batch, ring, dtype, state_len):
    g = gen(10 * batch + blocks)
    D = blocks * 64 * (8 // torch.empty(0, dtype=dtype).element_size()) - 8      # the last block a partial one
    state = torch.randn(batch, state_len, D, generator=g).to(dtype).transpose(1, 2)
    x = torch.randn(batch, 1, D, generator=g).to(dtype).transpose(1, 2)
    w, b = make_wb(D, 4, True, g)
    lengths = torch.randint(0, 1000, (batch,), generator=g, dtype=torch.int32) if ring else None
    on_gpu = state.to(gpu_device)
    assert on_gpu.stride(1) == 1
    out = pkg.causal_conv1d_update(x.to(gpu_device), on_gpu, w.to(gpu_device), b.to(gpu_device), "silu",
                                   None if lengths is None else lengths.to(gpu_device))
    stepped = state.float()                            # the plain step moves bits unchanged, so fp32 holds the cache exactly
    ref = causal_conv1d_update_ref(x.float(), stepped, w, b, "silu", lengths)
    assert torch.equal(on_gpu.cpu(), stepped.to(dtype))
    assert_close(out, ref, dtype, "out")
