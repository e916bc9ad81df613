"""The channel-last forward at the edges of the rule that chooses its rows per run (8 up to 1600 wavefronts of
16 rows and from 2049 to 2500, 16 otherwise; 8 up to 1536 where the taps are not packed): the same bits as with 16
rows forced, and the oracle's values, with rows that are no whole number of runs, a partial last column block, states
and packed sequences."""
import pytest
import torch

import cabi
from helpers import assert_close, gen, make_states, make_wb, random_seq_idx
from oracle import causal_conv1d_oracle as orc

pytestmark = pytest.mark.gpu


# wavefronts = batch * ceil(seqlen / 16) * column blocks of 256 bytes
@pytest.mark.parametrize("extra", ["none", "states", "seq_idx"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("batch,seqlen,blocks", [(1, 16 * 1600, 1), (1, 16 * 1600 + 3, 1), (1, 16 * 2048 - 9, 1), (3, 16 * 683 - 5, 1),
                                                 (25, 16 * 20 - 7, 5), (41, 16 * 61 - 1, 1), (50, 43, 17)])
def test_rows_per_run(pkg, gpu_device, cc1d_lib, batch, seqlen, blocks, dtype, extra):
    _check(pkg, gpu_device, cc1d_lib, batch, seqlen, blocks, dtype, extra)


@pytest.mark.parametrize("taps", ["strided", "other type"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("batch,seqlen,blocks", [(1, 16 * 1536, 1), (1, 16 * 1536 + 3, 1), (3, 16 * 683 - 5, 1), (50, 43, 17)])
def test_rows_per_run_of_other_taps(pkg, gpu_device, cc1d_lib, batch, seqlen, blocks, dtype, taps):
    _check(pkg, gpu_device, cc1d_lib, batch, seqlen, blocks, dtype, "none", taps)


def _check(pkg, gpu_device, cc1d_lib, batch, seqlen, blocks, dtype, extra, taps="packed"):
    lib = cabi.declare(cc1d_lib)
    g = gen(seqlen + batch)
    dim = blocks * (128 if dtype == torch.bfloat16 else 64) - (8 if batch > 1 else 0)
    x = torch.randn(batch, seqlen, dim, generator=g).to(dtype).transpose(1, 2)
    w, b = make_wb(dim, 4, True, g)
    init = make_states(batch, dim, 3, dtype, g) if extra == "states" else None
    seq = random_seq_idx(batch, seqlen, g) if extra == "seq_idx" else None
    gpu = lambda t: None if t is None else t.to(gpu_device)
    if taps == "other type":
        w, b = w.to(torch.float16), b.to(torch.float16)
    w_gpu = torch.stack([w, w], 2).to(gpu_device)[..., 0] if taps == "strided" else gpu(w)
    on_gpu = x.transpose(1, 2).contiguous().to(gpu_device).transpose(1, 2)

    def run(rows):
        assert lib.cc1d_set_tunable(b"fwd_cl_rows", rows) == 0
        try:
            res = pkg.causal_conv1d_fn(on_gpu, w_gpu, gpu(b), gpu(seq), gpu(init), init is not None, activation="silu")
        finally:
            lib.cc1d_set_tunable(b"fwd_cl_rows", 0)
        return res if isinstance(res, tuple) else (res,)

    chosen, sixteen = run(0), run(16)
    assert all(torch.equal(p, q) for p, q in zip(chosen, sixteen))
    w, b = w.float(), b.float()                        # the oracle works in the taps' type, the kernel in fp32
    ref = (orc.fwd_seq_idx(x, w, b, seq, activation="silu") if seq is not None
           else orc.fwd(x, w, b, initial_states=init, return_final_states=init is not None, activation="silu"))
    ref = ref if isinstance(ref, tuple) else (ref,)
    assert_close(chosen[0], ref[0], dtype, "out")
    if init is not None:
        assert torch.equal(chosen[1].cpu(), ref[1])
