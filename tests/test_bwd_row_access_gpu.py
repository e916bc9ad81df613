"""The channel-last backward in fp16 with seq_idx and width 4, which names its rows through buffer
resources, at the edges of its runs of 32 rows and workgroups of four runs: against the oracle, and
against the 8-byte lanes, which use pointers.  dx must be the same bit for bit."""
import pytest
import torch

from helpers import TOL_W, assert_close, gen, make_wb, random_seq_idx
from oracle import causal_conv1d_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [torch.float32, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("sliced", [False, True], ids=["dense", "sliced"])
@pytest.mark.parametrize("seqlen", [1, 2, 3, 4, 31, 32, 33, 35, 127, 128, 129, 300])
def test_rows_through_resources(pkg, gpu_device, cc1d_lib, seqlen, sliced, wtype):
    g = gen(4000 + seqlen)
    B, D = 3, 136
    wide, lo = (D + 24, 8) if sliced else (D, 0)

    def tensor():
        return torch.randn(B, seqlen, wide, generator=g).to(torch.float16)

    x, dout = tensor()[..., lo:lo + D].transpose(1, 2), tensor()[..., :D].transpose(1, 2)
    seq = random_seq_idx(B, seqlen, g, pad=seqlen > 8)
    w, b = make_wb(D, 4, True, g, w_dtype=wtype)
    big_x, big_d = torch.zeros(B, seqlen, wide, dtype=x.dtype, device=gpu_device), torch.zeros(B, seqlen, wide, dtype=x.dtype, device=gpu_device)
    xd, dd = big_x[..., lo:lo + D].transpose(1, 2), big_d[..., :D].transpose(1, 2)
    xd.copy_(x)
    dd.copy_(dout)

    def run(lane_bytes):
        big_dx = torch.full((B, seqlen, wide), 7.0, dtype=x.dtype, device=gpu_device)
        dx = big_dx[..., lo:lo + D].transpose(1, 2)
        dw, db = torch.zeros(D, 4, device=gpu_device), torch.zeros(D, device=gpu_device)
        assert cc1d_lib.cc1d_set_tunable(b"bwd_cl_lane_bytes", lane_bytes) == 0
        try:
            torch.ops.DaoAILab._causal_conv1d_bwd_cpp(xd, w.to(gpu_device), b.to(gpu_device), dd, seq.to(gpu_device), None, None,
                                                      dx, dw, db, None, True)
        finally:
            cc1d_lib.cc1d_set_tunable(b"bwd_cl_lane_bytes", 0)
        assert bool((big_dx[..., :lo] == 7.0).all()) and bool((big_dx[..., lo + D:] == 7.0).all())
        return dx, dw, db

    narrow, wide_lanes = run(4), run(8)
    assert torch.equal(narrow[0], wide_lanes[0])
    rdx, rdw, rdb, _ = orc.bwd(x, w.float(), b.float(), dout, seq_idx=seq, activation="silu")
    assert_close(narrow[0], rdx, torch.float16, "dx")
    for got in (narrow, wide_lanes):
        assert_close(got[1], rdw, what="dweight", tol=TOL_W)
        assert_close(got[2], rdb, what="dbias", tol=TOL_W)
