"""The channel-last backward in fp16 with seq_idx, width 4 and SiLU, which names its rows through buffer
resources in launches of more than 1024 wavefronts and through pointers in others, at the edges of its
runs of 32 rows and workgroups of four runs: against the oracle, and against the 8-byte lanes, which
always use pointers.  dx must be the same bit for bit."""
import pytest
import torch

from helpers import TOL_W, assert_close, gen, make_wb, random_seq_idx
from oracle import causal_conv1d_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("wtype", [torch.float32, torch.float16], ids=["fp32", "fp16"])
@pytest.mark.parametrize("sliced", [False, True], ids=["dense", "sliced"])
@pytest.mark.parametrize("resources", [False, True], ids=["pointers", "resources"])
@pytest.mark.parametrize("seqlen", [1, 2, 3, 4, 31, 32, 33, 35, 127, 128, 129, 300])
def test_rows_through_resources(pkg, gpu_device, cc1d_lib, seqlen, resources, sliced, wtype):
    g = gen(4000 + seqlen)
    D = 136                                            # two wavefronts to a row
    B = 1024 // (2 * ((seqlen + 31) // 32)) + 1 if resources else 3
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


@pytest.mark.parametrize("row_bytes", [53687088, 53687104], ids=["last-32-row-stride", "16-row-runs"])
def test_rows_far_apart(pkg, gpu_device, row_bytes):
    """40 rows of 53687088 bytes end 128 bytes short of 2^31, the largest stride that keeps runs of 32
    rows; one step more halves them.  Batch entries side by side inside a row, more than 1024 wavefronts:
    the resources' offsets reach 37 rows.  The same values packed must give the same gradients."""
    g = gen(4999)
    B, D, L = 260, 136, 35

    def packed():
        return torch.randn(B, L, D, generator=g).to(torch.float16).to(gpu_device).transpose(1, 2)

    def spread(t=None):
        buf = torch.empty(L * row_bytes // 2, dtype=torch.float16, device=gpu_device)
        far = buf.as_strided((B, D, L), (D, 1, row_bytes // 2))
        return far if t is None else far.copy_(t)

    x, dout = packed(), packed()
    seq = random_seq_idx(B, L, g, pad=True).to(gpu_device)
    w, b = (t.to(gpu_device) for t in make_wb(D, 4, True, g))

    def run(x, dout, dx):
        dw, db = torch.zeros(D, 4, device=gpu_device), torch.zeros(D, device=gpu_device)
        torch.ops.DaoAILab._causal_conv1d_bwd_cpp(x, w, b, dout, seq, None, None, dx, dw, db, None, True)
        return dx, dw, db

    near = run(x, dout, torch.empty_like(x))
    far = run(spread(x), spread(dout), spread())
    assert torch.equal(near[0], far[0])
    if row_bytes == 53687088:
        assert torch.equal(near[1], far[1]) and torch.equal(near[2], far[2])
    else:                                              # other runs, other order of the sums
        assert_close(far[1], near[1].cpu(), what="dweight", tol=TOL_W)
        assert_close(far[2], near[2].cpu(), what="dbias", tol=TOL_W)
