"""Channel-first backward of rows of at most 64 vectors anywhere in memory: every length around one and two
vectors and around the most a wavefront takes, odd starts, rows odd numbers of elements apart, one and
several rows to a wavefront and items to a workgroup, states.  Against the oracle; what lies between and
around the rows of dx keeps its value."""
import pytest
import torch

from helpers import TOL_W, assert_close, gen, make_states, make_wb
from oracle import causal_conv1d_oracle as orc

pytestmark = pytest.mark.gpu

LENGTHS = {torch.bfloat16: (1, 2, 7, 8, 9, 10, 11, 13, 15, 16, 17, 31, 100, 255, 257, 300, 500, 505, 511, 512),
           torch.float32: (1, 3, 4, 5, 6, 7, 8, 9, 63, 100, 129, 251, 253, 255, 256)}
CASES = [(dtype, L) for dtype, lengths in LENGTHS.items() for L in lengths]


@pytest.mark.parametrize("states", [False, True], ids=["plain", "states"])
@pytest.mark.parametrize("batch,dim,width", [(3, 40, 4), (24, 16, 3), (130, 8, 2)])
@pytest.mark.parametrize("dtype,seqlen", CASES, ids=["%s-%d" % (str(d)[6:], n) for d, n in CASES])
def test_rows_anywhere(pkg, gpu_device, dtype, seqlen, batch, dim, width, states):
    g = gen(1000 * width + seqlen)
    apart, start = seqlen + (3 if seqlen % 2 else 2), 5                # rows of x, dout and dx an odd number of elements apart

    def spread(value=None):
        buf = torch.full((start + batch * dim * apart,), 7.0, dtype=dtype, device=gpu_device)
        rows = buf.as_strided((batch, dim, seqlen), (dim * apart, apart, 1), start)
        if value is not None:
            rows.copy_(value)
        return buf, rows

    x, dout = (torch.randn(batch, dim, seqlen, generator=g).to(dtype) for _ in range(2))
    w, b = make_wb(dim, width, True, g)
    init = make_states(batch, dim, width - 1, dtype, g) if states else None
    dfin = make_states(batch, dim, width - 1, dtype, g) if states else None
    dinit = torch.empty(batch, width - 1, dim, dtype=dtype, device=gpu_device).transpose(1, 2) if states else None
    _, xg = spread(x)
    _, dg = spread(dout)
    buf, dx = spread()
    dw, db = torch.empty(dim, width, device=gpu_device), torch.empty(dim, device=gpu_device)
    gpu = lambda t: None if t is None else t.to(gpu_device)
    torch.ops.DaoAILab._causal_conv1d_bwd_overwrite_cpp(xg, gpu(w), gpu(b), dg, None, gpu(init), gpu(dfin), dx, dw, db, dinit, True)
    ref = orc.bwd(x, w, b, dout, initial_states=init, dfinal_states=dfin, activation="silu")
    assert_close(dx, ref[0], dtype, "dx")
    assert_close(dw, ref[1], what="dweight", tol=TOL_W)
    assert_close(db, ref[2], what="dbias", tol=TOL_W)
    if states:
        assert_close(dinit, ref[3], dtype, "dinitial_states")
    dx.fill_(7.0)
    assert bool((buf == 7.0).all())


@pytest.mark.parametrize("dense", [True, False], ids=["contiguous", "apart"])
@pytest.mark.parametrize("states", [False, True], ids=["plain", "states"])
@pytest.mark.parametrize("batch,dim,width,silu", [(3, 40, 4, True), (24, 16, 3, False), (2, 1032, 2, True)])
@pytest.mark.parametrize("dtype,seqlen", CASES, ids=["%s-%d" % (str(d)[6:], n) for d, n in CASES])
def test_forward_of_rows_anywhere(pkg, gpu_device, dtype, seqlen, batch, dim, width, silu, states, dense):
    """The forward of the same rows, one buffer for initial and final states."""
    g = gen(2000 * width + seqlen)
    apart, start = (seqlen, 0) if dense else (seqlen + (3 if seqlen % 2 else 2), 5)

    def spread():
        buf = torch.full((start + batch * dim * apart + 8,), 7.0, dtype=dtype, device=gpu_device)
        return buf, buf.as_strided((batch, dim, seqlen), (dim * apart, apart, 1), start)

    x = torch.randn(batch, dim, seqlen, generator=g).to(dtype)
    w, b = make_wb(dim, width, True, g)
    init = make_states(batch, dim, width - 1, dtype, g) if states else None
    _, xg = spread()
    xg.copy_(x)
    buf, out = spread()
    held = init.to(gpu_device) if states else None
    torch.ops.DaoAILab._causal_conv1d_fwd_cpp(xg, w.to(gpu_device), b.to(gpu_device), None, held, out, held, silu)
    ref = orc.fwd(x, w, b, initial_states=init, return_final_states=states, activation="silu" if silu else None)
    ref, fin = ref if states else (ref, None)
    assert_close(out, ref, dtype, "out")
    if states:
        assert torch.equal(held.cpu(), fin)
    out.fill_(7.0)
    assert bool((buf == 7.0).all())
