"""Channel-first forward of contiguous short rows that are no whole number of vectors: the flat array and the
short rows' lanes, whichever the launcher takes, give the same bits as rows spread apart (which only the
short-row kernel takes), on both sides of the lines between the two; nothing around the tensor is touched."""
import pytest
import torch

from helpers import assert_close, gen, make_states, make_wb
from oracle import causal_conv1d_oracle as orc

pytestmark = pytest.mark.gpu

BF16, FP16, FP32 = torch.bfloat16, torch.float16, torch.float32
# dtype, batch, dim, seqlen, width, silu: small launches of either kernel, one round of wavefronts and more (8192: 512 x 512 rows
# of two lanes), the shares of used lanes around the lines (9 and 13 of 16 positions, 43 and 47 of 64), long last vectors and short
# ones, rows that end in a wavefront's first and last lane, one row, one channel
CASES = [(BF16, 3, 40, 9, 2, True), (BF16, 3, 40, 15, 2, False), (FP16, 5, 33, 511, 2, True), (BF16, 64, 40, 23, 4, False),
         (FP16, 513, 512, 9, 4, True), (BF16, 600, 520, 13, 4, True), (BF16, 160, 520, 43, 4, True), (FP16, 160, 520, 47, 3, True),
         (BF16, 1200, 300, 10, 4, True), (BF16, 1, 1, 509, 2, True), (FP32, 3, 40, 5, 3, True), (FP32, 1, 70, 255, 4, False),
         (FP32, 300, 520, 9, 4, True), (FP32, 300, 520, 13, 4, True), (FP32, 70, 520, 33, 4, True), (FP32, 70, 130, 129, 2, True),
         (FP32, 129, 1, 63, 3, False)]


@pytest.mark.parametrize("states", ["none", "init", "final"])
@pytest.mark.parametrize("w_in_type", [False, True], ids=["w32", "wx"])
@pytest.mark.parametrize("dtype,batch,dim,seqlen,width,silu", CASES, ids=["-".join(str(v)[6:] if i == 0 else str(v) for i, v in enumerate(c)) for c in CASES])
def test_contiguous_rows_as_rows_apart(pkg, gpu_device, dtype, batch, dim, seqlen, width, silu, w_in_type, states):
    g = gen(31 * seqlen + width)
    x = torch.randn(batch, dim, seqlen, generator=g).to(dtype)
    w, b = make_wb(dim, width, True, g, w_dtype=dtype if w_in_type else FP32)
    init = make_states(batch, dim, width - 1, dtype, g) if states == "init" else None

    def run(apart):
        n = batch * dim * apart
        buf = torch.full((n + 64,), 7.0, dtype=dtype, device=gpu_device)
        out = buf[32:32 + n].view(batch, dim, apart)[..., :seqlen]
        rows = torch.full((batch, dim, apart), float("nan"), dtype=dtype, device=gpu_device)[..., :seqlen]
        rows.copy_(x)
        fin = torch.empty(batch, width - 1, dim, dtype=dtype, device=gpu_device).transpose(1, 2) if states == "final" else None
        torch.ops.DaoAILab._causal_conv1d_fwd_cpp(rows, w.to(gpu_device), b.to(gpu_device), None,
                                                  None if init is None else init.to(gpu_device), out, fin, silu)
        res = out.clone(), fin
        out.fill_(7.0)
        assert bool((buf == 7.0).all())
        return res

    dense, spread = run(seqlen), run(seqlen + 1)
    assert torch.equal(dense[0], spread[0])
    if states == "final":
        assert torch.equal(dense[1], spread[1])
    if batch * dim * seqlen < 200000:
        ref = orc.fwd(x, w, b, initial_states=init, activation="silu" if silu else None)
        assert_close(dense[0], ref, dtype, "out")
