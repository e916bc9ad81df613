"""dweight and dbias stored in the parameters' own 16-bit type by the kernel that finishes the sums: the
same bits as the fp32 sums rounded afterwards, whichever kernel that is, with and without a bias, with
a bias in the middle of a buffer, for launches cut into slices of the batch and for empty ones."""
import pytest
import torch

from helpers import gen, make_wb

pytestmark = pytest.mark.gpu

# (channel_last, (batch, dim, seqlen), knobs): the kernel that stores
SHAPES = {
    "second stage, channel-last": (True, (2, 136, 300), {}),
    "second stage, channel-last 8-byte lanes": (True, (2, 136, 300), {"bwd_cl_lane_bytes": 8}),
    "tiles of a channel": (False, (1, 72, 1537), {}),
    "second stage, tiles": (False, (2, 72, 1537), {"bwd_cf_direct": -1}),
    "short rows, one workgroup a channel": (False, (24, 72, 130), {}),
    "short rows, one wavefront a channel": (False, (2, 72, 20), {}),
    "second stage, short rows": (False, (24, 72, 130), {"bwd_cf_direct": -1}),
    "walking": (False, (2, 72, 1537), {"bwd_cf_parts": -1}),
    "batch slices": (True, (40, 136, 96), {"launch_limit_shift": 18}),
    "one row": (True, (1, 8, 1), {}),
    "no batch": (False, (0, 72, 40), {}),
}


@pytest.mark.parametrize("bias", [True, False], ids=["bias", "no_bias"])
@pytest.mark.parametrize("wtype", [torch.float16, torch.bfloat16], ids=lambda d: str(d)[6:])
@pytest.mark.parametrize("width", [2, 4])
@pytest.mark.parametrize("name", SHAPES)
def test_sums_in_the_type_of_weight(pkg, gpu_device, cc1d_lib, name, width, wtype, bias):
    channel_last, (B, D, L), knobs = SHAPES[name]
    g = gen(len(name) + width)

    def rows():
        t = torch.randn(B, L, D, generator=g).to(torch.bfloat16)
        return (t.transpose(1, 2) if channel_last else t.transpose(1, 2).contiguous()).to(gpu_device)

    x, dout = rows(), rows()
    w, b = (t.to(wtype).to(gpu_device) for t in make_wb(D, width, True, g))
    op = torch.ops.DaoAILab._causal_conv1d_bwd_overwrite_cpp

    def run(dtype):
        dx = torch.empty_like(x)
        sums = torch.full((D * (width + 1) + 3,), float("nan"), dtype=dtype, device=gpu_device)
        dw, db = sums[1:1 + D * width].view(D, width), sums[2 + D * width:2 + D * (width + 1)]
        op(x, w, b if bias else None, dout, None, None, None, dx, dw, db if bias else None, None, True)
        return dx, dw, db, sums

    try:
        for knob, value in knobs.items():
            assert cc1d_lib.cc1d_set_tunable(knob.encode(), value) == 0
        wide, narrow = run(torch.float32), run(wtype)
    finally:
        for knob in knobs:
            cc1d_lib.cc1d_set_tunable(knob.encode(), 0)
    assert torch.equal(wide[0], narrow[0])
    assert narrow[1].isfinite().all() and torch.equal(wide[1].to(wtype), narrow[1])
    if bias:
        assert torch.equal(wide[2].to(wtype), narrow[2])
    untouched = [0, 1 + D * width, -1] if bias else [0] + list(range(1 + D * width, narrow[3].numel()))
    assert narrow[3][untouched].isnan().all()
