"""dweight / dbias of the channel-first kernels at the edges of the rules that pick who adds up a
channel's tiles: the kernel's own workgroup (`own`) or the second launch (`second`; `bwd_cf_direct` = -1
forces it).  Which of the two ran shows in the workspace, which only the second launch's first stage writes.  dx and
dinitial_states must not depend on it; dweight and dbias are the same fp32 terms added in another order.  Taps of
every type, packed and strided."""
import ctypes

import pytest
import torch

from oracle import causal_conv1d_oracle as orc
import cabi
from helpers import TOL_W, assert_close, gen, make_states

pytestmark = pytest.mark.gpu

BF16, FP16, FP32 = torch.bfloat16, torch.float16, torch.float32
CASES = [   # batch, dim, seqlen, width, dtype, weight dtype, strided weight, (dim, batch, seqlen) in memory, who adds
    (1, 24, 513, 4, BF16, FP32, False, False, "own"),        # one tile of one step and a tail
    (2, 24, 2049, 4, FP16, FP16, False, False, "own"),       # two tiles, the second a tail only
    (1, 17, 601, 4, BF16, BF16, False, False, "own"),        # channels by twos, the last one alone; rows off the dword grid
    (2, 263, 1001, 4, FP16, FP32, False, False, "own"),
    (2, 16, 12000, 3, BF16, BF16, True, False, "second"),    # 12 tiles of four steps, few channels
    (12, 95, 1001, 4, BF16, FP32, False, False, "own"),      # 12 of two steps
    (9, 95, 1100, 4, BF16, FP32, False, False, "second"),    # 9 of three
    (9, 96, 1100, 4, BF16, FP32, False, False, "own"),
    (9, 256, 600, 4, BF16, FP16, False, False, "own"),       # as many channels as CUs
    (9, 257, 600, 4, BF16, FP16, False, False, "second"),
    (14, 96, 1990, 4, BF16, BF16, False, False, "own"),      # 14 of four steps: 61,656 bytes of LDS
    (15, 96, 1990, 4, BF16, FP32, False, False, "second"),   # 15 of them: more than 64 KiB
    (16, 96, 1001, 2, BF16, FP32, True, False, "own"),       # 16 wavefronts
    (16, 96, 505, 4, FP32, FP32, False, False, "own"),
    (16, 96, 1001, 2, FP32, FP32, True, False, "second"),    # 16 of four steps: more than 64 KiB
    (17, 96, 600, 4, BF16, FP16, False, False, "second"),    # 17
    (8, 1024, 520, 4, BF16, FP32, False, False, "own"),      # 8192 wavefronts
    (8, 1032, 520, 4, BF16, FP32, False, False, "second"),   # 8256
    (8, 1032, 520, 4, BF16, FP32, False, True, "own"),       # a channel's rows adjacent
    (2, 4200, 520, 4, BF16, FP32, False, False, "own"),      # two places, one tile to a row: 8400 wavefronts
    (2, 1366, 4200, 4, BF16, FP32, False, False, "second"),  # three tiles to a row: 8196
    # short rows; parts of a channel x items of a part
    (1, 24, 512, 4, BF16, FP32, False, False, "one part"),
    (2, 24, 512, 4, BF16, BF16, False, False, "own"),        # 2 x 1
    (16, 24, 512, 4, FP16, FP16, False, False, "own"),       # 16 x 1
    (17, 24, 256, 4, FP32, FP32, False, False, "second"),    # 17 x 1
    (256, 256, 64, 4, FP32, FP32, False, False, "own"),      # 16 x 4, as many channels as CUs
    (260, 256, 64, 4, FP32, FP32, False, False, "second"),   # 13 x 5
    (48, 257, 64, 4, FP32, BF16, True, False, "own"),        # 12 x 1, more channels
    (52, 257, 64, 4, FP32, FP32, False, False, "second"),    # 13 x 1
    (72, 700, 64, 3, FP32, FP32, False, False, "own"),       # 6 x 3
    (76, 700, 64, 3, FP32, FP32, False, False, "second"),    # 5 x 4
    (48, 800, 64, 4, FP32, FP32, False, False, "own"),       # 6 x 2
    (52, 800, 64, 4, FP32, FP32, False, False, "second"),    # 5 x 3
    (96, 2048, 32, 2, FP32, FP32, False, False, "own"),      # 2 x 6, rows of a cache line each
    (104, 2048, 32, 2, FP32, FP32, False, False, "second"),  # 2 x 7
    (32, 2048, 40, 4, BF16, FP32, False, False, "own"),      # 2 x 2, rows that share cache lines
    (40, 2048, 40, 4, BF16, FP32, False, False, "second"),   # 2 x 3
    (32, 2056, 40, 4, BF16, FP32, False, False, "second"),   # 2 x 2, 8 x 256 channels and more
    (80, 24, 32, 4, BF16, FP32, False, False, "own"),        # 5 x 1, rows of 64 bytes
    (80, 24, 31, 4, BF16, FP32, False, False, "second"),     # 62 bytes
    (64, 24, 31, 4, BF16, FP32, False, False, "own"),        # 4 x 1
    (65, 256, 8, 3, BF16, BF16, False, False, "own"),        # 2 x 1
    (320, 1024, 8, 3, BF16, BF16, False, False, "second"),   # 3 x 2
    (65, 768, 8, 3, BF16, BF16, False, False, "own"),        # 2 x 1
    (65, 776, 8, 3, BF16, BF16, False, False, "second"),
    (12, 24, 505, 3, FP16, FP32, True, False, "own"),        # 16-bit rows off the vector grid: 12 x 1, few channels
    (16, 24, 505, 3, FP16, FP32, True, False, "second"),     # 16 x 1
    (16, 128, 505, 3, FP16, FP32, True, False, "own"),
    (64, 512, 61, 4, BF16, FP32, False, False, "own"),       # 8 x 1
    (64, 513, 61, 4, BF16, FP32, False, False, "second"),
    (32, 513, 61, 4, BF16, FP32, False, False, "own"),       # 4 x 1
    (16, 24, 253, 4, FP32, FP32, False, False, "own"),       # fp32 rows off the vector grid: 16 x 1, few channels
    (56, 600, 61, 4, FP32, FP32, False, False, "own"),       # 7 x 2
    (60, 600, 61, 4, FP32, FP32, False, False, "second"),    # 5 x 3
    (32, 2049, 61, 4, BF16, FP32, False, False, "second"),   # 2 x 2, 8 x 256 channels and one more
    (88, 400, 64, 4, FP32, FP32, False, False, "own"),       # 11 x 2
    (132, 400, 64, 4, FP32, FP32, False, False, "second"),   # 11 x 3
    (44, 400, 61, 4, FP32, FP16, False, False, "own"),       # 11 x 1
    (88, 400, 61, 4, FP32, FP16, False, False, "second"),    # 11 x 2
    (64, 24, 60, 2, BF16, FP32, False, False, "own"),        # eight rows to a wavefront, 8 x 1
    (100, 24, 1, 4, FP32, FP32, False, False, "own"),        # rows of one element, 2 x 1
    (5, 1500, 100, 4, FP16, FP16, False, True, "own"),       # a channel's rows adjacent, 2 x 1
]


@pytest.mark.parametrize("has_bias", [True, False], ids=["bias", "no_bias"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v).replace("torch.", "") for v in c))
def test_sums_do_not_depend_on_who_adds_them(gpu_device, cc1d_lib, case, has_bias):
    lib, dev = cabi.declare(cc1d_lib), gpu_device
    B, D, L, W, dtype, wtype, strided, batch_inner, who = case
    g = gen(B * 1000 + L)

    def tensor():
        t = torch.randn(D, B, L, generator=g).transpose(0, 1) if batch_inner else torch.randn(B, D, L, generator=g)
        return t.to(dtype)

    x, dout = tensor(), tensor()
    w = (torch.rand(D, 2 * W if strided else W, generator=g) - 0.5).to(wtype)
    w = w[:, ::2] if strided else w
    b = (torch.rand(D, generator=g) - 0.5).to(wtype)
    init, dfin = make_states(B, D, W - 1, dtype, g), make_states(B, D, W - 1, dtype, g)
    xd, dd, bd, initd, dfind = x.to(dev), dout.to(dev), b.to(dev) if has_bias else None, init.to(dev), dfin.to(dev)
    wd = torch.empty(D, 2 * W, dtype=wtype, device=dev)[:, ::2] if strided else torch.empty(D, W, dtype=wtype, device=dev)
    wd.copy_(w)

    def run(knob):
        dx = torch.empty_like(xd)
        dinit = torch.empty(B, W - 1, D, device=dev, dtype=dtype).transpose(1, 2)
        dw, db = torch.full((D, W), float("nan"), device=dev), torch.full((D,), float("nan"), device=dev)
        got = []
        for overwrite in (1, 0):                        # stored, then the same once more on top
            p = cabi.bwd_params(xd, wd, bd, dd, dx, dw, db if has_bias else None, True, initial_states=initd, dfinal_states=dfind,
                                dinitial_states=dinit)
            p.overwrite_dweight = overwrite
            assert lib.cc1d_set_tunable(b"bwd_cf_direct", knob) == 0
            try:
                need = ctypes.c_size_t()
                assert lib.cc1d_bwd_workspace_bytes(ctypes.byref(p), ctypes.byref(need)) == 0
                ws = torch.full((max(16, need.value),), 0xA5, dtype=torch.uint8, device=dev)
                stream = torch.cuda.current_stream().cuda_stream
                assert lib.cc1d_bwd(ctypes.byref(p), ws.data_ptr(), need.value, stream) == 0
                torch.cuda.synchronize()
            finally:
                lib.cc1d_set_tunable(b"bwd_cf_direct", 0)
            assert (need.value == 0) == (who == "one part")
            assert bool((ws == 0xA5).all()) == (who == "one part" or (who == "own" and knob == 0))
            assert has_bias or bool(db.isnan().all())
            got += [dw.clone(), db.clone()] if has_bias else [dw.clone()] * 2
        return [dx, dinit] + got

    own, second = run(0), run(-1)
    assert torch.equal(own[0], second[0]) and torch.equal(own[1], second[1])
    assert torch.equal(own[4], 2 * own[2]) and torch.equal(own[5], 2 * own[3])
    # At most 32 + 6 + 17 additions in a row per sum, of terms of at most 1.1 |dout| |x|: the two
    # orders differ by no more than twice 55 roundings of the sum of the terms' magnitudes.
    terms = 1.1 * dout.float().abs().sum((0, 2)) * x.float().abs().amax((0, 2)).clamp(min=1.0)
    bound = (2 * 55 * 2.0 ** -24 * terms).to(dev)
    assert bool(((own[2] - second[2]).abs() <= bound[:, None]).all())
    rdx, rdw, rdb, rdi = orc.bwd(x, w.float().contiguous(), b.float() if has_bias else None, dout, initial_states=init, dfinal_states=dfin, activation="silu")
    assert_close(own[0], rdx, dtype, "dx")
    assert_close(own[1], rdi, dtype, "dinitial_states")
    assert_close(own[2], rdw, what="dweight", tol=TOL_W)
    if has_bias:
        assert bool(((own[3] - second[3]).abs() <= bound).all())
        assert_close(own[3], rdb, what="dbias", tol=TOL_W)
