"""The z-marching convolution kernels against the per-tap gathering kernel (PVNET_GATHER), which the other
tests hold to the oracle: the k-steps are the same in the same order, so every output is the same bit for
bit.  Sizes where a tile, a ring slot, a k-step or a channel tile ends early."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # shape, cin, cout, x slice (ldx, offset), y slice (ldy, offset), f32 output, ReLU mask
    ((1, 1, 1, 1), 8, 16, 8, 0, 16, 0, False, False),      # one voxel: every neighbour is outside
    ((2, 2, 3, 5), 32, 4, 32, 0, 4, 0, False, False),      # less than one row tile, a quarter channel tile
    ((1, 7, 9, 33), 16, 16, 24, 8, 48, 32, False, True),   # two taps per k-step, slices, mask
    ((3, 5, 17, 31), 24, 20, 24, 0, 20, 0, False, False),  # 21 steps, the last partly beyond K
    ((1, 6, 10, 26), 40, 36, 48, 8, 40, 4, False, True),   # a chunk count no ring in registers takes
    ((2, 3, 11, 19), 48, 16, 48, 0, 16, 0, True, False),   # 41 steps, float output
    ((1, 1, 13, 50), 64, 48, 64, 0, 48, 0, False, True),   # one plane: each dz alone
    ((2, 2, 12, 12), 96, 32, 96, 0, 32, 0, False, False),  # two planes
    ((1, 9, 12, 20), 160, 160, 160, 0, 160, 0, False, True),
    ((1, 4, 6, 14), 224, 68, 232, 8, 72, 4, False, False),
    ((1, 5, 7, 9), 136, 16, 136, 0, 16, 0, False, False),  # no plan: stays on the gathering kernel
    ((1, 4, 8, 8), 32, 18, 32, 0, 18, 0, False, False),    # rows not writable by fours: likewise
]


@pytest.mark.parametrize("case", CASES, ids=[f"m{i}" for i in range(len(CASES))])
def test_march_equals_gather(case):
    import torch
    from pv_dec_original_amd import _native as N
    shape, cin, cout, ldx, xoff, ldy, yoff, f32, mask = case
    m = int(np.prod(shape))
    kpad = -(-27 * cin // 32) * 32
    g = torch.Generator(device="cuda")
    g.manual_seed(7)
    x = torch.randn((m, ldx), generator=g, device="cuda").to(torch.bfloat16)
    w = torch.zeros((cout, kpad), dtype=torch.bfloat16, device="cuda")
    w[:, :27 * cin] = (torch.randn((cout, 27 * cin), generator=g, device="cuda") / (27 * cin) ** 0.5).to(torch.bfloat16)
    b = torch.randn(cout, generator=g, device="cuda")
    act = torch.randn((m, cout), generator=g, device="cuda").to(torch.bfloat16)
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    out = []
    for flags in (0, N.NET_GATHER):
        y = torch.full((m, ldy), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
        c = N.NetConv(N.NetShape(*shape), 27, cin, cout, kpad, C.c_void_p(x.data_ptr() + 2 * xoff), ldx,
                      (0 if mask else N.NET_RELU) | (N.NET_F32OUT if f32 else 0) | flags, C.c_void_p(w.data_ptr()),
                      C.c_void_p(b.data_ptr()), C.c_void_p(y.data_ptr() + y.element_size() * yoff), ldy, cout,
                      C.c_void_p(act.data_ptr()) if mask and cout % 4 == 0 else None)
        N.net_check(N.net().pvnet_conv_fwd(C.byref(c), st))
        out.append(y)
    torch.cuda.synchronize()
    assert torch.equal(out[0].view(torch.int32 if f32 else torch.int16), out[1].view(torch.int32 if f32 else torch.int16))
    rest = out[0].clone()
    rest[:, yoff:yoff + cout] = 7.0
    assert bool((rest == 7.0).all()), "wrote outside the output slice"
