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


WGRAD = [
    # shape, cin, cout, x slice (ldx, offset), dy slice (lddy, offset)
    ((1, 1, 4, 8), 8, 8, 8, 0, 8, 0),         # one plane, one 32-voxel group
    ((2, 3, 4, 4), 16, 16, 24, 8, 32, 16),    # half a group per tile, slices
    ((1, 32, 5, 7), 24, 40, 24, 0, 40, 0),    # odd plane, partial channel tiles
    ((4, 8, 37, 31), 32, 24, 32, 0, 24, 0),   # prime plane sizes: rows are the tiles
    ((3, 7, 16, 10), 48, 16, 48, 0, 16, 0),   # three x tiles per block
    ((1, 9, 12, 40), 64, 160, 64, 0, 160, 0),
    ((1, 4, 8, 64), 224, 72, 224, 0, 72, 0),
    ((1, 64, 1, 2), 8, 16, 8, 0, 16, 0),      # two voxels per plane
]


@pytest.mark.parametrize("case", WGRAD, ids=[f"w{i}" for i in range(len(WGRAD))])
def test_wgrad_march_sums(case):
    """Against 64-bit products of the same bf16 operands.  A sum of M FP32 products, each rounded to 2^-24 of
    the running sum, strays by at most M 2^-24 of the sum of magnitudes; with at most 36,704 voxels and partial
    sums far shorter than M that is below 1e-4 of the largest sum of magnitudes, and 1e-5 of the result's norm."""
    import torch
    from pv_dec_original_amd import _native as N
    shape, cin, cout, ldx, xoff, lddy, doff = case
    nb, d, h, w = shape
    m = int(np.prod(shape))
    g = torch.Generator(device="cuda")
    g.manual_seed(11)
    x = torch.randn((m, ldx), generator=g, device="cuda").to(torch.bfloat16)
    dy = torch.randn((m, lddy), generator=g, device="cuda").to(torch.bfloat16)
    sh = N.NetShape(*shape)
    ws = torch.full((int(N.net().pvnet_wgrad_ws_floats(C.byref(sh), 27, cin, cout)),), 9.0, device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    got = []
    for _ in range(2):
        dw = torch.zeros((cout, 27 * cin), device="cuda")
        db = torch.zeros(cout, device="cuda")
        q = N.NetWgrad(sh, 27, cin, cout, C.c_void_p(x.data_ptr() + 2 * xoff), ldx, lddy,
                       C.c_void_p(dy.data_ptr() + 2 * doff), C.c_void_p(ws.data_ptr()), C.c_void_p(dw.data_ptr()),
                       C.c_void_p(db.data_ptr()))
        N.net_check(N.net().pvnet_conv_wgrad(C.byref(q), st))
        got.append((dw, db))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), "not deterministic"
    xd = x[:, xoff:xoff + cin].double().reshape(nb, d, h, w, cin)
    gd = dy[:, doff:doff + cout].double()
    pad = torch.nn.functional.pad(xd, (0, 0, 1, 1, 1, 1, 1, 1))
    ref = torch.stack([gd.t().contiguous() @ pad[:, a:a + d, b:b + h, e:e + w].reshape(m, cin)
                       for a in range(3) for b in range(3) for e in range(3)], dim=1).reshape(cout, 27 * cin)
    assert float((got[0][0] - ref).norm() / ref.norm()) < 1e-5
    assert float((got[0][1] - gd.sum(0)).norm() / gd.sum(0).norm()) < 1e-5
