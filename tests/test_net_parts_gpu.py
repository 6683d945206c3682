"""Convolutions whose input or output lies in two parts (an upsampled half-size tensor in front of a skip)
against the same kernels on the laid-out concatenation: forward and input gradient bit for bit, weight
gradients the same sums in the same order.  Marching and gathering kernels, sizes with ragged tiles."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # shape, cup, skip channels, cout, ldu, ldx, flags (4: gathering kernel)
    ((1, 2, 2, 2), 8, 8, 16, 8, 8, 0),        # eight voxels, one parent
    ((2, 4, 6, 10), 32, 16, 16, 32, 16, 0),   # 41 steps in registers, two boxes
    ((1, 6, 14, 34), 32, 16, 16, 40, 24, 0),  # ragged tiles, wider rows
    ((2, 8, 12, 16), 64, 32, 32, 64, 32, 0),  # rolling accumulators
    ((1, 2, 10, 26), 160, 64, 64, 160, 64, 0),
    ((1, 4, 6, 8), 8, 24, 24, 8, 24, 0),      # a channel tile with both parts
    ((1, 4, 4, 12), 128, 8, 16, 128, 8, 0),   # no plan: the gathering kernel
    ((2, 4, 6, 8), 24, 16, 40, 32, 16, 4),
    ((1, 8, 8, 4), 16, 48, 64, 16, 56, 4),
]


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("case", CASES, ids=[f"p{i}" for i in range(len(CASES))])
def test_parts_equal_laid_out(case):
    import torch
    from pv_dec_original_amd import _native as N
    shape, cup, cs, cout, ldu, ldx, flags = case
    nb, d, h, w = shape
    m, cin, NL = int(np.prod(shape)), cup + cs, N.net()
    gen = torch.Generator(device="cuda")
    gen.manual_seed(11)

    def rnd(*sz):
        return torch.randn(sz, generator=gen, device="cuda").to(torch.bfloat16)

    up, skip, dy = rnd(m // 8, ldu), rnd(m, ldx), rnd(m, cout)
    kpad, kpad_d = -(-27 * cin // 32) * 32, -(-27 * cout // 32) * 32
    wt = torch.zeros((cout, kpad), dtype=torch.bfloat16, device="cuda")
    wt[:, :27 * cin] = rnd(cout, 27 * cin) / (27 * cin) ** 0.5
    wd = torch.zeros((cin, kpad_d), dtype=torch.bfloat16, device="cuda")
    wd[:, :27 * cout] = rnd(cin, 27 * cout) / (27 * cout) ** 0.5
    bias = torch.randn(cout, generator=gen, device="cuda")
    u = up[:, :cup].reshape(nb, d // 2, h // 2, w // 2, cup)
    u = u.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3).reshape(m, cup)
    cat = torch.cat([u, skip[:, :cs]], 1).contiguous()
    S, st = N.NetShape(*shape), C.c_void_p(torch.cuda.current_stream().cuda_stream)

    y = [torch.full((m, cout), 7.0, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    conv = [N.NetConv(S, 27, cin, cout, kpad, _ptr(x), ld, N.NET_RELU | flags, _ptr(wt), _ptr(bias), _ptr(o), cout, 0, None)
            for x, ld, o in ((cat, cin, y[0]), (skip, ldx, y[1]))]
    N.net_check(NL.pvnet_conv_fwd(C.byref(conv[0]), st))
    N.net_check(NL.pvnet_conv_up_fwd(C.byref(conv[1]), _ptr(up), ldu, cup, st))
    torch.cuda.synchronize()
    assert torch.equal(y[0].view(torch.int16), y[1].view(torch.int16))

    dcat = torch.full((m, cin), 7.0, dtype=torch.bfloat16, device="cuda")
    du, ds = torch.full((m, ldu), 7.0, dtype=torch.bfloat16, device="cuda"), torch.full_like(skip, 7.0)
    whole = N.NetConv(S, 27, cout, cin, kpad_d, _ptr(dy), cout, flags, _ptr(wd), None, _ptr(dcat), cin, 0, None)
    split = N.NetConv(S, 27, cout, cin, kpad_d, _ptr(dy), cout, flags, _ptr(wd), None, _ptr(ds), ldx, 0, None)
    N.net_check(NL.pvnet_conv_fwd(C.byref(whole), st))
    N.net_check(NL.pvnet_conv_split_fwd(C.byref(split), _ptr(du), ldu, cup, st))
    torch.cuda.synchronize()
    assert torch.equal(torch.cat([du[:, :cup], ds[:, :cs]], 1).view(torch.int16), dcat.view(torch.int16))
    assert bool((du[:, cup:] == 7.0).all()) and bool((ds[:, cs:] == 7.0).all()), "wrote outside the channels"

    if m % 32:
        return
    ws = torch.zeros(NL.pvnet_wgrad_ws_floats(C.byref(S), 27, cin, cout), device="cuda")
    out = []
    for x, ld in ((cat, cin), (skip, ldx)):
        dw, db = torch.full((cout, 27 * cin), 7.0, device="cuda"), torch.full((cout,), 7.0, device="cuda")
        g = N.NetWgrad(S, 27, cin, cout, _ptr(x), ld, cout, _ptr(dy), _ptr(ws), _ptr(dw), _ptr(db), flags)
        if x is cat:
            N.net_check(NL.pvnet_conv_wgrad(C.byref(g), st))
        else:
            N.net_check(NL.pvnet_conv_up_wgrad(C.byref(g), _ptr(up), ldu, cup, st))
        out.append((dw, db))
    torch.cuda.synchronize()
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def test_parts_refused():
    """Odd sizes, part widths that are not whole chunks, missing tensors."""
    import torch
    from pv_dec_original_amd import _native as N
    NL, st = N.net(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    t = torch.zeros(4 * 6 * 8 * 32, dtype=torch.bfloat16, device="cuda")
    for shape, up, ldu, cup in (((1, 3, 6, 8), t, 8, 8), ((1, 4, 6, 8), t, 8, 4), ((1, 4, 6, 8), t, 8, 16),
                                ((1, 4, 6, 8), None, 8, 8), ((1, 4, 6, 8), t, 4, 8)):
        c = N.NetConv(N.NetShape(*shape), 27, 16, 16, 448, _ptr(t), 8, 0, _ptr(t), None, _ptr(t), 16, 0, None)
        assert NL.pvnet_conv_up_fwd(C.byref(c), _ptr(up) if up is not None else None, ldu, cup, st) == 1
        g = N.NetWgrad(N.NetShape(*shape), 27, 16, 16, _ptr(t), 8, 16, _ptr(t), _ptr(t), _ptr(t), None, 0)
        assert NL.pvnet_conv_up_wgrad(C.byref(g), _ptr(up) if up is not None else None, ldu, cup, st) == 1
    c = N.NetConv(N.NetShape(1, 4, 6, 8), 27, 16, 16, 448, _ptr(t), 16, 0, _ptr(t), None, _ptr(t), 8, 0, None)
    assert NL.pvnet_conv_split_fwd(C.byref(c), _ptr(t), 8, 16, st) == 1
    assert NL.pvnet_conv_split_fwd(C.byref(c), None, 8, 8, st) == 1
