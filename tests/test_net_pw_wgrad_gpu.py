"""Weight and bias gradients of pointwise layers (at most 32 inputs and 16 outputs: one pass over x and dy) against
64-bit products of the same bf16 operands, at voxel counts around a wave's chunk of 128 and a block's run."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # shape, cin, cout, x slice (ldx, offset), dy slice (lddy, offset)
    ((1, 1, 4, 8), 8, 8, 8, 0, 8, 0),          # a quarter of one chunk
    ((2, 3, 4, 4), 16, 8, 24, 8, 8, 0),        # 96 voxels, slice of x
    ((1, 4, 8, 20), 24, 16, 24, 0, 32, 16),    # five chunks, half a channel tile, slice of dy
    ((3, 8, 32, 42), 32, 8, 40, 8, 16, 8),     # 252 chunks
    ((4, 8, 37, 31), 16, 16, 16, 0, 16, 0),    # the last chunk ends early
    ((5, 64, 45, 32), 16, 8, 16, 0, 8, 0),     # more than one round of the device's blocks
]


@pytest.mark.parametrize("case", CASES, ids=[f"h{i}" for i in range(len(CASES))])
def test_pointwise_wgrad_sums(case):
    """A sum of M FP32 products, each rounded to 2^-24 of the running sum, strays by at most M 2^-24 of the sum of
    magnitudes; partial sums are far shorter than M (at most 2304 terms), so the result is within 1e-5 of its norm."""
    import torch
    from pv_dec_original_amd import _native as N
    shape, cin, cout, ldx, xoff, lddy, doff = case
    m = shape[0] * shape[1] * shape[2] * shape[3]
    g = torch.Generator(device="cuda")
    g.manual_seed(5)
    x = torch.randn((m, ldx), generator=g, device="cuda").to(torch.bfloat16)
    dy = torch.randn((m, lddy), generator=g, device="cuda").to(torch.bfloat16)
    sh = N.NetShape(*shape)
    ws = torch.full((int(N.net().pvnet_wgrad_ws_floats(C.byref(sh), 1, cin, cout)),), 9.0, device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    got = []
    for _ in range(2):
        dw, db = torch.zeros((cout, cin), device="cuda"), torch.zeros(cout, device="cuda")
        q = N.NetWgrad(sh, 1, cin, cout, C.c_void_p(x.data_ptr() + 2 * xoff), ldx, lddy,
                       C.c_void_p(dy.data_ptr() + 2 * doff), C.c_void_p(ws.data_ptr()), C.c_void_p(dw.data_ptr()),
                       C.c_void_p(db.data_ptr()), 0)
        N.net_check(N.net().pvnet_conv_wgrad(C.byref(q), st))
        got.append((dw, db))
    torch.cuda.synchronize()
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), "not deterministic"
    xd, gd = x[:, xoff:xoff + cin].double(), dy[:, doff:doff + cout].double()
    ref = gd.t().contiguous() @ xd
    assert float((got[0][0] - ref).norm() / ref.norm()) < 1e-5
    assert float((got[0][1] - gd.sum(0)).norm() / gd.sum(0).norm()) < 1e-5


WIDE = [
    # the tiled kernel, whose bias sums ride on its first blocks: each tile height, several k-tiles, part chunks
    ((1, 1, 4, 8), 40, 8, 40, 0, 8, 0),
    ((2, 3, 4, 4), 8, 24, 8, 0, 32, 8),
    ((1, 8, 32, 43), 72, 64, 80, 8, 64, 0),
    ((3, 8, 37, 32), 224, 136, 224, 0, 136, 0),
]


@pytest.mark.parametrize("case", WIDE, ids=[f"t{i}" for i in range(len(WIDE))])
def test_wide_pointwise_wgrad_sums(case):
    test_pointwise_wgrad_sums(case)
