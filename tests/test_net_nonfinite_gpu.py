"""Weight gradients of inputs that are not finite: a value reaches the sums of the voxel pairs inside the box that it is
part of, and no other tap.  Against the same sums in 64 bits over those pairs alone; finite sums to 1e-5 of their norm,
as for finite inputs (partial sums of at most a few thousand FP32 terms)."""
import ctypes as C

import pytest

from tests import plan_probe as P

pytestmark = pytest.mark.gpu

CASES = [
    # shape, cin, cout, x tiles per block, runs per block > 1
    ((2, 3, 8, 8), 8, 64, 1, False),
    ((2, 5, 18, 48), 64, 8, 1, False),     # the last run of planes is short
    ((2, 5, 15, 16), 32, 64, 1, False),    # part of a 32-voxel group
    ((2, 8, 14, 20), 200, 160, 1, True),
    ((3, 32, 20, 21), 120, 8, 2, False),
    ((2, 8, 10, 40), 200, 160, 2, True),   # the last x tiles are one
    ((2, 3, 16, 64), 136, 160, 3, False),
    ((2, 3, 32, 48), 224, 160, 3, True),
]
INF, NAN = float("inf"), float("nan")


@pytest.mark.parametrize("where", ["x", "dy", "both"])
@pytest.mark.parametrize("case", CASES, ids=[f"n{i}" for i in range(len(CASES))])
def test_wgrad_of_values_that_are_not_finite(case, where):
    import torch
    from pv_dec_original_amd import _native as N
    shape, cin, cout, cf, runs = case
    nb, d, h, w = shape
    plan = P.wgrad_plan(shape, cin, cout)
    assert plan["marches"] and plan["cf"] == cf and (plan["per"] > 1) == runs
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    x = torch.randn((nb, d, h, w, cin), generator=g, device="cuda").to(torch.bfloat16)
    dy = torch.randn((nb, d, h, w, cout), generator=g, device="cuda").to(torch.bfloat16)
    if where != "dy":
        x[0, 0, 0, 0, 1] = INF                     # a corner
        x[0, d // 2, 0, w // 2, 3] = NAN           # a face
        x[nb - 1, d - 1, h - 1, w // 3, 5] = -INF  # an edge
        x[nb - 1, d // 2, h // 2, w // 2, cin - 1] = INF
    if where != "x":
        dy[0, 0, 0, 0, 2] = -INF
        dy[0, d // 2, h - 1, w // 2, 4] = NAN
        dy[nb - 1, d - 1, h // 2, w - 1, 6] = INF
        dy[nb - 1, d // 2, h // 2, w // 2, cout - 1] = INF
    sh = N.NetShape(*shape)
    ws = torch.zeros(int(N.net().pvnet_wgrad_ws_floats(C.byref(sh), 27, cin, cout)), device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    dw, db = torch.zeros((cout, 27, cin), device="cuda"), torch.zeros(cout, device="cuda")
    q = N.NetWgrad(sh, 27, cin, cout, x.data_ptr(), cin, cout, dy.data_ptr(), ws.data_ptr(), dw.data_ptr(), db.data_ptr(), 0)
    N.net_check(N.net().pvnet_conv_wgrad(C.byref(q), st))
    torch.cuda.synchronize()

    def part(n, o):  # voxels with a neighbour at offset o, and those neighbours
        return slice(max(0, -o), n - max(0, o)), slice(max(0, o), n - max(0, -o))

    ref = torch.zeros((cout, 27, cin), dtype=torch.float64, device="cuda")
    for tap in range(27):
        (z0, z1), (y0, y1), (x0, x1) = part(d, tap // 9 - 1), part(h, tap // 3 % 3 - 1), part(w, tap % 3 - 1)
        ref[:, tap] = dy[:, z0, y0, x0].double().reshape(-1, cout).t().contiguous() @ x[:, z1, y1, x1].double().reshape(-1, cin)
    for a, b in ((dw, ref), (db, dy.double().sum((0, 1, 2, 3)))):
        assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.isposinf(), b.isposinf()) and torch.equal(a.isneginf(), b.isneginf())
        fin = a.isfinite()
        assert float((a - b)[fin].norm()) <= 1e-5 * float(b[fin].norm())
