"""Convolutions and weight gradients at the largest voxel counts that are accepted (below 2^31, multiples of 32), where the last chunk's
end lies beyond 2^31 and a launch needs 2^32 threads.  Small whole numbers in a few voxels, zeros elsewhere: every sum is exact."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(1, 96, 2731, 8191), (64, 31, 601, 1801), (1, 1, 32, 67106816)]  # 2^31 - 32, - 64, - 65,536


@pytest.mark.parametrize("shape", SHAPES)
def test_pointwise_wgrad_at_the_voxel_limit(shape):
    import torch
    from pv_dec_original_amd import _native as N
    m = shape[0] * shape[1] * shape[2] * shape[3]
    assert 2 ** 31 - 2 ** 18 < m < 2 ** 31 and m % 32 == 0
    if torch.cuda.mem_get_info()[0] < 80 * 2 ** 30:
        pytest.skip("needs 80 GB of device memory")
    x = torch.zeros((m, 8), dtype=torch.bfloat16, device="cuda")
    dy = torch.zeros((m, 8), dtype=torch.bfloat16, device="cuda")
    v = torch.tensor([0, 127, 128, m // 2, m - 129, m - 128, m - 33, m - 32, m - 1], device="cuda")
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    xv = torch.randint(-8, 9, (len(v), 8), generator=g, device="cuda").float()
    dv = torch.randint(-8, 9, (len(v), 8), generator=g, device="cuda").float()
    x[v], dy[v] = xv.to(torch.bfloat16), dv.to(torch.bfloat16)
    sh = N.NetShape(*shape)
    ws = torch.zeros(int(N.net().pvnet_wgrad_ws_floats(C.byref(sh), 1, 8, 8)), device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for flags in (0, N.NET_GATHER):
        dw, db = torch.full((8, 8), 7.0, device="cuda"), torch.full((8,), 7.0, device="cuda")
        q = N.NetWgrad(sh, 1, 8, 8, x.data_ptr(), 8, 8, dy.data_ptr(), ws.data_ptr(), dw.data_ptr(), db.data_ptr(), flags)
        N.net_check(N.net().pvnet_conv_wgrad(C.byref(q), st))
        torch.cuda.synchronize()
        assert torch.equal(dw, dv.t() @ xv) and torch.equal(db, dv.sum(0)), f"flags {flags}"
    del x, dy
    torch.cuda.empty_cache()


@pytest.mark.parametrize("shape,cout", [(SHAPES[0], 8), (SHAPES[1], 24)])
def test_convolution_at_the_voxel_limit(shape, cout):
    """The centre tap alone, an identity: what is in a few voxels comes out there, and nothing anywhere else."""
    import torch
    from pv_dec_original_amd import _native as N
    m = shape[0] * shape[1] * shape[2] * shape[3]
    if torch.cuda.mem_get_info()[0] < (8 + cout) * 4.5 * 2 ** 30:
        pytest.skip("needs 75 to 145 GB of device memory")
    x = torch.zeros((m, 8), dtype=torch.bfloat16, device="cuda")
    v = torch.tensor([0, 127, 128, m // 2, m - 129, m - 128, m - 33, m - 1], device="cuda")
    xv = torch.arange(1, 8 * len(v) + 1, device="cuda").view(-1, 8).to(torch.bfloat16)
    x[v] = xv
    w = torch.zeros((cout, 224), dtype=torch.bfloat16, device="cuda")
    w[torch.arange(8), 13 * 8 + torch.arange(8)] = 1
    y = torch.full((m, cout), 7.0, dtype=torch.bfloat16, device="cuda")
    st = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    for flags in (0, N.NET_GATHER):
        y.fill_(7.0)
        c = N.NetConv(N.NetShape(*shape), 27, 8, cout, 224, x.data_ptr(), 8, flags, w.data_ptr(), None, y.data_ptr(), cout, 0, None)
        N.net_check(N.net().pvnet_conv_fwd(C.byref(c), st))
        torch.cuda.synchronize()
        assert torch.equal(y[v, :8], xv) and not y[v, 8:].any(), f"flags {flags}"
        y[v] = 0
        assert not any(bool(part.any()) for part in y.view(torch.int16).view(-1).split(2 ** 30)), f"flags {flags}"
    del x, y
    torch.cuda.empty_cache()
