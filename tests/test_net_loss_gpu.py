"""Loss with its channel weights in host memory: the bits of the entry that reads them on the device."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,nc", [(1, 1), (255, 4), (257, 4), (5000, 8), (70000, 3)])
def test_host_weights_equal_device_weights(m, nc):
    import torch
    from pv_dec_original_amd import _native as N
    NL, st = N.net(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    g = torch.Generator(device="cuda")
    g.manual_seed(9)
    y = torch.randn((m, 8), generator=g, device="cuda")
    t = torch.randn((m, nc), generator=g, device="cuda").to(torch.bfloat16)
    code = (torch.rand(m, generator=g, device="cuda") < 0.6).to(torch.uint8)
    w = [1.0, 0.3, 2.5, 0.0, 7.0, 0.125, 1e-3, 40.0][:nc]
    wd = torch.tensor(w, device="cuda")
    out = []
    for host in (False, True):
        dy = torch.full((m, 8), 7.0, dtype=torch.bfloat16, device="cuda")
        part = torch.zeros(int(NL.pvnet_loss_ws_doubles(m)), dtype=torch.float64, device="cuda")
        loss = torch.zeros(2, dtype=torch.float64, device="cuda")
        wc = C.cast((C.c_float * nc)(*w), C.c_void_p) if host else C.c_void_p(wd.data_ptr())
        f = NL.pvnet_mse_loss_host_weights if host else NL.pvnet_mse_loss
        N.net_check(f(m, nc, C.c_void_p(y.data_ptr()), 8, C.c_void_p(t.data_ptr()), C.c_void_p(code.data_ptr()), wc,
                      C.c_void_p(dy.data_ptr()), 8, C.c_void_p(part.data_ptr()), C.c_void_p(loss.data_ptr()), st))
        torch.cuda.synchronize()
        out.append((dy.view(torch.int16), loss.view(torch.int64)))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
