"""Weight layouts of several layers in one launch against the definition, bit for bit: more layers than one launch
takes, rows with padding, layouts that start off a 16-byte boundary."""
import ctypes as C

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers,shift", [([(1, 16, 8)], 0), ([(27, 8, 16), (1, 16, 8), (27, 40, 24), (27, 3, 5)], 0),
                                          ([(27, 8, 8)] * 31 + [(1, 8, 8), (27, 48, 16), (1, 5, 3)], 0),
                                          ([(27, 16, 8), (1, 8, 24)], 1)])
def test_pack_layers(layers, shift):
    import torch
    from pv_dec_original_amd import _native as N
    g = torch.Generator(device="cuda")
    g.manual_seed(2)
    jobs, keep = (N.NetPack * len(layers))(), []
    for j, (nt, ci, co) in zip(jobs, layers):
        w = torch.randn((co, nt, ci), generator=g, device="cuda")
        kp, kd = -(-nt * ci // 32) * 32, -(-nt * co // 32) * 32
        wt, wd = (torch.full((r * k + shift + 8,), 7.0, dtype=torch.bfloat16, device="cuda") for r, k in ((co, kp), (ci, kd)))
        j.w32, j.wt, j.wd = w.data_ptr(), wt.data_ptr() + 2 * shift, wd.data_ptr() + 2 * shift
        j.ntaps, j.cin, j.cout = nt, ci, co
        keep.append((w, wt, wd, kp, kd))
    N.net_check(N.net().pvnet_pack_layers(jobs, len(layers), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    for (nt, ci, co), (w, wt, wd, kp, kd) in zip(layers, keep):
        a, b = torch.zeros((co, kp), device="cuda"), torch.zeros((ci, kd), device="cuda")
        a[:, :nt * ci] = w.reshape(co, nt * ci)
        b[:, :nt * co] = w.flip(1).permute(2, 1, 0).reshape(ci, nt * co)
        for got, ref in ((wt, a), (wd, b)):
            n = ref.numel()
            assert torch.equal(got[shift:shift + n].view(torch.int16), ref.to(torch.bfloat16).reshape(-1).view(torch.int16))
            assert bool((got[:shift] == 7.0).all()) and bool((got[shift + n:] == 7.0).all()), "wrote outside the layout"
