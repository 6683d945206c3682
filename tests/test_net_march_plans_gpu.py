"""Every instance of the marching kernels in runs of several planes (net_march_cases.py; test_net_plans_cpu.py holds the
cases to the plans they are for): convolutions bit for bit against the gathering kernel, whole and in two parts, and
weight gradients of whole numbers, whose sums are exact (below 2^24) in any order."""
import ctypes as C

import pytest

from tests import net_march_cases as K
from tests.test_net_march_gpu import test_march_equals_gather as equals_gather
from tests.test_net_parts_gpu import test_parts_equal_laid_out as equals_laid_out

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("i", range(len(K.CONV)))
def test_convolution_instances(i):
    shape, cin, cout = K.CONV[i][:3]
    # slices, float outputs and ReLU masks in turn
    ldx, xo, ldy, yo = (cin, 0, cout, 0) if i % 2 else (cin + 16, 8, cout + 8, 4)
    equals_gather((shape, cin, cout, ldx, xo, ldy, yo, i % 3 == 0, i % 4 == 1))


@pytest.mark.parametrize("case", K.PARTS)
def test_convolutions_in_parts(case):
    shape, cup, cs, cout = case
    equals_laid_out((shape, cup, cs, cout, cup + 8, cs, 0))


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("case", K.WGRAD)
def test_weight_gradients_of_whole_numbers(case, bias):
    import torch
    from pv_dec_original_amd import _native as N
    (nb, d, h, w), cin, cout = case[:3]
    m = nb * d * h * w
    assert 16 * m < 2 ** 24
    g = torch.Generator(device="cuda")
    g.manual_seed(6)
    x = torch.randint(-4, 5, (m, cin + 8), generator=g, device="cuda").to(torch.bfloat16)
    dy = torch.randint(-4, 5, (m, cout + 16), generator=g, device="cuda").to(torch.bfloat16)
    sh = N.NetShape(nb, d, h, w)
    n = int(N.net().pvnet_wgrad_ws_floats(C.byref(sh), 27, cin, cout))
    ws = torch.full((n + 64,), 9.0, device="cuda")
    dw, db = torch.full((cout, 27 * cin), 7.0, device="cuda"), torch.full((cout,), 7.0, device="cuda")
    q = N.NetWgrad(sh, 27, cin, cout, x.data_ptr() + 16, cin + 8, cout + 16, dy.data_ptr() + 32, ws.data_ptr(), dw.data_ptr(),
                   db.data_ptr() if bias else None, 0)
    N.net_check(N.net().pvnet_conv_wgrad(C.byref(q), C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    torch.cuda.synchronize()
    xd, gd = x[:, 8:].double().reshape(nb, d, h, w, cin), dy[:, 16:].double()
    pad = torch.nn.functional.pad(xd, (0, 0, 1, 1, 1, 1, 1, 1))
    ref = torch.stack([gd.t().contiguous() @ pad[:, a:a + d, b:b + h, e:e + w].reshape(m, cin)
                       for a in range(3) for b in range(3) for e in range(3)], dim=1).reshape(cout, 27 * cin)
    assert torch.equal(dw.double(), ref)
    assert torch.equal(db.double(), gd.sum(0)) if bias else bool((db == 7.0).all())
    assert bool((ws[n:] == 9.0).all())
