"""pvnet_wall_distance where a ballot word, a column group or a line ends early, against the oracle: distances
are square roots of exact integers, so they are equal to the last bit."""
import ctypes as C

import numpy as np
import pytest

from tests import net_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(1, 1, 1, 1), (2, 3, 5, 63), (1, 33, 2, 64), (1, 2, 17, 65), (2, 16, 16, 129),
                                   (1, 9, 31, 200), (1, 2, 2, 512), (1, 512, 2, 3), (1, 3, 300, 2)])
@pytest.mark.parametrize("solid", [0.0, 0.003, 0.5])
def test_wall_distance_edges(shape, solid):
    import torch
    from pv_dec_original_amd import _native as N
    rng = np.random.default_rng(3)
    code = (rng.random(shape) >= solid).astype(np.uint8)
    cd = torch.from_numpy(code).cuda()
    out = torch.full((code.size,), -1.0, device="cuda")
    N.net_check(N.net().pvnet_wall_distance(C.byref(N.NetShape(*shape)), C.c_void_p(cd.data_ptr()),
                                            C.c_void_p(out.data_ptr()),
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    ref = O.wall_distance(shape, code).reshape(-1).astype(np.float32)
    assert np.array_equal(out.cpu().numpy(), ref)
