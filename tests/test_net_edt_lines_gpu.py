"""pvnet_wall_distance on more lines than one launch takes (2^32 threads): many copies of one box, whose distances the
oracle gives."""
import ctypes as C

import numpy as np
import pytest

from tests import net_oracle as O

pytestmark = pytest.mark.gpu


def test_wall_distance_of_many_lines():
    import torch
    from pv_dec_original_amd import _native as N
    box, nb = (16, 32, 1), 132000  # 67,584,000 lines of one voxel; 2^26 is 67,108,864
    rng = np.random.default_rng(5)
    one = (rng.random((1,) + box) >= 0.02).astype(np.uint8)
    code = torch.from_numpy(one).cuda().repeat(nb, 1, 1, 1)
    out = torch.full((code.numel(),), -1.0, device="cuda")
    N.net_check(N.net().pvnet_wall_distance(C.byref(N.NetShape(nb, *box)), C.c_void_p(code.data_ptr()), C.c_void_p(out.data_ptr()),
                                            C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    ref = torch.from_numpy(O.wall_distance((1,) + box, one).reshape(-1).astype(np.float32)).cuda()
    assert bool((out.view(nb, -1) == ref).all())
