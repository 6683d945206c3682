"""The planner of the marching kernels on the host: plans are searched once and kept, and are priced with the blocks
that a CU holds."""
import random

import pytest

from pv_dec_original_amd.warmnet import UNetSpec
from tests import net_march_cases as K
from tests import plan_probe as P


def _unet_keys(shape, levels=(16, 32, 64, 160)):
    """(shape, cin, cout) of every 3x3x3 convolution of a training step: forward and input gradient."""
    nb, d, h, w = shape
    keys = []
    for lay in UNetSpec(levels).layers:
        if lay.ntaps == 27:
            k = len(levels) - 1 if lay.name.startswith("bt") else int(lay.name[1:-1])
            s = (nb, d >> k, h >> k, w >> k)
            keys += [(s, lay.cin, lay.cout), (s, lay.cout, lay.cin)]
    return keys


def test_steady_calls_do_not_search():
    r = random.Random(1)
    shapes = [(8, 96, 96, 96), (1, 96, 96, 192)]
    shapes += [(r.choice([1, 2, 4, 8]),) + tuple(8 * r.randint(2, 14) for _ in range(3)) for _ in range(12)]
    for shape in shapes:
        keys = _unet_keys(shape)
        for k in keys:
            assert P.kept(*k)[1]
        n = P.kept(*keys[0])[0]
        for k in keys:
            assert P.kept(*k) == (n, True), (shape, k)


def test_table_starts_over_when_full():
    n0 = None
    for i in range(1200):
        n, same = P.kept((1, 4, 4 + i % 40, 4 + i // 40), 16, 16)
        assert same
        n0 = n if n0 is None else n0
    assert n - n0 >= 1199  # each shape was new


@pytest.mark.parametrize("key", [((0x7fff, 1, 1, 1), 8, 8), ((1, 1, 1, 4096), 8, 8), ((1, 512, 1, 1), 128, 256)])
def test_odd_shapes_plan_or_not(key):
    assert P.kept(*key)[1]


@pytest.mark.parametrize("lds,vgprs,waves,blocks", [
    (53760, 139, 4, 3),   # 42 pieces of 1,280 bytes, three times within 160 KB
    (54176, 139, 4, 2),   # 43 pieces: 160 KB divided by the bytes alone would be three
    (1280, 139, 4, 3),    # registers: 144 of 512 a lane
    (1280, 256, 4, 2),
    (160 * 1024, 40, 4, 1),
    (42496, 92, 5, 3),
])
def test_blocks_per_cu(lds, vgprs, waves, blocks):
    assert P.lib().probe_blocks_per_cu(lds, vgprs, waves) == blocks


@pytest.mark.parametrize("shape,cin,cout,conv,wgrad", [
    # where marching costs more than the kernel it takes the place of (both measured, us: marching, the other)
    ((8, 52, 6, 12), 120, 56, False, None),    # convolution 161, 62
    ((64, 30, 3, 2), 112, 216, False, None),   # 524, 70
    ((2, 54, 34, 8), 104, 136, False, None),   # 150, 100
    ((256, 2, 2, 2), 96, 32, None, False),     # weight gradient 34, 12
    ((8, 6, 2, 2), 160, 160, None, False),     # 41, 26
    ((8, 6, 89, 14), 8, 136, None, False),     # 77, 36
    ((2, 8, 8, 16), 8, 16, True, False),       # convolution 4, 12; weight gradient 9.6, 7.1
    # and where it is the cheaper
    ((8, 96, 96, 96), 16, 16, True, True),
    ((8, 48, 48, 48), 96, 32, True, True),
    ((8, 12, 12, 12), 160, 160, True, True),
    ((1, 24, 24, 48), 64, 64, True, True),
    ((3, 20, 18, 28), 64, 160, True, True),
])
def test_route_by_price(shape, cin, cout, conv, wgrad):
    if conv is not None:
        assert P.conv_plan(shape, cin, cout)["marches"] == conv
    if wgrad is not None:
        assert P.wgrad_plan(shape, cin, cout)["marches"] == wgrad


@pytest.mark.parametrize("shape,cin,cout", [((1 << 24, 4, 4, 4), 8, 16), ((1 << 24, 1, 8, 8), 8, 8), ((1 << 27, 2, 2, 2), 8, 16),
                                            ((3 << 22, 4, 4, 8), 8, 8), ((64, 31, 601, 1801), 8, 8), ((1 << 25, 2, 2, 8), 32, 16)])
def test_a_plan_fits_a_launch(shape, cin, cout):
    p = P.conv_plan(shape, cin, cout)
    if p:
        blocks = p["ntx"] * p["nty"] * p["nzs"] * p["ng"] * shape[0]
        assert blocks * 64 * (p["wx"] * p["wn"] + p["roll"]) < 2 ** 32


def _conv_instance(p):
    return p["roll"], p["rt"], p["wm"], p["nsteps"] if p["wm"] == 2 else 0


def test_cases_reach_every_convolution_instance():
    """What test_net_march_plans_gpu.py runs: if the prices change, its cases have to follow."""
    seen = set()
    for shape, cin, cout, kernel, rt, wm, wn in K.CONV:
        p = P.conv_plan(shape, cin, cout)
        assert p["marches"] and (p["roll"], p["rt"], p["wm"], p["wn"]) == (kernel == "roll", rt, wm, wn), (shape, cin, cout, p)
        assert p["zseg"] >= 4 and shape[1] % p["zseg"] and p["nzs"] > 1
        seen.add(_conv_instance(p))
    want = {(0, rt, wm, 0) for rt in (1, 2, 3, 4, 6) for wm in (0, 1)} | {(1, rt, wm, 0) for rt in (1, 2, 3, 4, 5) for wm in (0, 1)}
    want |= {(0, rt, 2, n) for rt in (1, 2, 3, 4, 6) for n in (7, 14, 21, 41) if (rt, n) != (6, 41)}
    assert seen == want, (want - seen, seen - want)


def test_cases_in_parts_march():
    kernels = set()
    for shape, cup, cs, cout in K.PARTS:
        f, b, g = P.conv_plan(shape, cup + cs, cout), P.conv_plan(shape, cout, cup + cs), P.wgrad_plan(shape, cup + cs, cout)
        assert f["marches"] and b["marches"] and g["marches"] and f["zseg"] >= 4 and b["zseg"] >= 4
        kernels |= {("up", f["roll"], f["wm"]), ("split", b["roll"], b["wm"]), ("wgrad", g["cf"])}
    assert kernels >= {("up", 0, 0), ("up", 0, 1), ("up", 0, 2), ("up", 1, 0), ("up", 1, 1), ("split", 0, 0), ("split", 0, 1),
                       ("split", 0, 2), ("split", 1, 0), ("split", 1, 1), ("wgrad", 1), ("wgrad", 2), ("wgrad", 3)}


def test_cases_of_weight_gradients():
    for shape, cin, cout, cf, runs, fewer, part, short in K.WGRAD:
        p = P.wgrad_plan(shape, cin, cout)
        got = (p["cf"], p["per"] > 1, -(-cin // 16) % p["cf"] != 0, p["tx"] * p["ty"] % 32 != 0, shape[1] % p["zseg"] != 0)
        assert p["marches"] and got == (cf, runs, fewer, part, short), (shape, cin, cout, p)
