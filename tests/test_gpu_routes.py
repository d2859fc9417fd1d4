"""Launch routes chosen by size: a scene gets the same bits whichever route
its engine takes (every resident scene small enough for the one-workgroup
sort, or not)."""
import numpy as np
import pytest

from tests.common import tiny_cfg
from tisphi_amd import _lib as L
from tisphi_amd.scene import build_scene

pytestmark = pytest.mark.gpu

STATE = ["pos", "offset", "cell", "vel", "density", "pressure", "d_vel", "cspm_f", "id0", "cell_start"]


def run(scenes, steps, cells=0):
    """State of the first of ``scenes`` after ``steps`` steps together."""
    eng = L.Engine(scenes[0].method, scenes[0].geo.dim, sum(s.n for s in scenes),
                   sum(s.geo.grid_num_total for s in scenes) + cells, len(scenes))
    slots = []
    for s in scenes:
        slots.append(eng.add_scene(s.desc()))
        L.upload_scene(eng, slots[-1], s)
    eng.step(steps)
    eng.sync()
    out = {f: eng.download(slots[0], f) for f in STATE}
    eng.close()
    return out


def shaken(dim, block, seed=0):
    """A small dam break in motion: particles cross cells in every step."""
    r = 0.005 if dim == 2 else 0.02
    sc = build_scene(tiny_cfg(dim=dim, r=r, domain=(2.0, 1.2, 0.2), block=block))
    rng = np.random.default_rng(seed)
    flow = sc.mat_type == 1
    sc.vel[flow, :dim] = rng.uniform(-2.0, 2.0, (int(flow.sum()), dim))
    return sc


# particles: below one per thread, a full and a part turn of eight per
# thread, the last size the one-workgroup sort takes and the first it leaves
@pytest.mark.parametrize("dim,block", [(2, (0.1, 0.1, 0.0)), (2, (0.8, 0.8, 0.0)), (2, (0.86, 0.8, 0.0)),
                                       (2, (1.5, 1.0, 0.0)), (2, (1.51, 1.0, 0.0)), (3, (0.4, 0.4, 0.1))])
def test_sort_route_of_small_scenes(dim, block):
    sc = shaken(dim, block)
    # a scene of more cells than the one-workgroup sort holds: general route
    wide = build_scene(tiny_cfg(dim=dim, r=0.005 if dim == 2 else 0.02,
                                domain=(6.0, 3.0, 0.2) if dim == 2 else (6.0, 3.0, 1.5),
                                block=(0.2, 0.2, 0.2)))
    assert wide.geo.grid_num_total > 16384
    assert (sc.n <= 16384) == (block[0] < 1.51)
    alone, beside = run([sc], 5), run([sc, wide], 5)
    for f in STATE:
        np.testing.assert_array_equal(alone[f], beside[f], err_msg=f)
