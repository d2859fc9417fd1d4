"""Launch routes chosen by size: a scene gets the same bits whichever route
its engine takes (every resident scene small enough for the one-workgroup
sort, or not)."""
from types import SimpleNamespace

import numpy as np
import pytest

from oracle.sph_numpy import NumpySPH
from tests.common import tiny_cfg
from tests.test_cell_rule import renorm
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


def sorts(sc):
    """(launches of the one-workgroup sort, of the general one) in a step."""
    eng = L.Engine(sc.method, sc.geo.dim, sc.n, sc.geo.grid_num_total, 1)
    L.upload_scene(eng, eng.add_scene(sc.desc()), sc)
    eng.timing(True)
    eng.step(1)
    eng.sync()
    out = eng.kernel_time("sort_small")[1], eng.kernel_time("scatter")[1]
    eng.close()
    return out


# cells: more than half of what the one-workgroup sort holds (64 KiB less 16
# words), all of it, and the next larger grid
@pytest.mark.parametrize("domain,cells", [((2.8, 2.7), 8832), ((3.9, 3.66), 16368), ((3.81, 3.75), 16383)])
def test_sort_route_of_many_cells(domain, cells):
    sc = build_scene(tiny_cfg(r=0.005, domain=domain + (0.2,), block=(1.0, 0.9, 0.0)))
    flow = sc.mat_type == 1
    sc.vel[flow, :2] = np.random.default_rng(0).uniform(-2.0, 2.0, (int(flow.sum()), 2))
    assert sc.geo.grid_num_total == cells and sc.n <= 16384
    assert sorts(sc) == ((1, 0) if cells <= 16368 else (0, 1))
    wide = build_scene(tiny_cfg(r=0.005, domain=(6.0, 3.0, 0.2), block=(0.2, 0.2, 0.0)))
    alone, beside = run([sc], 5), run([sc, wide], 5)
    for f in STATE:
        np.testing.assert_array_equal(alone[f], beside[f], err_msg=f)


def uneven(method, dim, nan, seed=3):
    """A scene whose flow particles lie from far apart to 80 per cell (lists
    longer than the engine keeps, cells of more than 32 particles, windows
    wider than a cell tile), in any order; ``nan``: one offset is not a
    number and one is infinite."""
    r = 0.006 if dim == 2 else 0.016
    sc = build_scene(tiny_cfg(method=method, dim=dim, xsph=True, r=r, domain=(1.0, 0.6, 0.24),
                              block=(0.6, 0.3, 0.24) if dim == 2 else (0.4, 0.3, 0.24)))
    rng = np.random.default_rng(seed)
    flow = np.flatnonzero((sc.mat_type == 1) | (sc.mat_type == 2))
    n = flow.size
    # x crowds towards 0: the density falls off exponentially along x
    x = np.stack([rng.exponential(0.025 if dim == 2 else 0.05, n) % 0.9, rng.uniform(0.02, 0.5, n), rng.uniform(0.02, 0.2, n)], 1)
    sc.pos[flow, :dim] = (x + 0.02)[:, :dim]
    sc.vel[flow, :dim] = rng.uniform(-0.1, 0.1, (n, dim))
    bad = {int(flow[5]): np.nan, int(flow[70]): np.inf} if nan else {}
    return sc, bad


@pytest.mark.parametrize("method,dim,nan", [(1, 2, False), (1, 3, False), (2, 2, False), (3, 2, False), (3, 3, False),
                                            (1, 2, True)])
def test_list_modes_agree_on_uneven_scenes(method, dim, nan):
    """Walk in every pass (mode 0), lists from the walk (1) and from staged
    windows (2, every cell tile) give the same bits."""
    sc, bad = uneven(method, dim, nan)
    fields = STATE + (["stress"] if method != 1 else [])
    ref = None
    for mode, tile in [(0, 256), (1, 256), (2, 128), (2, 256), (2, 512)]:
        eng = L.Engine(sc.method, dim, sc.n, sc.geo.grid_num_total, 1)
        eng.set_neighbor_list(mode)
        eng.set_cell_tile(tile)
        slot = eng.add_scene(sc.desc())
        L.upload_scene(eng, slot, sc)
        if bad:
            off = eng.download(slot, "offset")
            for i, v in bad.items():
                off[i, 0] = v
            eng.upload(slot, "offset", off)
        if mode == 2 and not nan:
            eng.run("sort")
            eng.run("shepard")
            count = eng.neighbor_lists(slot)[0]
            assert (count == -1).any() and (count == 0).any() and (count > 0).any()
        eng.step(2)
        out = {f: eng.download(slot, f) for f in fields}
        eng.close()
        if ref is None:
            ref = out
        for f in fields:
            np.testing.assert_array_equal(out[f], ref[f], err_msg=f"mode {mode} tile {tile}: {f}")


@pytest.mark.parametrize("dim,kernel", [(2, 0), (2, 1), (3, 1)])
def test_stress_regularisation_sums(dim, kernel):
    """The regularised stress of uneven scenes in motion (0 to hundreds of
    pairs per particle, particles that have left their cell) against the sums
    in float64 over the same stencil."""
    sc, _ = uneven(2, dim, False)
    sc.kernel = kernel
    soil = sc.mat_type == 2
    rng = np.random.default_rng(5)
    step = 0.2 * sc.geo.grid_size / sc.dt  # at most a fifth of a cell
    sc.vel[soil, :dim] = rng.uniform(-step, step, (int(soil.sum()), dim))
    eng = L.Engine(sc.method, dim, sc.n, sc.geo.grid_num_total, 1)
    slot = eng.add_scene(sc.desc())
    L.upload_scene(eng, slot, sc)
    eng.upload(slot, "stress", rng.uniform(-1e4, 1e4, (sc.n, 6)))
    for what in ("sort", "shepard", "init_tmp", "advect_pos", "advect_something"):
        eng.run(what)
    off, cell, mv, ty, cs, tmp, out = (eng.download(slot, f) for f in
                                       ("offset", "cell", "m_V", "type", "cspm_f", "stress_tmp", "stress"))
    eng.close()
    gn, g, rs = sc.geo.grid_num, sc.geo.grid_size, sc.geo.support_radius
    c = np.stack(np.unravel_index(cell.astype(np.int64), gn), 1)[:, :dim]
    new = c + np.floor(off[:, :dim] / g).astype(np.int64)
    x = off[:, :dim] + c * g
    flow = np.flatnonzero(ty == 2)
    like = SimpleNamespace(h=sc.geo.smoothing_len, dim=dim, d={"kernel": kernel})
    moved, longest = 0, 0
    for i in flow[:: max(1, flow.size // 400)]:
        d = x[i] - x[flow]
        r = np.sqrt((d * d).sum(1))
        ok = (np.abs(c[flow] - new[i]).max(1) <= 1) & (r < rs) & (flow != i)
        j, w = flow[ok], NumpySPH.W(like, r[ok])
        t = mv[j, None] * tmp[j] * w[:, None]
        ref = t.sum(0) * cs[i]
        # float32 sums of n terms of a few roundings, and the distance's
        # error (2^-22 of the cell size, from the offsets) through W
        tol = abs(cs[i]) * ((j.size + 16) * 2.0 ** -24 * np.abs(t).sum(0)
                            + 2.0 ** -19 * (mv[j, None] * np.abs(tmp[j])).sum(0) * float(NumpySPH.W(like, 1e-3 * rs)))
        assert (np.abs(out[i] - ref) <= tol).all(), (i, j.size, out[i], ref, tol)
        moved += bool((new[i] != c[i]).any())
        longest = max(longest, j.size)
    assert moved > 0 and longest > 64


def test_read_outs_of_several_stages():
    """Fields of every row size come back as they were sent, also where a
    read-out takes several turns of its staging memory and the last is short."""
    sc = build_scene(tiny_cfg(method=2, dim=2, r=0.001, domain=(0.6, 0.6, 0.1), block=(0.5, 0.5, 0.0)))
    assert sc.n * 24 > 2.5 * 2 ** 19 and (sc.n * 4) % 2 ** 19
    rng = np.random.default_rng(1)
    eng = L.Engine(2, 2, sc.n, sc.geo.grid_num_total, 1)
    slot = eng.add_scene(sc.desc())
    L.upload_scene(eng, slot, sc)
    sent = {"vel": rng.normal(size=(sc.n, 3)), "density": rng.uniform(900, 1100, sc.n),
            "stress": rng.normal(size=(sc.n, 6)), "stress_tmp": rng.normal(size=(sc.n, 6))}
    ints = {"id0": rng.permutation(sc.n), "obj_id": rng.integers(0, 3, sc.n), "type": sc.mat_type}
    for f, v in list(sent.items()) + list(ints.items()):
        eng.upload(slot, f, v)
    for f, v in sent.items():
        np.testing.assert_array_equal(eng.download(slot, f), v.astype(np.float32).astype(np.float64), err_msg=f)
    for f, v in ints.items():
        np.testing.assert_array_equal(eng.download(slot, f), v, err_msg=f)
    eng.run("sort")
    cell, start = eng.download(slot, "cell"), eng.download(slot, "cell_start")
    np.testing.assert_array_equal(np.diff(start), np.bincount(cell, minlength=start.size - 1))
    off, pos = eng.download(slot, "offset"), eng.download(slot, "pos")
    gn, g = sc.geo.grid_num, sc.geo.grid_size
    c = np.stack(np.unravel_index(cell, gn), 1)
    want = sc.geo.vdomain_start[None] + c * g + off
    np.testing.assert_array_equal(pos[:, :2], want[:, :2])
    eng.close()


@pytest.mark.parametrize("method,dim,ti,xsph", [(1, 2, 4, False), (1, 3, 4, True), (2, 2, 4, True), (2, 3, 1, False),
                                                (3, 2, 4, True), (3, 2, 2, False), (3, 3, 2, True), (3, 2, 1, False)])
def test_fused_integrators_equal_the_passes(method, dim, ti, xsph):
    """The fused step's launches (stages of RK4, DP's rate and mapping within
    their neighbours) give the bits of the passes run one by one."""
    sc = build_scene(tiny_cfg(method=method, dim=dim, xsph=xsph, ti=ti, domain=(0.4, 0.3, 0.08),
                              block=(0.2, 0.15, 0.06)))
    rng = np.random.default_rng(7)
    flow = sc.mat_type > 0
    sc.vel[flow, :dim] = rng.uniform(-1.0, 1.0, (int(flow.sum()), dim))
    fields = STATE + ["density_tmp", "v_tmp", "m_V", "d_density"]
    if method != 1:
        fields += ["stress", "stress_tmp", "strain_equ", "d_strain_equ"]
    if method == 3:
        fields += ["strain_equ_p", "flag_retmap", "d_stress", "d_strain_equ_p"]
    out = []
    for fused in (False, True):
        eng = L.Engine(method, dim, sc.n, sc.geo.grid_num_total, 1)
        slot = eng.add_scene(sc.desc())
        L.upload_scene(eng, slot, sc)
        for _ in range(1 if fused else 4):
            eng.step(4) if fused else eng.run("step")
        out.append({f: eng.download(slot, f) for f in fields})
        eng.close()
    for f in fields:
        np.testing.assert_array_equal(out[1][f], out[0][f], err_msg=f)
    assert np.isfinite(out[0]["vel"]).all()


@pytest.mark.parametrize("method,dim", [(1, 2), (1, 3), (2, 2), (2, 3), (3, 2), (3, 3)])
def test_padding_adds_nothing_to_infinite_sums(method, dim):
    """The entries that fill up a list's last quad add nothing, also where a
    particle's own state makes its terms infinite: 0 times infinity is not a
    number, so they may not be formed from a neighbour of no volume.  Two
    to six flow particles in a row, the first infinitely fast."""
    for n in range(2, 7):
        sc = build_scene(tiny_cfg(method=method, dim=dim, domain=(0.4, 0.4, 0.4)))
        flow = np.flatnonzero(sc.mat_type > 0)
        # the others far from the row and from each other's reach
        d, top = 2 * sc.geo.particle_radius, 0.3
        sc.pos[flow, 0] = 0.3
        sc.pos[flow[:n], :dim] = np.array([0.1, top, 0.2])[:dim] + (np.arange(n) * 0.4 * d)[:, None] / n
        sc.vel[:] = 0.0
        sc.vel[flow[0], 0] = -np.inf
        out = []
        for mode in (0, 1, 2):
            eng = L.Engine(method, dim, sc.n, sc.geo.grid_num_total, 1)
            eng.set_neighbor_list(mode)
            slot = eng.add_scene(sc.desc())
            L.upload_scene(eng, slot, sc)
            for what in ("sort", "shepard", "init_tmp", "one_step"):
                eng.run(what)
            out.append({f: eng.download(slot, f) for f in ("id0", "d_density", "d_vel")})
            if mode:
                i = np.flatnonzero(out[-1]["id0"] == flow[0])[0]
                assert eng.neighbor_lists(slot)[0][i] == n - 1
            eng.close()
        assert np.isinf(out[0]["d_density"]).any()
        for o in out[1:]:
            for f in o:
                np.testing.assert_array_equal(o[f], out[0][f], err_msg=f"{n} particles: {f}")


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("tile", [128, 512])
def test_lists_of_particles_out_of_cell_order(dim, tile):
    """Positions uploaded after the sort: the particles of a tile are in any
    order, and every list mode still walks each one's own cells."""
    sc = build_scene(tiny_cfg(dim=dim, domain=(0.3, 0.3, 0.12), block=(0.15, 0.12, 0.06)))
    for share in (0.02, 1.0):  # a few particles moved, and all
        out = []
        for mode in (0, 1, 2):
            eng = L.Engine(sc.method, dim, sc.n, sc.geo.grid_num_total, 1)
            eng.set_neighbor_list(mode)
            eng.set_cell_tile(tile)
            slot = eng.add_scene(sc.desc())
            L.upload_scene(eng, slot, sc)
            eng.run("sort")
            pos, flow = eng.download(slot, "pos"), np.flatnonzero(eng.download(slot, "type") == 1)
            rng = np.random.default_rng(4)
            some = rng.choice(flow, max(2, int(share * flow.size)), replace=False)
            pos[some] = pos[rng.permutation(some)]
            eng.upload(slot, "pos", pos)
            for what in ("shepard", "init_tmp", "one_step"):
                eng.run(what)
            out.append({f: eng.download(slot, f) for f in ("cspm_f", "d_density", "d_vel")})
            if mode:
                out[-1]["lists"] = eng.neighbor_lists(slot)
            eng.close()
        for m, o in enumerate(out[1:], 1):
            for f in out[0]:
                np.testing.assert_array_equal(o[f], out[0][f], err_msg=f"mode {m}, share {share}: {f}")
        for a, b in zip(out[1]["lists"], out[2]["lists"]):
            np.testing.assert_array_equal(a, b)


@pytest.mark.parametrize("between", [False, True])  # a step between removal and addition
@pytest.mark.parametrize("fills", [False, True])    # the new scene's cells end where the next scene's begin
def test_scene_in_a_freed_range_is_empty_until_sorted(between, fills):
    """A scene that takes the cells of a removed one has no neighbours before
    its first sort, as in a new engine, and the other scenes keep theirs."""
    low, mid, top = (shaken(2, b, s) for s, b in enumerate([(0.3, 0.2, 0.0), (0.4, 0.3, 0.0), (0.2, 0.4, 0.0)]))
    new = build_scene(tiny_cfg(dim=2, r=0.005, domain=(2.0, 1.2, 0.1) if fills else (1.0, 0.6, 0.1), block=(0.2, 0.1, 0.0)))
    assert (new.geo.grid_num_total == mid.geo.grid_num_total) == fills and new.n <= mid.n
    eng = L.Engine(1, 2, low.n + mid.n + top.n, sum(s.geo.grid_num_total for s in (low, mid, top)), 3)
    slots = []
    for sc in (low, mid, top):
        slots.append(eng.add_scene(sc.desc()))
        L.upload_scene(eng, slots[-1], sc)
    eng.step(3)
    eng.remove_scene(slots[1])
    if between:
        eng.step(1)
    eng.sync()
    keep = [slots[0], slots[2]]
    before = [eng.neighbor_stats(s) for s in keep]
    starts = [eng.download(s, "cell_start") for s in keep]
    slot = eng.add_scene(new.desc())
    L.upload_scene(eng, slot, new)
    assert not eng.download(slot, "cell_start").any()
    assert not eng.neighbor_stats(slot)[0].any()
    for s, b, c in zip(keep, before, starts):
        np.testing.assert_array_equal(eng.download(s, "cell_start"), c)
        for x, y in zip(eng.neighbor_stats(s), b):
            np.testing.assert_array_equal(x, y)
    eng.step(2)
    eng.sync()
    got = {f: eng.download(slot, f) for f in STATE}
    eng.close()
    alone = run([new], 2)
    for f in STATE:
        np.testing.assert_array_equal(got[f], alone[f], err_msg=f)


def test_residents_that_come_and_go_capture_once_per_route():
    """Scenes of any size admitted and retired: the step's graphs are captured
    once for each route of the sort."""
    small = [shaken(2, b, s) for s, b in enumerate([(0.1, 0.1, 0.0), (0.6, 0.5, 0.0)])]
    few = build_scene(tiny_cfg(r=0.005, domain=(0.3, 0.3, 0.2), block=(0.1, 0.1, 0.0)))
    large = build_scene(tiny_cfg(r=0.005, domain=(6.0, 3.0, 0.2), block=(0.2, 0.2, 0.0)))
    scenes = [few, small[0], small[1], large]
    eng = L.Engine(1, 2, sum(s.n for s in scenes), sum(s.geo.grid_num_total for s in scenes), 4)

    def add(sc):
        slot = eng.add_scene(sc.desc())
        L.upload_scene(eng, slot, sc)
        eng.step(2)
        return slot

    assert eng.kernel_time("capture")[1] == 0
    add(few)
    a, b = add(small[0]), add(small[1])
    eng.remove_scene(b)
    eng.step(1)
    assert eng.kernel_time("capture")[1] == 1
    for _ in range(3):
        c = add(large)
        eng.remove_scene(c)
        eng.step(1)
    assert eng.kernel_time("capture")[1] == 2
    got = {f: eng.download(a, f) for f in STATE}
    steps = eng.steps(a)
    eng.close()
    alone = run([small[0]], steps)
    for f in STATE:
        np.testing.assert_array_equal(got[f], alone[f], err_msg=f)


def test_sort_of_more_slots_than_workgroups():
    """An engine of more scene slots than the one-workgroup sort launches
    workgroups: the scenes left in the first and in later turns of one
    workgroup, and in others, get the bits they have alone."""
    empty = build_scene(tiny_cfg(r=0.02, domain=(0.1, 0.1, 0.1), block=(0.04, 0.04, 0.0)))
    keep = {0: shaken(2, (0.5, 0.4, 0.0), 1), 2048: shaken(2, (0.3, 0.8, 0.0), 2), 4096: shaken(2, (0.2, 0.2, 0.0), 3),
            2047: shaken(2, (0.4, 0.1, 0.0), 4), 4199: shaken(2, (0.1, 0.6, 0.0), 5)}
    scenes = [keep.get(s, empty) for s in range(4200)]
    eng = L.Engine(1, 2, sum((s.n + 63) // 64 * 64 for s in scenes), sum(s.geo.grid_num_total for s in scenes), 4200)
    for sc in scenes:
        eng.add_scene(sc.desc())
    for s in range(4200):
        if s not in keep:
            eng.remove_scene(s)
    for s, sc in keep.items():
        L.upload_scene(eng, s, sc)
    eng.step(4)
    eng.sync()
    for s, sc in keep.items():
        alone = run([sc], 4)
        for f in STATE:
            np.testing.assert_array_equal(eng.download(s, f), alone[f], err_msg=f"slot {s}: {f}")
    eng.close()


def test_read_outs_from_a_thread_on_another_device():
    """Fields, globals and the colour range are read on the engine's device,
    whatever device the calling thread has chosen, which it keeps."""
    if L.device_count() < 2:
        pytest.skip("needs two devices")
    import torch
    sc = shaken(2, (0.3, 0.3, 0.0))
    eng = L.Engine(1, 2, sc.n, sc.geo.grid_num_total, 1)
    slot = eng.add_scene(sc.desc())
    L.upload_scene(eng, slot, sc)
    eng.step(2)
    eng.assign_value_color(slot, 3)

    def read():
        return [eng.download(slot, "vel"), eng.globals(slot), np.array(eng.v_maxmin(slot))]

    here = read()
    with torch.cuda.device(1):
        there = read()
        assert torch.cuda.current_device() == 1
    eng.close()
    for a, b in zip(there, here):
        np.testing.assert_array_equal(a, b)


def test_sort_of_scenes_that_come_and_go():
    """Small scenes whose slot order is not their cell order, with a gap in
    the cells, against the same scenes beside one that forces the general
    sort: state and cell ranges of every scene."""
    a, b, c = (shaken(2, blk, s) for s, blk in enumerate([(0.4, 0.3, 0.0), (0.3, 0.5, 0.0), (0.5, 0.2, 0.0)]))
    d = build_scene(tiny_cfg(dim=2, r=0.005, domain=(1.0, 0.6, 0.1), block=(0.3, 0.2, 0.0)))
    late = build_scene(tiny_cfg(dim=2, r=0.005, domain=(2.4, 1.4, 0.1), block=(0.2, 0.3, 0.0)))
    wide = build_scene(tiny_cfg(dim=2, r=0.005, domain=(6.0, 3.0, 0.2), block=(0.2, 0.2, 0.0)))
    assert d.geo.grid_num_total < b.geo.grid_num_total and a.geo.grid_num_total < late.geo.grid_num_total
    out = []
    for general in (False, True):
        eng = L.Engine(1, 2, sum(s.n for s in (a, b, c, d, late, wide)),
                       sum(s.geo.grid_num_total for s in (a, b, c, d, late, wide)), 5)

        def add(sc):
            slot = eng.add_scene(sc.desc())
            L.upload_scene(eng, slot, sc)
            return slot

        slots = {"a": add(a), "b": add(b), "c": add(c)}
        if general:
            add(wide)
        eng.step(2)
        # the first goes; a larger one takes its slot but cells past the others'
        eng.remove_scene(slots.pop("a"))
        slots["late"] = add(late)
        eng.step(2)
        # the middle one goes; a smaller one leaves a gap in its cells
        eng.remove_scene(slots.pop("b"))
        slots["d"] = add(d)
        eng.step(2)
        eng.sync()
        out.append({(k, f): eng.download(s, f) for k, s in slots.items() for f in STATE})
        eng.close()
    assert out[0].keys() == out[1].keys()
    for k in out[0]:
        np.testing.assert_array_equal(out[0][k], out[1][k], err_msg=str(k))


@pytest.mark.parametrize("dim", [2, 3])
def test_cell_update_of_offsets_at_the_edges(dim):
    """Cell and offset after the sort, bit for bit, of offsets on and beside
    the edges of a cell: the rule floor(o / grid) in float64, whichever way
    the kernel takes.  Also -0, and in 2D a z offset that is not zero."""
    sc = build_scene(tiny_cfg(dim=dim, domain=(0.4, 0.4, 0.4), block=(0.08, 0.08, 0.08)))
    grid = sc.geo.grid_size
    top = np.float32(grid)
    while np.float64(top) >= grid:
        top = np.nextafter(top, np.float32(0))
    over = np.nextafter(top, np.float32(1))
    f = np.float32
    edges = [f(0), f(-0.0), f(1e-45), f(-1e-45), f(-1e-9), f(0.4 * grid), np.nextafter(top, f(0)), top, over,
             np.nextafter(over, f(1)), f(1.5 * grid), f(-0.5 * grid), f(-grid), f(2 * grid)]
    eng = L.Engine(sc.method, dim, sc.n, sc.geo.grid_num_total, 1)
    slot = eng.add_scene(sc.desc())
    L.upload_scene(eng, slot, sc)
    gn = np.asarray(sc.geo.grid_num)
    flow = np.flatnonzero(sc.mat_type == 1)[: len(edges) * 3]
    cell0 = np.zeros((sc.n, 3), dtype=np.int64) + np.asarray([3, 3, 3 if dim == 3 else 0])
    assert (gn[:dim] > 6).all() and flow.size == len(edges) * 3
    off0 = np.full((sc.n, 3), 0.25 * grid, dtype=np.float32)
    off0[:, 2] *= dim - 2
    for k, i in enumerate(flow):
        off0[i, (k // len(edges)) % 3] = edges[k % len(edges)]
    eng.upload(slot, "cell", (cell0[:, 0] * gn[1] + cell0[:, 1]) * gn[2] + cell0[:, 2])
    eng.upload(slot, "offset", off0)
    eng.upload(slot, "id0", np.arange(sc.n))
    eng.run("sort")
    order = np.argsort(eng.download(slot, "id0"))
    cell, off = eng.download(slot, "cell")[order], eng.download(slot, "offset")[order].astype(np.float32)
    eng.close()
    want_c, want_o = cell0.copy(), off0.copy()
    for i in range(sc.n):
        for ax in range(3):
            if dim == 2 and ax == 2:
                want_o[i, 2] = 0
                continue
            k, o = renorm(off0[i, ax], grid)
            want_c[i, ax] += k
            want_o[i, ax] = o
    np.testing.assert_array_equal(cell, (want_c[:, 0] * gn[1] + want_c[:, 1]) * gn[2] + want_c[:, 2])
    np.testing.assert_array_equal(off.view(np.uint32), want_o.view(np.uint32))


@pytest.mark.parametrize("kernel", [0, 1])
@pytest.mark.parametrize("case", ["vx", "vy", "vz", "nan_vz", "wall_vz", "large"])
def test_two_dimensions_keep_the_third_components_sums(case, kernel):
    """In 2D the third components' terms are products with 0: +-0, but not a
    number beside an infinity, which d_vel and d_density then carry (and the
    step reports).  Against the pairs' forces in numpy: where one is not finite
    the sum's third component is NaN, and nowhere else."""
    sc = build_scene(tiny_cfg(dim=2, kernel=kernel, boundary=2, domain=(0.2, 0.2, 0.1)))
    flow, wall = np.flatnonzero(sc.mat_type == 1), np.flatnonzero(sc.mat_type < 0)
    hit = int(flow[len(flow) // 2])
    rng = np.random.default_rng(2)
    sc.vel[flow, :2] = rng.uniform(-0.1, 0.1, (flow.size, 2))
    if case == "wall_vz":
        hit = int(wall[np.argmin(np.abs(sc.pos[wall] - sc.pos[flow[0]]).sum(1))])
        sc.vel[hit, 2] = np.inf
    elif case == "large":
        sc.vel[hit, 0] = 3e38  # its dot product with a distance is finite, the force may not be
    else:
        sc.vel[hit, {"vx": 0, "vy": 1}.get(case, 2)] = np.nan if case == "nan_vz" else np.inf
    got = []
    for mode in (0, 2):
        eng = L.Engine(1, 2, sc.n, sc.geo.grid_num_total, 1)
        eng.set_neighbor_list(mode)
        slot = eng.add_scene(sc.desc())
        L.upload_scene(eng, slot, sc)
        for what in ("sort", "shepard", "init_tmp", "one_step"):
            eng.run(what)
        got.append({f: eng.download(slot, f) for f in ("d_vel", "d_density", "type", "v_tmp", "density_tmp", "pressure",
                                                       "offset", "cell", "m_V")})
        eng.close()
    for f in got[0]:
        np.testing.assert_array_equal(got[0][f], got[1][f], err_msg=f)
    g = {k: v.astype(np.float32) if v.dtype.kind == "f" else v for k, v in got[0].items()}
    c = np.stack(np.unravel_index(g["cell"], np.asarray(sc.geo.grid_num)), 1)[:, :2]
    o = g["offset"][:, :2]
    desc = sc.desc()
    c2 = 0.01 * desc["smoothing_len"] ** 2
    c1, rho0 = 2.0 * 4 * desc["viscosity"], desc["density0"]
    seen = 0
    with np.errstate(all="ignore"):
        for i in np.flatnonzero(g["type"] == 1):
            # pair vector and reach as the kernels form them: zeros, signs and
            # the pairs on the edge matter
            d = (o[i] + (c[i] - c).astype(np.float32) * np.float32(sc.geo.grid_size)) - o
            r2 = (d[:, 1].astype(np.float64) ** 2 + d[:, 0] * d[:, 0]).astype(np.float32)
            j = np.flatnonzero((r2 < np.float32(desc["support_radius"]) ** 2) & (np.arange(r2.size) != i))
            u = g["v_tmp"][i] - g["v_tmp"][j]
            dot = (u[:, :2] * d[j]).sum(1) + u[:, 2] * np.float32(0)
            mn = np.where(dot < 0, dot, np.float32(0))
            rr = np.where(g["type"][j] < 0, rho0 / g["density_tmp"][i], 1.0)
            vis = (c1 * g["m_V"][j] * rr).astype(np.float32) * mn / (r2[j] + np.float32(c2))
            q = g["pressure"] / g["density_tmp"] ** 2
            sc_ = vis - np.float32(rho0) * g["m_V"][j] * (q[i] + q[j])
            bad_z = not np.isfinite(sc_).all()
            bad_uz = not np.isfinite(u[:, 2]).all()
            assert np.isnan(g["d_vel"][i, 2]) == bad_z, (i, sc_, g["d_vel"][i])
            if bad_uz:
                assert np.isnan(g["d_density"][i])
                if not bad_z:
                    assert np.isfinite(g["d_vel"][i]).all()
            seen += bad_z or bad_uz
    assert seen > 0
