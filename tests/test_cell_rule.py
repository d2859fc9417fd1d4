"""The cell update's shortcut: an offset in [0, grid) is one that the rule
floor((double)o / grid) leaves as it is, up to the last float below grid."""
import numpy as np


def renorm(o, grid):
    """(cell shift, offset) of the FP64 rule, from a float32 offset."""
    od = np.float64(o)
    k = np.floor(od / grid)
    r = od - k * grid
    if r >= grid:
        k, r = k + 1.0, r - grid
    on = np.float32(r)
    if on < 0:
        on = np.float32(0)
    if np.float64(on) >= grid:
        k, on = k + 1.0, np.float32(0)
    return int(k), on


def test_offsets_inside_the_cell_keep_cell_and_bits():
    rng = np.random.default_rng(7)
    grids = list(np.exp(rng.uniform(np.log(1e-5), np.log(10.0), 300))) + [0.015, 0.0015, 0.03, 1.0, 2.0 ** -7]
    for grid in grids:
        top = np.float32(grid)
        while np.float64(top) >= grid:
            top = np.nextafter(top, np.float32(0))
        o = [np.float32(0), np.float32(1e-45), np.nextafter(top, np.float32(0)), top]
        o += list((rng.random(20) * grid).astype(np.float32))
        for v in o:
            if v >= 0 and np.float64(v) < grid:
                k, on = renorm(v, grid)
                assert k == 0 and on.tobytes() == v.tobytes(), (grid, v)
