"""The map kernel's two forms -- launches of few tiles, where every lane reads and those out of reach
read zeros, and launches of many, where only the lanes in reach read -- on both sides of the line
between them, and tiles that look up more than a wavefront's lanes of cell rows (a coarse grid).
Every map point against the FP64 oracle; tolerance as test_gpu_core.py: 1e-4 relative plus the change
of an r^2 within 0.003 bins of an edge."""
import numpy as np
import pytest

import oracle as orc

pytestmark = pytest.mark.gpu


COMPUTE_UNITS = 256   # of an MI355X; the line lies at 112 tiles per compute unit


def check(ctx, xyz, xs, box):
    ctx.set_receptor(xyz, xs)
    ctx.grid_populate(box)
    maps = ctx.grid_download()
    b, e, n = box.as_tuple()
    grid = orc.Grid(orc.Lut(), b, e, n)
    grid.set_receptor(xyz.astype(np.float64), xs)
    slack = grid.populate_with_slack(0.003)
    ref = grid.maps()
    assert (np.abs(maps - ref) <= 1e-4 * np.maximum(1.0, np.abs(ref)) + slack).all()
    return maps


# tiles are 4 x 4 x 2 points: 16 x 16 x nz / 2 of them, and one layer of 16 x 16 more
@pytest.mark.parametrize("layers_more", [0, 1])
def test_both_forms_at_the_line(module_ctx, layers_more):
    import vdock
    layers = 112 * COMPUTE_UNITS // 256 + layers_more
    steps = [63, 63, 2 * layers - 1]
    xyz, xs = vdock.synth_receptor(900, 36.0, 4.0, 11)
    box = vdock.box_from_center([2.0, -1.0, 3.0], [0.375 * s - 1e-3 for s in steps], 0.375)
    assert box.dims == (64, 64, 2 * layers)
    print("tiles", 256 * layers, flush=True)
    maps = check(module_ctx, xyz, xs, box)
    assert np.abs(maps).max() > 1


def test_more_cell_rows_than_lanes(module_ctx):
    """8 A steps: a tile reaches 24 + 2 x 8 A along y, 8 + 2 x 8 A along z, some 70 rows of 4 A cells."""
    import vdock
    xyz, xs = vdock.synth_receptor(4000, 70.0, 0.0, 12)
    box = vdock.box_from_center([0, 0, 0], [64, 64, 64], 8.0)
    assert np.abs(check(module_ctx, xyz, xs, box)).max() > 0
