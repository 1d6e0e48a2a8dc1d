"""FD steps at the edges of the stencil kernels' tiles and y chunks, against the FP32 oracle.

The first-derivative passes work on 64 x 8 tiles (z lanes x x rows) with a ring of R+2 plane tiles, and drop the
PML code in blocks that touch no layer: grids just below, at and past a tile, fewer planes than the stencil's
radius, 2D (kernels of its own), layers on some faces only and without the cross axes.  Both sides run FP32 in different
association: a step adds at most about 6 roundings of 6e-8 of the field per cell, which four leapfrog steps
(errors grow with the square of the step count, 10 step errors in all) turn into 4e-6 relative."""
import numpy as np
import pytest

import oracle
from konglong_amd._lib import DeviceArray, ENGINE_FD, ISO, VTI, TTI
from konglong_amd.kernel import KernelCPU
from tests.helpers import rel_l2, smooth_field, tilt_axis

pytestmark = pytest.mark.gpu

# (ny, nx, nz), order, model, layer widths x1 x2 y1 y2 z1 z2, pml3d, tile (tz, tx, ychunk) or None
CASES = [
    ((1, 21, 70), 8, VTI, (5, 6, 0, 0, 4, 7), True, None),
    ((1, 33, 64), 16, TTI, (0, 0, 0, 0, 5, 5), True, None),
    ((3, 9, 65), 16, TTI, (3, 3, 0, 0, 20, 30), True, None),
    ((5, 16, 128), 8, VTI, (0, 0, 2, 2, 0, 0), True, None),
    ((40, 17, 63), 12, TTI, (0, 7, 0, 9, 0, 0), True, None),
    ((33, 8, 129), 8, TTI, (0, 0, 6, 6, 40, 40), False, None),
    ((20, 70, 20), 10, VTI, (32, 33, 8, 8, 9, 9), True, None),
    ((37, 24, 66), 16, VTI, (6, 7, 5, 8, 6, 9), True, (16, 16, 5)),
    ((37, 24, 66), 8, TTI, (6, 7, 5, 8, 6, 9), True, (128, 4, 37)),
    ((37, 40, 10), 8, VTI, (6, 7, 5, 8, 3, 4), True, (4, 128, 7)),
    ((6, 9, 65), 8, ISO, (2, 2, 2, 2, 10, 10), True, None),
    ((70, 8, 129), 16, ISO, (0, 0, 0, 20, 0, 33), True, (64, 8, 1)),
    # 2D: one layer, no layer, no cross axes, tiles of other shapes, several tiles with a rest on both axes
    ((1, 70, 129), 16, VTI, (0, 9, 0, 0, 20, 0), False, None),
    ((1, 64, 64), 12, VTI, (0, 0, 0, 0, 0, 0), True, None),
    ((1, 9, 20), 8, TTI, (2, 3, 0, 0, 5, 5), True, (16, 16, 5)),
    ((1, 41, 300), 14, TTI, (8, 8, 0, 0, 0, 31), True, (32, 16, 1)),
    ((1, 130, 33), 10, VTI, (20, 60, 0, 0, 3, 4), True, (8, 64, 1)),
]


@pytest.mark.parametrize("shape,order,model,nb,pml3d,tile", CASES,
                         ids=[f"{'x'.join(map(str, c[0]))}-FD{c[1]}-{c[2]}{'-tile' if c[5] else ''}" for c in CASES])
def test_step_at_tile_edges(klrtm, shape, order, model, nb, pml3d, tile):
    ny, nx, nz = shape
    print(f"[fd-tiles] {shape} FD{order} model {model} layers {nb} pml3d {pml3d} tile {tile}", flush=True)
    d, dt, vmax = 10.0, 8e-4, 2500.0
    m = (smooth_field(shape, 1500.0, vmax, 3) * np.float32(dt)).astype(np.float32) ** 2
    eps = dl = px = py = None
    if model != ISO:
        eps, dl = smooth_field(shape, 0.0, 0.3, 5), smooth_field(shape, 0.0, 0.15, 7)
    if model == TTI:
        px, py = tilt_axis(shape, 9)
    w1 = smooth_field(shape, -1.0, 1.0, 11, passes=2)
    w0 = (0.97 * w1).astype(np.float32)
    o = oracle.Engine(nx, ny, nz, d, d, d, ENGINE_FD, order, np.float32)
    o.set_model(m, eps, dl, px, py)
    o.set_boundary(nb, dt, vmax, pml3d=pml3d, dim_pml=3 if ny > 1 else 2)
    ow1, ow0, owr = w1.copy(), w0.copy(), np.zeros_like(w1)
    k = KernelCPU(nx, ny, nz, d, d, d, ENGINE_FD, order)
    if tile:
        k.set_tile(*tile)
    k.setModel(*[None if a is None else DeviceArray.from_host(a) for a in (m, None, dl, eps, px, py)])
    k.setPmlOptions(pml3d=pml3d)
    k.setBoundary(*nb, dt, vmax)
    g1, g0, gr = DeviceArray.from_host(w1), DeviceArray.from_host(w0), DeviceArray(shape)
    for _ in range(4):
        o.step(model, ow1, ow0, owr)
        ow0, ow1 = ow1, ow0
        k.step(model, g1, g0, gr)
        g0, g1 = g1, g0
    err = rel_l2(g1.download(), ow1)
    print(f"  rel_l2 after 4 steps = {err:.2e}", flush=True)
    assert err <= 4e-6
