"""Compact-FD lines whose batches and chunks end at every position, bit for bit against the FP32 oracle.

The line sweeps work in batches of 12 samples forward and 8, 6 or 4 backward (by the number of streams), z lines in
chunks of 16 and steps of 8, with plain code for whole batches and checked code for the rest: the shortest lines,
lines around one to three batches, and layers narrower than a batch, as wide as one, or filling the line."""
import numpy as np
import pytest

import oracle
from konglong_amd._lib import DeviceArray, ENGINE_CFD, ISO, VTI
from konglong_amd.kernel import KernelCPU
from tests.helpers import smooth_field

pytestmark = pytest.mark.gpu

# (ny, nx, nz), model, layer widths x1 x2 y1 y2 z1 z2
CASES = [
    ((10, 10, 10), ISO, (0, 0, 0, 0, 0, 0)),
    ((11, 12, 16), VTI, (1, 2, 3, 4, 0, 1)),
    ((22, 23, 17), VTI, (8, 8, 7, 9, 0, 0)),
    ((28, 29, 21), VTI, (0, 3, 0, 16, 8, 0)),
    ((30, 34, 32), ISO, (16, 16, 15, 15, 16, 16)),
    ((35, 33, 37), VTI, (5, 2, 6, 12, 11, 5)),
    ((1, 47, 49), VTI, (9, 1, 0, 0, 17, 2)),
    ((64, 41, 65), VTI, (12, 13, 20, 24, 1, 3)),
]


@pytest.mark.parametrize("shape,model,nb", CASES, ids=["x".join(map(str, c[0])) for c in CASES])
def test_lines_of_every_remainder(klrtm, shape, model, nb):
    ny, nx, nz = shape
    print(f"[cfd-lines] {shape} model {model} layers {nb}", flush=True)
    d, dt, vmax = 10.0, 8e-4, 2500.0
    m = (smooth_field(shape, 1500.0, vmax, 3) * np.float32(dt)).astype(np.float32) ** 2
    eps = dl = None
    if model == VTI:
        eps, dl = smooth_field(shape, 0.0, 0.3, 5), smooth_field(shape, 0.0, 0.15, 7)
    w1 = smooth_field(shape, -1.0, 1.0, 11, passes=1)
    w0 = (0.97 * w1).astype(np.float32)
    o = oracle.Engine(nx, ny, nz, d, d, d, ENGINE_CFD, 10, np.float32)
    o.set_model(m, eps, dl, None, None)
    o.set_boundary(nb, dt, vmax, dim_pml=3 if ny > 1 else 2)
    ow1, ow0, owr = w1.copy(), w0.copy(), np.zeros_like(w1)
    k = KernelCPU(nx, ny, nz, d, d, d, ENGINE_CFD, 10)
    k.setModel(*[None if a is None else DeviceArray.from_host(a) for a in (m, None, dl, eps)])
    k.setBoundary(*nb, dt, vmax)
    g1, g0, gr = DeviceArray.from_host(w1), DeviceArray.from_host(w0), DeviceArray(shape)
    for it in range(3):
        o.step(model, ow1, ow0, owr)
        ow0, ow1 = ow1, ow0
        k.step(model, g1, g0, gr)
        g0, g1 = g1, g0
        bad = int(np.sum(g1.download().view(np.uint32) != ow1.view(np.uint32)))
        print(f"  step {it}: {bad} samples differ", flush=True)
        assert bad == 0
