"""Injection and extraction at the edges of their workgroups against dense FP64 sums over the receivers' own taps:
plane boxes below, at and past 64 columns and 4 rows and past 65536 cells, one station, few and many (> 4096) scattered stations, gridded
stations, several depths, and the ghost mirror.

A cell's sum has at most a few hundred terms of one sign-mixed kernel product each: FP32 rounding of the terms and
of the running sum stays below 300 * 6e-8 of the largest partial sum, and the fields compare in the 2-norm, so 2e-6."""
import numpy as np
import pytest

from konglong_amd._lib import DeviceArray
from konglong_amd.receiver import Receiver
from tests.helpers import rel_l2

pytestmark = pytest.mark.gpu

CASES = [  # ny, nx, stations, depths, mirror plane
    (40, 40, 1, 1, -1), (40, 40, 1, 1, 13), (30, 90, 7, 3, -1), (64, 71, 300, 2, 12), (90, 70, 5000, 1, -1),
    (43, 64, "grid1", 1, -1), (41, 65, "grid1", 1, 12), (45, 130, "grid2", 2, -1), (42, 30, "grid1", 1, 11),
    # few and many stations on either side of 12 terms a cell (spread 6: 144 terms a station)
    (40, 40, 90, 1, 12), (40, 40, 400, 1, -1), (50, 44, 2100, 2, 13), (190, 170, 2040, 1, -1), (190, 170, 2060, 1, -1),
    # a station at every cell of a box past 65536 cells (four plane rows a workgroup): 3 rows and 5 columns left over
    (259, 261, "grid1", 1, -1), (259, 261, "grid1", 1, 12),
]


@pytest.mark.parametrize("ny,nx,ns,ndep,mirror", CASES, ids=[f"{c[0]}x{c[1]}-{c[2]}-{c[3]}dep{'-ghost' if c[4] >= 0 else ''}"
                                                            for c in CASES])
def test_inject_extract(klrtm, ny, nx, ns, ndep, mirror):
    print(f"[inject] {ny}x{nx}, {ns} stations at {ndep} depths, mirror {mirror}", flush=True)
    nz, nt, spread, dd = 48, 3, 6, 0.7
    rng = np.random.default_rng(ny + nx)
    if isinstance(ns, str):
        st = int(ns[4:])
        y, x = np.meshgrid(np.arange(0, ny, st), np.arange(0, nx, st), indexing="ij")
        xyz = np.stack([x.ravel(), y.ravel(), 14.0 + (np.arange(x.size) % ndep)], 1)
    else:
        lo = 0 if ns > 1 else 9  # (a station at the grid's rim has no taps)
        xyz = np.stack([rng.uniform(lo, nx - 1 - lo, ns), rng.uniform(lo, ny - 1 - lo, ns), 14.0 + (np.arange(ns) % ndep)], 1)
    xyz = xyz.astype(np.float32)
    r = Receiver(nx, ny, nz, xyz, spread, 0.3, 0.3, nt, dd)
    tr = rng.standard_normal((len(xyz), nt)).astype(np.float32)
    r.set_traces(tr)
    t = r.tables()
    K = [np.zeros((len(xyz), n)) for n in (nx, ny, nz)]
    for a, (k, l, o) in enumerate((("kx", "lx", "offx"), ("ky", "ly", "offy"), ("kz", "lz", "offz"))):
        for i in range(len(xyz)):
            K[a][i, t[o][i]:t[o][i] + t[l][i]] = t[k][i, :t[l][i]]
    Z = K[2].copy()
    if mirror >= 0:
        for iz in range(nz):
            if 0 <= 2 * mirror - iz < nz:
                Z[:, 2 * mirror - iz] -= K[2][:, iz]
    w = rng.standard_normal((ny, nx, nz)).astype(np.float32)
    vel = rng.uniform(0.5, 1.5, (ny, nx, nz)).astype(np.float32)
    dw, dv = DeviceArray.from_host(w), DeviceArray.from_host(vel)
    add = np.zeros((ny, nx, nz))
    for it in (1, 2):
        r.apply(dw, it, dv, 0.5, mirror)
        add += np.einsum("rz,ryx->yxz", Z, np.einsum("r,ry,rx->ryx", tr[:, it].astype(np.float64) * 0.5 * dd, K[1], K[0])) \
            if len(xyz) < 400 else sum(np.einsum("r,ry,rx,z->yxz", tr[g, it].astype(np.float64) * 0.5 * dd, K[1][g], K[0][g],
                                                 Z[g[0]], optimize=True)
                                       for g in (np.flatnonzero(xyz[:, 2] == d) for d in np.unique(xyz[:, 2])))
    got = dw.download().astype(np.float64) - w
    assert rel_l2(got, add * vel) < 2e-6 + 1e-6 * np.linalg.norm(w) / np.linalg.norm(add * vel)
    r.extract(DeviceArray.from_host(w), 0, mirror)
    P = {d: np.tensordot(w.astype(np.float64), Z[np.flatnonzero(xyz[:, 2] == d)[0]], 1) for d in np.unique(xyz[:, 2])}
    ref = np.array([K[1][i] @ P[xyz[i, 2]] @ K[0][i] for i in range(len(xyz))])
    assert rel_l2(r.record()[:, 0], ref) < 2e-6
    r.close()
