"""COMPRESS_16 in eight-code chunks: slices whose codes start at every 16-byte phase, shorter than a chunk,
with one and several workgroups per maximum, and volumes and codes at odd addresses, bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle
from konglong_amd._lib import DeviceArray, check, lib

pytestmark = pytest.mark.gpu


class At:
    """A device array seen from an offset of some bytes."""

    def __init__(self, d, off):
        self.ptr = d.ptr + off


@pytest.mark.parametrize("shape,fo,co", [((1, 1, 1), 0, 0), ((4, 1, 3), 0, 0), ((5, 3, 5), 4, 2), ((9, 7, 13), 8, 6),
                                         ((45, 43, 21), 4, 10), ((3, 130, 127), 0, 0), ((2, 256, 64), 12, 14),
                                         ((42, 41, 200), 0, 4),
                                         # several slices a workgroup: up to 1016 samples encoding, 508 decoding
                                         ((300, 4, 8), 0, 0), ((41, 10, 16), 4, 2), ((70, 1, 31), 0, 6), ((3, 127, 8), 0, 0),
                                         ((3, 113, 9), 8, 10), ((9, 127, 4), 0, 2), ((9, 509, 1), 4, 0), ((5, 1, 1), 0, 14)])
def test_chunks_bit_exact(klrtm, shape, fo, co):
    print(f"[c16] {shape}, volume at +{fo}, codes at +{co} bytes", flush=True)
    ny, nx, nz = shape
    rng = np.random.default_rng(ny * nx * nz)
    vol = (rng.standard_normal(shape) * 10.0 ** rng.uniform(-12, 0, shape)).astype(np.float32)
    vol[0].flat[0] = 0.0
    if ny > 1:
        vol[1] = 0.0  # a silent slice
    n, nc = vol.size, lib().klrtm_nshort_volume(nz, nx, ny)
    dv, dc, do = DeviceArray((n + 4,)), DeviceArray((nc + 8,), np.uint16), DeviceArray((n + 4,))
    v, c, o = At(dv, fo), At(dc, co), At(do, fo)
    check(lib().klrtm_memcpy_h2d(v.ptr, vol.ctypes.data, vol.nbytes))
    check(lib().klrtm_compress16(v.ptr, c.ptr, nx, ny, nz))
    check(lib().klrtm_uncompress16(c.ptr, o.ptr, nx, ny, nz))
    codes, out = np.empty(nc, np.uint16), np.empty(shape, np.float32)
    check(lib().klrtm_memcpy_d2h(codes.ctypes.data, c.ptr, codes.nbytes))
    check(lib().klrtm_memcpy_d2h(out.ctypes.data, o.ptr, out.nbytes))
    ref = oracle.compress16(vol)
    assert np.array_equal(codes, np.asarray(ref).ravel())
    assert np.array_equal(out.view(np.uint32), oracle.uncompress16(ref, ny, nx, nz).view(np.uint32))
    assert not dc.download()[co // 2 + nc:].any() and not do.download()[fo // 4 + n:].any()  # nothing past the end
