"""The upsampling layers of the autoencoder keep every bit that FP32 accumulation of their 27 products holds.

One channel, constant input 16 (the layer before has zero weights and bias 16, and GELU(16) = 16), and three taps
1, 2^-9 and 2^-20 at offsets 0 and +1: their products sum to 16 + 2^-5 + 2^-16, 21 bits, exact in FP32 in any order.
The bias takes away 16 + 2^-5, so the pre-activation is 2^-16 where all three taps lie inside the grid, and the
output, behind GELU (x/2 near zero) and layers that pass one tap on, is 2^-17 (2^-18 behind one GELU more).  Weights
that are summed before they meet the activation and kept in 16 bits lose the third tap."""
import ctypes as C

import numpy as np
import pytest

from konglong_amd._lib import DeviceArray, check, lib
from tests import convae_ref as ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layer", [5, 6])
@pytest.mark.parametrize("taps", [((1, 1, 1), (1, 1, 2), (1, 2, 1)), ((1, 1, 1), (2, 1, 1), (2, 2, 2)),
                                  ((1, 1, 1), (0, 1, 1), (1, 0, 0))], ids=["yz", "diagonal", "low"])
def test_no_bit_of_a_weight_sum_is_lost(klrtm, layer, taps):
    print(f"[convae] layer {layer}, taps {taps}", flush=True)
    p = np.zeros(lib().klrtm_convae_param_count(), np.float32)
    par = ref.split_params(p)  # views
    par[layer - 1][1][0] = 16.0
    for t, w in zip(taps, (1.0, 2.0 ** -9, 2.0 ** -20)):
        par[layer][0][(0, 0) + t] = w
    par[layer][1][0] = -(16.0 + 2.0 ** -5)
    for l in range(layer + 1, 8):
        par[l][0][0, 0, 1, 1, 1] = 1.0
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 1))
    check(lib().klrtm_convae_set_params(h.value, p.ctypes.data))
    x, rec = DeviceArray((2, 32, 32, 32)), DeviceArray((2, 32, 32, 32))
    check(lib().klrtm_convae_forward(h.value, x.ptr, 2, None, rec.ptr))
    lib().klrtm_convae_destroy(h.value)
    got = rec.download()[:, 2:-2, 2:-2, 2:-2]  # cells whose taps all lie inside the layer's output grid
    want = 2.0 ** (-17 if layer == 6 else -18)
    assert np.all(np.abs(got - want) < 1e-3 * want), (float(got.min()) / want, float(got.max()) / want)


@pytest.mark.parametrize("nb", [5, 9, 17, 33, 65])
def test_a_block_does_not_depend_on_the_batch(klrtm, nb):
    """How many workgroups share a tile follows from the number of blocks (8 for one block; with these numbers every
    other choice of the three layers); each output's products are added in the same order all the same."""
    print(f"[convae] {nb} blocks at once and one by one", flush=True)
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 31))
    x = np.random.default_rng(nb).standard_normal((nb, 32, 32, 32)).astype(np.float32)
    dx, rec, one = DeviceArray.from_host(x), DeviceArray(x.shape), DeviceArray(x.shape)
    check(lib().klrtm_convae_forward(h.value, dx.ptr, nb, None, rec.ptr))
    for b in range(nb):
        check(lib().klrtm_convae_forward(h.value, dx.ptr + b * 131072, 1, None, one.ptr + b * 131072))
    lib().klrtm_convae_destroy(h.value)
    assert np.array_equal(rec.download().view(np.uint32), one.download().view(np.uint32))
