"""Layers of the autoencoder near the edges of their tiles, and their weight gradients tap by tap.

The upsampling layers are computed per output phase from the coarse grid in tiles of 2 x 8 x D cells, the
output layer in columns of 8 rows, cut along y for few blocks: rough inputs and non-zero biases, so
that every tap, phase, halo and tile boundary carries weight, for one block and for odd counts.

Bounds: the device and the reference round the same operands to BF16, but their FP32 summation orders
differ by about 1e-6, so now and then an operand falls on the other side of a rounding boundary and moves by
one BF16 step, up to 2^-7 of itself.  In the last layer one such step moves an output by up to
2^-7 max|a| max|W| (a: its inputs); four times that is left for steps of earlier layers and for several at
once.  Steps are rare: over any one plane of cells the rms error stays under 2^-7 of the output's rms (27
cells at the largest step seen, 2.8 % of the rms, are 0.5 % over a plane of 1024).  A dropped or misplaced
tap of one cell is off by 1/sqrt(27) of the rms, and of one row of 32 cells by 3.4 % over the plane."""
import ctypes as C

import numpy as np
import pytest
import torch

from konglong_amd._lib import DeviceArray, check, lib
from tests import convae_ref as ref
from tests.helpers import smooth_field

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nb", [1, 2, 7])
def test_every_cell_of_rough_blocks(klrtm, nb):
    print(f"[convae] forward of {nb} rough blocks, cell by cell", flush=True)
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 21))
    rng = np.random.default_rng(900 + nb)
    p = np.empty(lib().klrtm_convae_param_count(), np.float32)
    check(lib().klrtm_convae_get_params(h.value, p.ctypes.data))
    o = 0
    for ci, co in zip(ref.CIN, ref.COUT):
        o += co * ci * 27
        p[o:o + co] = rng.uniform(-0.3, 0.3, co)
        o += co
    check(lib().klrtm_convae_set_params(h.value, p.ctypes.data))
    x = rng.standard_normal((nb, 32, 32, 32)).astype(np.float32)
    dx, rec = DeviceArray.from_host(x), DeviceArray((nb, 32, 32, 32))
    check(lib().klrtm_convae_forward(h.value, dx.ptr, nb, None, rec.ptr))
    lib().klrtm_convae_destroy(h.value)
    a7 = ref.forward(p, torch.from_numpy(x.reshape(nb, 1, 32, 32, 32)), l1=7)[0]
    want = ref.forward(p, a7, l0=7)[0].numpy().reshape(nb, 32, 32, 32)
    w7 = ref.split_params(p)[7][0]
    rms = np.sqrt(np.mean(want.astype(np.float64) ** 2))
    err = np.abs(rec.download().astype(np.float64) - want)
    planes = [np.sqrt(np.mean(err ** 2, axis=tuple(i for i in range(1, 4) if i != ax))) for ax in (1, 2, 3)]
    bound = 4.0 * 2.0 ** -7 * float(a7.abs().max()) * float(np.abs(w7).max())
    print(f"[convae] largest error {err.max():.2e} (bound {bound:.2e}), of a plane {np.max(planes):.2e} (rms {rms:.2e})",
          flush=True)
    assert err.max() <= bound
    assert np.max(planes) <= 2.0 ** -7 * rms


@pytest.mark.parametrize("nb", [1, 5, 33])
def test_weight_gradient_of_every_tap(klrtm, nb):
    """The weight gradients tap by tap against torch autograd in FP32, for one block, and for numbers of blocks
    whose tiles leave a remainder over the workgroups of the upsampling layers (64 tiles a block over 256, 8 over
    128); the other layers have a workgroup for every task of these batches.
    Bound: each of K products carries two BF16 roundings (2^-9 each) and the layers before and behind add
    theirs; the eight layers together stay within 5e-2 as in the whole-layer comparison.  A tap taken from a
    neighbouring cell is uncorrelated with its reference."""
    print(f"[convae] weight gradients of {nb} blocks, tap by tap", flush=True)
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 22))
    p = np.empty(lib().klrtm_convae_param_count(), np.float32)
    check(lib().klrtm_convae_get_params(h.value, p.ctypes.data))
    x = np.stack([smooth_field((32, 32, 32), -1.0, 1.0, 950 + i, passes=1) for i in range(nb)]).astype(np.float32)
    dx = DeviceArray.from_host(x)
    g, loss = np.empty_like(p), C.c_float()
    check(lib().klrtm_convae_loss_grad(h.value, dx.ptr, nb, g.ctypes.data, C.byref(loss)))
    lib().klrtm_convae_destroy(h.value)
    _, g_ref = ref.loss_and_grad(p, x)
    worst = 0.0
    for l, ((w, _), (w_ref, _)) in enumerate(zip(ref.split_params(g), ref.split_params(g_ref))):
        w, w_ref = (t.reshape(-1, 27).T for t in (w, w_ref))
        e = [float(np.linalg.norm(w[t] - w_ref[t]) / np.linalg.norm(w_ref[t])) for t in range(27)]
        print(f"[convae] layer {l}: largest tap error {max(e):.2e}", flush=True)
        worst = max(worst, max(e))
    assert worst < 5e-2


@pytest.mark.parametrize("nb,active", [(67, (66,)), (67, (2, 66)), (131, (130,)), (131, (2, 130)), (259, (258,)),
                                       (259, (2, 66, 130, 258))])
def test_weight_gradient_of_blocks_past_the_first_round(klrtm, nb, active):
    """Workgroups that take several tasks: 4 tiles a block of the 8^3 layers over 256 workgroups (a second task from
    block 64 on), 8 slabs of the output layer and 4 of the input layer over 1024 (from blocks 128 and 256 on).  All
    blocks but a few are zero, and so are their gradients as long as the biases are zero, so the batch's gradient
    times nb is the sum of the few blocks' own, each from a call of one block, in which no workgroup takes a second
    task.  Bound: the loss scale 1/nb moves the BF16 roundings of the gradients that pass the eight layers, 2^-9 each
    and both sides rounded: 2 * sqrt(8) * 2^-9 = 1.1e-2, and as much again for the operands of the weight gradient.
    A task that is lost or counted twice is a quarter or an eighth of one of at most four blocks: 3 % or more."""
    print(f"[convae] weight gradients of {nb} blocks, all zero but {active}", flush=True)
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 24))
    p = np.empty(lib().klrtm_convae_param_count(), np.float32)
    check(lib().klrtm_convae_get_params(h.value, p.ctypes.data))
    assert all(not b.any() for _, b in ref.split_params(p))
    rng = np.random.default_rng(nb)
    x = np.zeros((nb, 32, 32, 32), np.float32)
    want = np.zeros(p.size)
    for i in active:
        x[i] = rng.standard_normal((32, 32, 32))
    dx = DeviceArray.from_host(x)
    g, loss = np.empty_like(p), C.c_float()
    for i in active:
        check(lib().klrtm_convae_loss_grad(h.value, dx.ptr + i * 131072, 1, g.ctypes.data, C.byref(loss)))
        want += g
    check(lib().klrtm_convae_loss_grad(h.value, dx.ptr, nb, g.ctypes.data, C.byref(loss)))
    lib().klrtm_convae_destroy(h.value)
    for l, ((w, _), (v, _)) in enumerate(zip(ref.split_params(g.astype(np.float64) * nb), ref.split_params(want))):
        err = float(np.linalg.norm(w - v) / np.linalg.norm(v))
        print(f"[convae] layer {l}: {err:.2e}", flush=True)
        assert err < 2.2e-2


def test_gradient_of_a_shifted_input(klrtm):
    """A batch that starts one element into its allocation gives the same bits in the input layer's weight
    gradient (its operand is the caller's tensor; every sum it depends on runs in a fixed order)."""
    print("[convae] gradient with an input aligned to one element", flush=True)
    h = C.c_void_p()
    check(lib().klrtm_convae_create(C.byref(h), 23))
    n = lib().klrtm_convae_param_count()
    x = np.random.default_rng(77).standard_normal(2 * 32768).astype(np.float32)
    out = []
    for shift in (0, 1, 3):
        dx = DeviceArray.from_host(np.concatenate([np.zeros(shift, np.float32), x, np.zeros(4, np.float32)]))
        g, loss = np.empty(n, np.float32), C.c_float()
        check(lib().klrtm_convae_loss_grad(h.value, dx.ptr + 4 * shift, 2, g.ctypes.data, C.byref(loss)))
        out.append(ref.split_params(g)[0][0])
    lib().klrtm_convae_destroy(h.value)
    assert all(np.array_equal(o.view(np.uint32), out[0].view(np.uint32)) for o in out)
