"""The split form of the Laplacian pass on weights of wide range (per-column scales of the FP16 parts, and the BF16 and FP32
kernels where FP16 parts are not enough)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu
N, B, D = 14, 200, 4


def problem():
    R, Z = random_molecule(np.random.default_rng(N), N)
    R = R.astype(np.float32)
    shape = ModelShape(N, 7, len(Z), D)
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, N, 7))
    cuda = [torch.as_tensor(np.asarray(v), dtype=torch.float32, device="cuda").contiguous() for v in (r0, R, Z)]
    return shape, init_params(shape, 3), cuda


def leaf(params, suffix):
    return next(lv for p, lv in params.items() if p.endswith(suffix))


def energies(shape, params, cuda, form):
    from deeperwin_amd._native import NativeModel

    m = NativeModel(shape)
    m.set_params(params)
    m.set_lap_form(form)
    e, lp = torch.empty(B, device="cuda"), torch.empty(B, device="cuda")
    m.local_energy(*cuda, e, lp)
    return e.cpu().numpy().astype(np.float64), lp.cpu().numpy()


@pytest.mark.parametrize("power", [-24, -32, -45, 12])
def test_energy_does_not_depend_on_an_orbital_columns_scale(cuda, power):
    """The third orbital of every determinant times a power of two: every determinant gets the same factor, and each product
    and sum is scaled exactly, so that E_loc changes by roundings of the last bits only (its own, and the FP64 sum of
    logarithms': 2^-21 (1 + |E|))."""
    from deeperwin_amd._native import LAP_SPLIT

    shape, params, dev = problem()
    e0, _ = energies(shape, params, dev, LAP_SPLIT)
    for spin in ("up", "dn"):
        w = leaf(params, "bf_%s/linear_0" % spin)["w"].copy()
        w.reshape(w.shape[0], D, N)[:, :, 2] *= np.float32(2.0 ** power)
        leaf(params, "bf_%s/linear_0" % spin)["w"] = w
    e, _ = energies(shape, params, dev, LAP_SPLIT)
    assert np.all(np.abs(e - e0) <= (1 + np.abs(e0)) * 2.0 ** -21)


def small_units(params, layer, power):
    """Units 5, 77 and 200 of a layer with inputs scaled by 2^power (their tanh becomes linear) and outputs scaled back."""
    w = leaf(params, "h_el_%d/linear_0" % layer)
    w["w"], w["b"] = w["w"].copy(), w["b"].copy()
    nxt = leaf(params, "h_el_%d/linear_0" % (layer + 1))
    nxt["w"] = nxt["w"].copy()
    for u in (5, 77, 200):
        w["w"][:, u] *= np.float32(2.0 ** power)
        w["b"][u] *= np.float32(2.0 ** power)
        for block in range(3):
            nxt["w"][256 * block + u] *= np.float32(2.0 ** -power)


def large_unit(params, layer, power):
    w = leaf(params, "h_el_%d/linear_0" % layer)
    w["w"] = w["w"].copy()
    w["w"][:, 9] *= np.float32(2.0 ** power)


def large_orbitals(params, power):
    for spin in ("up", "dn"):
        lv = leaf(params, "bf_%s/linear_0" % spin)
        lv["w"] = lv["w"] * np.float32(2.0 ** power)


def quiet_units(params, layer, power):
    """The same units' outputs scaled down: inputs of the next layer that hardly count."""
    nxt = leaf(params, "h_el_%d/linear_0" % (layer + 1))
    nxt["w"] = nxt["w"].copy()
    for u in (5, 77, 200):
        nxt["w"][u] *= np.float32(2.0 ** power)


@pytest.mark.parametrize("change,args", [(small_units, (1, -8)), (small_units, (1, -24)), (small_units, (0, -32)),
                                         (small_units, (2, -24)), (large_unit, (1, 37)), (large_orbitals, (40,)),
                                         (large_orbitals, (-60,)), (quiet_units, (1, -20))],
                         ids=lambda x: x.__name__ if callable(x) else "_".join(map(str, x)))
def test_forms_agree_on_weights_of_wide_range(cuda, change, args):
    """E_loc of the split form against FP32 MFMA: within 2e-6 of 1 + |E| for the median walker (walkers near a node differ by
    more, in proportion to their conditioning), log|psi|^2 the same bits."""
    from deeperwin_amd._native import LAP_FP32, LAP_SPLIT

    shape, params, dev = problem()
    change(params, *args)
    e0, lp0 = energies(shape, params, dev, LAP_FP32)
    e, lp = energies(shape, params, dev, LAP_SPLIT)
    assert np.all(np.isfinite(e0))
    np.testing.assert_array_equal(lp, lp0)
    assert np.median(np.abs(e - e0) / (1 + np.abs(e0))) <= 2e-6
