"""The loss's FP64 statistics bit for bit: loss, clipping state and local energies (dpe4 model) against values stored in
``golden/loss_bits.npz``, local energies of ill-conditioned walkers (FermiNet) against ``golden/energy_bits.npz``.

The stored values are the library's own, from commit 9ab37b9 (``golden/make_loss_bits.py``): these quantities leave in FP64
or feed a clipping state that is carried from run to run, so kernels may be replaced but their roundings may not.
What the values should be is held by the parity tests against the oracle.
"""
from __future__ import annotations

import os

import numpy as np
import pytest

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu
FILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "loss_bits.npz")

# (embedding, electrons, determinants, walkers): up to 16, 17 to 32 and more electrons, odd counts, ragged blocks
CASES = [("dpe4", 2, 16, 30), ("dpe4", 5, 32, 19), ("dpe4", 9, 8, 13), ("dpe4", 14, 16, 12), ("dpe4", 16, 8, 9),
         ("dpe4", 17, 32, 8), ("dpe4", 26, 8, 7), ("dpe4", 33, 8, 6), ("dpe4", 42, 16, 5)]

ENERGY_FILE = os.path.join(os.path.dirname(FILE), "energy_bits.npz")

# (precision, electrons, determinants, seeded walkers, those taken): walkers whose last bit shows the order of FP64 sums
ENERGIES = [("fp32", 16, 8, 8000, (1055,)), ("fp32", 17, 8, 8000, (5569, 7831)), ("fp32", 26, 8, 4000, (3225,)),
            ("fp32", 32, 8, 2000, (1069, 1805)), ("fp32", 33, 8, 4000, (645, 925, 962, 2560, 2699)),
            ("fp32", 42, 8, 3000, (952, 2970)), ("fp32", 52, 4, 2000, (2, 54, 119, 1555)),
            ("fp32", 63, 4, 1000, (131, 257, 305, 570, 887, 968)),
            ("fp64", 14, 8, 15000, (3158, 6227)), ("fp64", 16, 8, 10000, (5816,)), ("fp64", 17, 8, 7500, (975, 1496)),
            ("fp64", 26, 8, 4000, (887, 988, 1230, 1314, 2039)), ("fp64", 33, 8, 2500, (20, 950, 1594, 2383)),
            ("fp64", 42, 8, 1500, (176,)), ("fp64", 52, 4, 1000, (54, 119, 284)), ("fp64", 63, 4, 500, (131, 257))]


def key(case) -> str:
    return "_".join(str(x) for x in case[:4])


def statistics(case):
    """(loss, clip, E_loc) of seeded parameters and walkers through the public loss."""
    import torch

    from deeperwin_amd.config import ClippingConfig
    from deeperwin_amd.hamiltonian import build_local_energy
    from deeperwin_amd.loss import build_value_and_grad_func
    from deeperwin_amd.wavefunction import NativeLogPsiSquared

    embedding, n, D, B = case
    R, Z = random_molecule(np.random.default_rng(n), n)
    R, z = R.astype(np.float32), np.asarray(Z).astype(int)
    dpe4 = embedding == "dpe4"
    shape = ModelShape(n, (n + 1) // 2, len(Z), D, embedding=embedding, z_min=int(z.min()) if dpe4 else 1,
                       n_ion_types=int(z.max() - z.min() + 1) if dpe4 else 0)
    params = init_params(shape, n)
    r = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    func = NativeLogPsiSquared(z_min=shape.z_min)
    loss = build_value_and_grad_func(func, build_local_energy(func), ClippingConfig(from_previous_step=False))
    batch = (torch.as_tensor(r, dtype=torch.float32, device="cuda").contiguous(),
             torch.as_tensor(R, dtype=torch.float32, device="cuda"),
             torch.as_tensor(np.asarray(Z), dtype=torch.float32, device="cuda"), None)
    (value, (clip, aux)), _ = loss(params, None, (shape.n_up, shape.n_dn), batch)
    return [np.asarray(x.cpu().numpy()) for x in (value, clip, aux["E_loc"])]


@pytest.mark.parametrize("case", CASES, ids=key)
def test_loss_statistics_keep_their_bits(cuda, case):
    with np.load(FILE) as g:
        want = [g[key(case) + s] for s in ("_loss", "_clip", "_eloc")]
    for got, ref in zip(statistics(case), want):
        assert got.dtype == ref.dtype
        np.testing.assert_array_equal(got, ref)


def energies(case):
    """E_loc of the case's walkers, in the form that the loss takes."""
    import torch

    from deeperwin_amd._native import LAP_FP32, NativeModel

    precision, n, D, B, rows = case
    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), D)
    m = NativeModel(shape, precision)
    m.set_params(init_params(shape, n))
    m.set_lap_form(LAP_FP32)
    r = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r[list(rows)], dtype=torch.float32, device="cuda").contiguous()
    e = torch.empty(len(r), device="cuda")
    m.local_energy(r, torch.as_tensor(R, device="cuda"), torch.as_tensor(np.asarray(Z), dtype=torch.float32, device="cuda"), e)
    return e.cpu().numpy()


@pytest.mark.parametrize("case", ENERGIES, ids=key)
def test_energies_of_ill_conditioned_walkers_keep_their_bits(cuda, case):
    with np.load(ENERGY_FILE) as g:
        np.testing.assert_array_equal(energies(case), g[key(case)])
