"""Laplacian-mode determinants of more than 16 electrons (det_lap.hip) at the edges of their 16 x 16 blocks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule
from oracle import hamiltonian as oh
from oracle import wavefunction as owf

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("n,D", [(17, 1), (31, 3), (32, 2), (33, 1), (48, 2), (49, 1), (63, 1)])
def test_large_determinants_against_the_oracle(cuda, n, D):
    """E_loc and log|psi|^2 of two walkers: FP64 form against the FP64 oracle (float32 rounding of the outputs plus
    1e-13 kappa), FP32 form within the parity tests' bound."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), D)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(5), 2, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    x = r0.astype(np.float32)
    r = torch.as_tensor(x, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    u, d = shape.n_up, shape.n_dn
    kappa = owf.conditioning(params, u, d, x, R)
    lp_ref = owf.log_psi_sqr(params, u, d, torch.tensor(x), R)[1].numpy()
    e_ref = oh.local_energy(params, u, d, x, R, Z).numpy()
    for prec in ("fp64", "fp32"):
        m = NativeModel(shape, prec)
        m.set_params(params)
        e, lp = torch.empty(2, device="cuda"), torch.empty(2, device="cuda")
        m.local_energy(r, Rd, Zd, e, lp)
        torch.cuda.synchronize()
        tol = 2.0 ** -23 + 1e-13 * kappa if prec == "fp64" else 1e-4 + 4 * U32 * kappa
        assert np.all(np.abs(e.cpu().numpy() - e_ref) <= (1 + np.abs(e_ref)) * tol)
        assert np.all(np.abs(lp.cpu().numpy() - lp_ref) <= (1 + np.abs(lp_ref)) * tol)
