"""Laplacian-mode determinants (det_lap.hip) at the edges of their 16 x 16 blocks."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule
from oracle import wavefunction as owf

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("n,D", [(2, 1), (7, 5), (8, 1), (15, 3), (16, 7), (17, 1), (31, 3), (32, 2), (33, 1), (48, 2), (49, 1), (63, 1)])
def test_large_determinants_at_block_edges(cuda, n, D):
    """log|psi|^2 of the Laplacian pass against the FP64 oracle (FP64 form: float32 rounding of the output plus 1e-13
    kappa; FP32 form: the parity tests' bound); E_loc of a walker bit-equal in a batch (which fills the workgroups
    and XCD ranges differently) and alone, and finite.
    E_loc itself is held to the oracle at 17 to 60 electrons by the parity tests."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), D)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(5), 9, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    x = r0.astype(np.float32)
    r = torch.as_tensor(x, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    u, d = shape.n_up, shape.n_dn
    kappa = owf.conditioning(params, u, d, x, R)
    lp_ref = owf.log_psi_sqr(params, u, d, torch.tensor(x), R)[1].numpy()
    for prec in ("fp64", "fp32"):
        m = NativeModel(shape, prec)
        m.set_params(params)

        def run(y):
            e, lp = torch.empty(len(y), device="cuda"), torch.empty(len(y), device="cuda")
            m.local_energy(y, Rd, Zd, e, lp)
            torch.cuda.synchronize()
            return e.cpu().numpy(), lp.cpu().numpy()

        e, lp = run(r)
        tol = 2.0 ** -23 + 1e-13 * kappa if prec == "fp64" else 1e-4 + 4 * U32 * kappa
        assert np.all(np.isfinite(e))
        assert np.all(np.abs(lp - lp_ref) <= (1 + np.abs(lp_ref)) * tol)
        for b in (0, 4, 8):
            e1, lp1 = run(r[b:b + 1].contiguous())
            assert e1[0] == e[b] and lp1[0] == lp[b]
