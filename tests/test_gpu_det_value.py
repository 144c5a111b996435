"""Value-pass determinants (k_det_value) at the edges of their lane groups (8, 16, 32) and of their workgroups."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule
from oracle import wavefunction as owf

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("n,D", [(2, 1), (3, 16), (8, 5), (9, 1), (13, 16), (16, 3), (17, 8), (24, 1), (31, 2), (32, 1)])
def test_value_determinants_at_group_edges(cuda, n, D):
    """log|psi|^2 against the FP64 oracle (FP64 form: float32 rounding of the output plus 1e-13 kappa; FP32 form: the
    parity tests' bound) and the sign's phase, for D that does and does not divide a workgroup's matrices (combine in
    the kernel or after it) and a batch whose last workgroup is partly filled; each walker bit-equal alone."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), D)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(6), 11, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    x = r0.astype(np.float32)
    r = torch.as_tensor(x, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    u, d = shape.n_up, shape.n_dn
    kappa = owf.conditioning(params, u, d, x, R)
    phase_ref, lp_ref = (v.numpy() for v in owf.log_psi_sqr(params, u, d, torch.tensor(x), R))
    for prec in ("fp64", "fp32"):
        m = NativeModel(shape, prec)
        m.set_params(params)

        def run(y):
            lp, ph = torch.empty(len(y), device="cuda"), torch.empty(len(y), device="cuda")
            m.logpsi(y, Rd, Zd, lp, ph)
            torch.cuda.synchronize()
            return lp.cpu().numpy(), ph.cpu().numpy()

        lp, ph = run(r)
        tol = 2.0 ** -23 + 1e-13 * kappa if prec == "fp64" else 1e-4 + 4 * U32 * kappa
        assert np.all(np.abs(lp - lp_ref) <= (1 + np.abs(lp_ref)) * tol)
        sure = tol < 0.01  # the sign of psi is determined at this precision
        assert np.all((np.cos(ph) * np.cos(phase_ref) > 0)[sure])
        for b in (0, 5, 10):
            lp1, ph1 = run(r[b:b + 1].contiguous())
            assert lp1[0] == lp[b] and ph1[0] == ph[b]
