"""Which form the local energies of a call take: the loss FP32 MFMA for whatever computes its energies, everyone else (another
thread meanwhile, the model afterwards) its own; and what the two forms share."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


def problem(n, B, embedding="ferminet"):
    R, Z = random_molecule(np.random.default_rng(n), n)
    R, z = R.astype(np.float32), np.asarray(Z).astype(int)
    dpe4 = embedding == "dpe4"
    shape = ModelShape(n, (n + 1) // 2, len(Z), 3, embedding=embedding, z_min=int(z.min()) if dpe4 else 1,
                       n_ion_types=int(z.max() - z.min() + 1) if dpe4 else 0)
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    cuda = [torch.as_tensor(np.asarray(v), dtype=torch.float32, device="cuda").contiguous() for v in (r0, R, Z)]
    return shape, init_params(shape, n), cuda


def test_the_loss_takes_fp32_energies_and_nobody_else_does(cuda):
    from deeperwin_amd._native import LAP_FP32, lap_form
    from deeperwin_amd.config import ClippingConfig
    from deeperwin_amd.hamiltonian import build_local_energy
    from deeperwin_amd.loss import build_value_and_grad_func
    from deeperwin_amd.wavefunction import NativeLogPsiSquared

    shape, params, (r, R, Z) = problem(9, 64)
    spin = (shape.n_up, shape.n_dn)
    func, other = NativeLogPsiSquared(), NativeLogPsiSquared()
    eloc = build_local_energy(func)
    split = eloc(params, spin, r, R, Z)
    with lap_form(LAP_FP32):
        fp32 = eloc(params, spin, r, R, Z)
    assert not torch.equal(split, fp32)
    assert torch.equal(build_local_energy(func, lap_form="fp32")(params, spin, r, R, Z), fp32)
    seen = []

    def in_a_thread(*a):  # the loss's energies, and another thread's taken meanwhile
        t = threading.Thread(target=lambda: seen.append(eloc(params, spin, r, R, Z)))
        t.start()
        t.join()
        return eloc(*a)

    def energies_of_the_loss(get_local_energy):
        loss = build_value_and_grad_func(func, get_local_energy, ClippingConfig(from_previous_step=False))
        return loss(params, None, spin, (r, R, Z, None))[0][1][1]["E_loc"]

    for get_local_energy in (eloc, lambda *a: eloc(*a), build_local_energy(other), in_a_thread):
        assert torch.equal(energies_of_the_loss(get_local_energy), fp32)
    assert len(seen) == 1 and torch.equal(seen[0], split)
    assert torch.equal(eloc(params, spin, r, R, Z), split)


@pytest.mark.parametrize("embedding", ["ferminet", "dpe4"])
@pytest.mark.parametrize("n,B", [(4, 300), (10, 200), (14, 200), (20, 100), (26, 60), (31, 60), (36, 40), (42, 30),
                                 (47, 30), (52, 20), (58, 20), (60, 20)])
def test_the_two_forms_share_log_psi_and_agree_in_energy(cuda, embedding, n, B):
    """Every tile height of the split kernels: log|psi|^2 bit-equal; E_loc of the median walker within 2e-6 of 1 + |E|, or
    within a quarter of the FP32 form's own error (against the FP64 form) where that is more; of any walker within the parity
    tests' bound, (1 + |E|)(1e-4 + 4 u kappa)."""
    from deeperwin_amd._native import LAP_FP32, LAP_SPLIT, NativeModel, lap_form

    shape, params, dev = problem(n, B, embedding)
    m64 = NativeModel(shape, "fp64")
    m64.set_params(params)
    e64 = torch.empty(B, device="cuda")
    m64.local_energy(*dev, e64)
    e64 = e64.cpu().numpy().astype(np.float64)
    m = NativeModel(shape)
    m.set_params(params)
    out = []
    for form in (LAP_FP32, LAP_SPLIT):
        e, lp = torch.empty(B, device="cuda"), torch.empty(B, device="cuda")
        with lap_form(form):
            m.local_energy(*dev, e, lp)
        kappa = m.conditioning(B)
        out.append((e.cpu().numpy().astype(np.float64), lp.cpu().numpy(), kappa.cpu().numpy()))
    (e0, lp0, kappa), (e1, lp1, _) = out
    np.testing.assert_array_equal(lp1, lp0)
    rel = np.abs(e1 - e0) / (1 + np.abs(e0))
    assert np.median(rel) <= max(2e-6, np.median(np.abs(e0 - e64) / (1 + np.abs(e0))) / 4)
    assert np.all(rel <= 1e-4 + 4 * 2.0 ** -24 * kappa)
