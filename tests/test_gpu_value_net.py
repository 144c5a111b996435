"""Value layers of larger batches, all layers in one launch (k_value_net): bit-equal to the separate kernels at every
row-tile height, with partly filled last workgroups, both models, the gradient's kept activations and the value rows
of the Laplacian pass."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("embedding", ["ferminet", "dpe4"])
@pytest.mark.parametrize("n,B", [(2, 2100), (4, 3001), (6, 3000), (9, 1000), (14, 500), (14, 1030), (14, 2049), (17, 501),
                                 (25, 700), (30, 250), (42, 257), (42, 500), (60, 130)])
def test_larger_batch_layers_equal_the_separate_kernels(cuda, embedding, n, B):
    """log|psi|^2, phase and parameter gradient with the launch shapes left to the library and with fwd_main_tile set
    (which keeps the separate kernels), each K split of the mean product; E_loc of the first and last walkers equal in
    the batch and on their own."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    z = np.asarray(Z).astype(int)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 2, embedding=embedding, z_min=int(z.min()),
                       n_ion_types=int(z.max() - z.min() + 1) if embedding == "dpe4" else 0)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(3), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    m = NativeModel(shape)
    m.set_params(params)

    def run(**tuning):
        m.set_tuning(**tuning)
        lp, ph = torch.empty(B, device="cuda"), torch.empty(B, device="cuda")
        m.logpsi(r, Rd, Zd, lp, ph)
        torch.cuda.synchronize()
        return lp.cpu().numpy(), ph.cpu().numpy()

    for split in (0, 1, 4):
        a = run(fwd_main_tile=0, fwd_mu_split=split)
        b = run(fwd_main_tile=-1, fwd_mu_split=split)
        assert np.all(np.isfinite(a[0]))
        np.testing.assert_array_equal(b[0], a[0])
        np.testing.assert_array_equal(b[1], a[1])

    w = torch.linspace(-1, 1, B, device="cuda")
    m.set_tuning(fwd_main_tile=0, fwd_mu_split=0)
    g0 = m.param_grad(r, Rd, Zd, w).clone() if n <= 52 else None  # the gradient takes up to 52 electrons
    m.set_tuning(fwd_main_tile=-1, fwd_mu_split=0)
    assert g0 is None or torch.equal(m.param_grad(r, Rd, Zd, w), g0)

    if n <= 17:
        def energy(y):
            e = torch.empty(len(y), device="cuda")
            m.local_energy(y.contiguous(), Rd, Zd, e)
            return e
        e = energy(r)
        assert torch.equal(energy(r[:5]), e[:5]) and torch.equal(energy(r[-5:]), e[-5:])
