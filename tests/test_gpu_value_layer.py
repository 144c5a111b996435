"""The one-launch value layers and orbital GEMMs of small batches (value_layer.hip): bit-equal to the separate
kernels at every row-tile height, K split, ragged last tiles and both models."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("embedding", ["ferminet", "dpe4"])
@pytest.mark.parametrize("n,B", [(2, 1), (3, 7), (4, 256), (5, 500), (7, 255), (14, 64), (14, 129), (17, 101), (26, 64),
                                 (33, 60), (42, 63), (60, 1), (60, 64), (10, 700)])
def test_small_batch_layers_equal_the_separate_kernels(cuda, embedding, n, B):
    """log|psi|^2 and phase with the launch shapes left to the library and with fwd_main_tile / fwd_orb_tile set
    (which keeps the separate kernels); each K split of the mean product too."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    z = np.asarray(Z).astype(int)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 3, embedding=embedding, z_min=int(z.min()),
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

    for split in (0, 1, 2, 4):
        a = run(fwd_main_tile=0, fwd_orb_tile=0, fwd_mu_split=split)
        b = run(fwd_main_tile=-1, fwd_orb_tile=-1, fwd_mu_split=split)
        assert np.all(np.isfinite(a[0]))
        np.testing.assert_array_equal(b[0], a[0])
        np.testing.assert_array_equal(b[1], a[1])
