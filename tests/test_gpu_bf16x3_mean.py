"""BF16x3 form: the mean product of the Laplacian pass with its spin means formed in it (large batches) against the separate
kernels, bit for bit, and a walker's energy the same in every batch."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("embedding,n,B", [("ferminet", 2, 2401), ("ferminet", 5, 1203), ("ferminet", 14, 803),
                                           ("dpe4", 9, 1201), ("ferminet", 42, 301)])
def test_fused_mean_product_equals_the_separate_kernels(cuda, embedding, n, B):
    """Over 600 tiles of 64 rows, mostly with a ragged one; lap_mu_tile >= 0 keeps the separate kernels, and so does a batch of 40."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R, z = R.astype(np.float32), np.asarray(Z).astype(int)
    dpe4 = embedding == "dpe4"
    shape = ModelShape(n, (n + 1) // 2, len(Z), 2, embedding=embedding, z_min=int(z.min()) if dpe4 else 1,
                       n_ion_types=int(z.max() - z.min() + 1) if dpe4 else 0)
    rows = B * ((3 * n + 2 + 15) // 16 * 16)
    assert rows > 600 * 64
    m = NativeModel(shape, "bf16x3")
    m.set_params(init_params(shape, n))
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")

    def run(y):
        e, lp = torch.empty(len(y), device="cuda"), torch.empty(len(y), device="cuda")
        m.local_energy(y.contiguous(), Rd, Zd, e, lp)
        return e.cpu().numpy(), lp.cpu().numpy()

    fused = run(r)
    assert np.all(np.isfinite(fused[0]))
    m.set_tuning(lap_mu_tile=0)
    separate = run(r)
    m.set_tuning(lap_mu_tile=-1)
    few = run(r[-40:])
    for a, b, c in zip(fused, separate, few):
        np.testing.assert_array_equal(a, b)
        np.testing.assert_array_equal(a[-40:], c)
