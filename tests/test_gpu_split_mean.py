"""Mean product of the split Laplacian pass: every tile of the separate kernels and the fused kernel form the same sums, so a
walker's energy is the same bits whichever its batch takes."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width1,n,rows", [(256, 4, (24700, 24500, 18000, 8100, 4000, 32)),
                                           (256, 14, (24960, 24000, 18400, 8000, 4090, 48)),
                                           (256, 42, (24960, 18300, 8000, 3000, 128)),
                                           (128, 9, (40000, 30000, 16300, 8000, 32)), (384, 6, (13000, 12000, 5000, 2500, 32)),
                                           (512, 14, (12500, 12000, 9000, 4000, 2000, 48))])
def test_energy_does_not_depend_on_the_mean_product_kernel(cuda, width1, n, rows):
    """Rows (channels of all walkers) on either side of each rule's line, down to one walker."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 1, width1=width1, n_iter=3)
    m = NativeModel(shape)
    m.set_params(init_params(shape, n))
    per = (3 * n + 2 + 15) // 16 * 16
    r0 = init_walkers_gaussian(np.random.default_rng(1), -(-rows[0] // per), R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")

    def energy(y):
        e, lp = torch.empty(len(y), device="cuda"), torch.empty(len(y), device="cuda")
        m.local_energy(y.contiguous(), Rd, Zd, e, lp)
        return e, lp

    e, lp = energy(r)
    assert torch.isfinite(e).all()
    for k in rows[1:]:
        b = max(1, k // per)
        eb, lpb = energy(r[-b:])
        assert torch.equal(eb, e[-b:]) and torch.equal(lpb, lp[-b:])
