"""Convolution of the dpe4 model's Laplacian pass: a walker's energy does not depend on how a batch of its size splits the
kernel (blocks of electrons and parts of the channel rows per workgroup)."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n,batches", [("fp32", 3, (600, 300, 1)), ("fp32", 14, (520, 200, 5)),
                                                 ("fp32", 20, (300, 200, 100, 2)), ("fp32", 26, (140, 60, 1)),
                                                 ("fp32", 42, (90, 40, 3)), ("fp32", 63, (20, 1)),
                                                 ("fp64", 11, (300, 100, 1)), ("fp64", 25, (60, 7)), ("fp64", 63, (5, 1))])
def test_energy_does_not_depend_on_the_split(cuda, precision, n, batches):
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R, z = R.astype(np.float32), np.asarray(Z).astype(int)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 1, embedding="dpe4", z_min=int(z.min()),
                       n_ion_types=int(z.max() - z.min() + 1))
    m = NativeModel(shape, precision)
    m.set_params(init_params(shape, n))
    r0 = init_walkers_gaussian(np.random.default_rng(1), batches[0], R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")

    def energy(y):
        e = torch.empty(len(y), device="cuda")
        m.local_energy(y.contiguous(), Rd, Zd, e)
        return e

    e = energy(r)
    assert torch.isfinite(e).all()
    for b in batches[1:]:
        assert torch.equal(energy(r[-b:]), e[-b:])
