"""The split-operand GEMMs of the Laplacian pass (three BF16 parts per FP32 operand, gemm_split.hip): every
tile height (1 to 12 row blocks of 16 channels per electron), ragged last tiles, both tile choices."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from deeperwin_amd.params import ModelShape, init_params
from deeperwin_amd.physics import generate_el_ion_mapping, init_walkers_gaussian, random_molecule

pytestmark = pytest.mark.gpu
U32 = 2.0 ** -24


@pytest.mark.parametrize("n,B", [(4, 513), (10, 103), (14, 49), (20, 27), (26, 17), (31, 13), (36, 9), (42, 7),
                                 (47, 5), (52, 5), (58, 5), (60, 3)])
def test_split_laplacian_matches_fp64_form_for_every_tile(cuda, n, B):
    """E_loc of the FP32 form against the FP64 form (per walker, the bound of the parity tests:
    (1 + |E|)(1e-4 + 4 u kappa), kappa the walker's conditioning), and bit-equal for every tile choice."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 3)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")

    def eloc(m):
        e, lp = torch.empty(B, device="cuda"), torch.empty(B, device="cuda")
        m.local_energy(r, Rd, Zd, e, lp)
        kappa = m.conditioning(B)
        torch.cuda.synchronize()
        return e.cpu().numpy(), lp.cpu().numpy(), kappa.cpu().numpy()

    m64 = NativeModel(shape, "fp64")
    m64.set_params(params)
    e64, _, kappa = eloc(m64)
    m = NativeModel(shape)
    m.set_params(params)
    e, lp, _ = eloc(m)
    assert np.all(np.abs(e - e64) <= (1 + np.abs(e64)) * (1e-4 + 4 * U32 * kappa))
    for choice in ({"lap_electrons": 1, "lap_cols": 128, "lap_orb_tile": 0},
                   {"lap_electrons": 0, "lap_cols": 256, "lap_orb_tile": 2}):
        m.set_tuning(**choice)
        e1, lp1, _ = eloc(m)
        np.testing.assert_array_equal(e1, e)
        np.testing.assert_array_equal(lp1, lp)
    # what the scratch held before (rows of padding channels stay as they were) does not reach the results
    for byte in (0x7E, 0xFF, 0x00):  # 8.5e37, NaN, 0
        ws = torch.full((m.workspace_bytes(B, 1),), byte, dtype=torch.uint8, device="cuda")
        m.set_workspace(ws)
        e1, lp1, _ = eloc(m)
        np.testing.assert_array_equal(e1, e)
        np.testing.assert_array_equal(lp1, lp)
    m.set_workspace(None)


@pytest.mark.parametrize("scale", [2.0 ** -20, 1.0, 2.0 ** 12])
def test_split_operands_of_any_magnitude(cuda, scale):
    """Orbital weights scaled by a power of two (E_loc does not change): the power-of-two scales of the FP16 parts
    follow the operands (bound as above)."""
    from deeperwin_amd._native import NativeModel

    n, B = 14, 21
    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, 7, len(Z), 2)
    params = init_params(shape, 3)
    for path, leaves in params.items():
        if path.endswith("bf_up/linear_0") or path.endswith("bf_dn/linear_0"):
            leaves["w"] = (leaves["w"] * np.float32(scale)).astype(np.float32)  # every orbital by one factor
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, 7))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    out = []
    for prec in ("fp64", "fp32"):
        m = NativeModel(shape, prec)
        m.set_params(params)
        e = torch.empty(B, device="cuda")
        m.local_energy(r, Rd, Zd, e)
        kappa = m.conditioning(B).cpu().numpy() if prec == "fp64" else kappa
        torch.cuda.synchronize()
        out.append(e.cpu().numpy())
    assert np.all(np.abs(out[1] - out[0]) <= (1 + np.abs(out[0])) * (1e-4 + 4 * U32 * kappa))


@pytest.mark.parametrize("n,B", [(3, 5), (4, 700), (14, 33), (14, 601), (26, 18), (45, 4)])
def test_bf16x3_mean_product_with_the_means_formed_in_it(cuda, n, B):
    """BF16x3 form: log|psi|^2 the same bits whichever kernels form the mean product (the value rows keep theirs), E_loc
    within the form's own accuracy of the other (the parity tests' bound, u = 2^-17), at both tile widths."""
    from deeperwin_amd._native import LAP_FP32, LAP_SPLIT, NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 2)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    m = NativeModel(shape, "bf16x3")
    m.set_params(params)
    out = []
    for form in (LAP_FP32, LAP_SPLIT):
        m.set_lap_form(form)
        e, lp = torch.empty(B, device="cuda"), torch.empty(B, device="cuda")
        m.local_energy(r, Rd, Zd, e, lp)
        kappa = m.conditioning(B)
        torch.cuda.synchronize()
        out.append((e.cpu().numpy(), lp.cpu().numpy(), kappa.cpu().numpy()))
    (e0, lp0, kappa), (e1, lp1, _) = out
    np.testing.assert_array_equal(lp1, lp0)
    assert np.all(np.abs(e1 - e0) <= (1 + np.abs(e0)) * (1e-4 + 4 * 2.0 ** -17 * kappa))


@pytest.mark.parametrize("n,B", [(2, 3), (4, 50), (5, 19), (7, 33), (8, 21), (9, 21)])
def test_mean_product_of_small_batches(cuda, n, B):
    """Up to four electrons of a spin and 64-column workgroups: the means of a thread formed together.  E_loc bit-equal to
    the batch repeated until it takes the 256-column workgroups (the same sums)."""
    from deeperwin_amd._native import NativeModel

    R, Z = random_molecule(np.random.default_rng(n), n)
    R = R.astype(np.float32)
    shape = ModelShape(n, (n + 1) // 2, len(Z), 2)
    params = init_params(shape, n)
    r0 = init_walkers_gaussian(np.random.default_rng(1), B, R, generate_el_ion_mapping(R, Z, n, shape.n_up))
    r = torch.as_tensor(r0, dtype=torch.float32, device="cuda").contiguous()
    Rd = torch.as_tensor(R, dtype=torch.float32, device="cuda")
    Zd = torch.as_tensor(Z, dtype=torch.float32, device="cuda")
    m = NativeModel(shape)
    m.set_params(params)

    def eloc(y):
        e = torch.empty(len(y), device="cuda")
        m.local_energy(y, Rd, Zd, e)
        return e

    rows = B * ((3 * n + 2 + 15) // 16 * 16)  # channel rows; the wide workgroups take over at 512 tiles of 48
    big = r.repeat(512 * 48 // rows + 2, 1, 1).contiguous()
    e = eloc(r)
    assert torch.isfinite(e).all()
    assert torch.equal(eloc(big)[:B], e)
