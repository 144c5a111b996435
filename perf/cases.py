"""The work of this framework, as cases that can be timed and checked.

The framework evaluates neural wavefunctions for variational Monte Carlo: a Metropolis-Hastings chain over
walkers (`run_mcmc_steps`), log|psi|^2 of given walkers, their local energies with the full Laplacian
(`build_local_energy`) and the clipped-energy loss with its parameter gradient (`build_value_and_grad_func`).
Each case is one such call through the public Python interface, from a handful of electrons (where a call is a
few launches long) to 42, for both wavefunction models, every precision form that is used in earnest and
Gaussian and Langevin proposals.

Inputs are what the calls meet in a run: biases and envelopes that differ from orbital to orbital as after some
training, and walkers that have left their Gaussian starting points along a short Metropolis chain in the same
wavefunction (formed here with plain torch, so that the inputs depend on the seed alone).
"""
import math

import numpy as np
import torch

from deeperwin_amd.config import (ClippingConfig, MCMCConfig, MCMCLangevinProposalConfig, MCMCSimpleProposalConfig,
                                  ModelConfigDeepErwin4, ModelConfigFermiNet, OrbitalsConfigFermiNet, PhysicalConfig)
from deeperwin_amd.hamiltonian import build_local_energy
from deeperwin_amd.loss import build_value_and_grad_func
from deeperwin_amd.mcmc import MCMCState, MetropolisHastingsMonteCarlo, make_chain
from deeperwin_amd.physics import geometry_c4h2, geometry_lih, geometry_n2, init_walkers_gaussian, random_molecule
from deeperwin_amd.wavefunction import build_log_psi_squared

BURN_IN = 30          # Metropolis steps of prepare()'s walkers
MOST_FLOPS = 1.6e12  # of a drawn case; a chain counts twice and FP64 five times, as they take longer


# --------------------------------------------------------------------------------------------------------
# The cases
# --------------------------------------------------------------------------------------------------------

def _case(op, molecule, n_el, n_det, walkers, name=None, steps=0, model="ferminet", precision="fp32",
          proposal="normal"):
    c = dict(op=op, molecule=molecule, n_el=n_el, n_det=n_det, walkers=walkers, steps=steps, model=model,
             precision=precision, proposal=proposal)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest run: LiH, few walkers; launches and host work decide
        _case("mcmc", "lih", 4, 4, 256, "mcmc_lih_256", steps=10),
        _case("eloc", "lih", 4, 4, 256, "eloc_lih_256"),
        # the inner loop of an N2 run: 20 steps between energies, then the local energy of every walker
        _case("mcmc", "n2", 14, 16, 2048, "mcmc_n2_2048", steps=20),
        _case("eloc", "n2", 14, 16, 2048, "eloc_n2_2048"),
        # one optimisation step's loss and gradient on the same molecule
        _case("grad", "n2", 14, 16, 2048, "grad_n2_2048"),
        # the same energies in the reduced and in the reference precision
        _case("eloc", "n2", 14, 16, 1000, "eloc_n2_bf16x3_1000", precision="bf16x3"),
        _case("eloc", "n2", 14, 16, 256, "eloc_n2_fp64_256", precision="fp64"),
        # the reference's default model: energies, and a chain with its Langevin proposal, ragged sizes
        _case("eloc", "n2", 14, 16, 1024, "eloc_dpe4_n2_1024", model="dpe4"),
        _case("mcmc", "random", 17, 8, 500, "mcmc_dpe4_17el_500", steps=10, model="dpe4", proposal="langevin"),
        # energies of a larger molecule, the largest case
        _case("eloc", "c4h2", 26, 16, 1024, "eloc_c4h2_1024"),
        # the largest molecules of a batch of geometries: energies, and log|psi|^2 of given walkers
        _case("eloc", "random", 42, 8, 192, "eloc_42el_192"),
        _case("logpsi", "random", 42, 8, 512, "logpsi_42el_512"),
    ]


def draw(rng):
    while True:
        op = rng.choice(["mcmc", "mcmc", "eloc", "eloc", "eloc", "grad", "logpsi"])
        molecule = rng.choice(["lih", "n2", "c4h2", "random", "random", "random", "random"])
        n = {"lih": 4, "n2": 14, "c4h2": 26}.get(molecule) or round(math.exp(rng.uniform(math.log(4), math.log(42))))
        precision = rng.choice(["fp32"] * 5 + ["bf16x3", "fp64"]) if op in ("eloc", "logpsi") else "fp32"
        c = _case(op, molecule, n, rng.choice([4, 8, 16, 16, 32]),
                  round(math.exp(rng.uniform(math.log(48), math.log(2048)))),
                  steps=rng.randint(5, 20) if op == "mcmc" else 0,
                  model=rng.choice(["ferminet", "ferminet", "ferminet", "dpe4"]), precision=precision,
                  proposal=rng.choice(["normal", "normal", "langevin"]) if op == "mcmc" else "normal")
        if work(c)["flops"] * (5 if precision == "fp64" else 2 if op == "mcmc" else 1) <= MOST_FLOPS:
            return c


def _geometry(case):
    if case["molecule"] == "lih":
        R, Z = geometry_lih()
    elif case["molecule"] == "n2":
        R, Z = geometry_n2()
    elif case["molecule"] == "c4h2":
        R, Z = geometry_c4h2(3)
    else:  # a neutral molecule of H, C, N and O with this many electrons
        R, Z = random_molecule(np.random.default_rng(case["n_el"]), case["n_el"])
    return np.asarray(R, np.float32).astype(np.float64), np.asarray(Z)


def work(case):
    """Multiply-adds that the wavefunction's layers cannot do without (spin means multiplied once per walker,
    not once per electron), times the 3 n + 2 derivative channels of a local energy."""
    n, D, B, L, W1, E = case["n_el"], case["n_det"], case["walkers"], 4, 256, 32
    n_ion = len(_geometry(case)[1])
    value = lap = 0.0
    C = 3 * n + 2
    for l in range(L):
        d, e = (4 * n_ion, 4) if l == 0 else (W1, E)
        layer = 2.0 * n * (d + 2 * e) * W1 + 2.0 * 2 * d * W1
        pairs = 2.0 * n * n * e * E if l < L - 1 else 0.0
        if case["model"] == "dpe4":
            pairs = 2 * pairs + 2.0 * n * d * E + 2.0 * n * n * E
        value += layer + pairs
        lap += C * layer + 5 * pairs
    orbitals = 2.0 * n * W1 * D * n
    value += orbitals + D * 2 / 3 * n ** 3
    lap += C * orbitals + D * (2 * n ** 3 + 3 * n * 2.0 * n ** 3)
    weights = 4.0 * (W1 * (3 * 4 * n_ion + 8) + 3 * W1 * (3 * W1 + 2 * E) + 2 * W1 * D * n + 4 * n_ion * D * n)
    flops, nbytes = {
        "mcmc": ((case["steps"] + 1) * value, 4.0 * (6 * n + 4 + 4 * case["steps"] * (3 * n + 1) / 4)),
        "logpsi": (value, 4.0 * (3 * n + 2)),
        "eloc": (lap, 4.0 * (3 * n + 2)),
        "grad": (lap + 3 * value, 4.0 * (3 * n + 3)),
    }[case["op"]]
    return {"bytes": B * nbytes + weights * (2 if case["op"] == "grad" else 1), "flops": B * flops}


# --------------------------------------------------------------------------------------------------------
# prepare and run
# --------------------------------------------------------------------------------------------------------

def _problem(case, seed):
    """What both prepare() and exact() start from: the wavefunction object, its parameters and the molecule."""
    R, Z = _geometry(case)
    phys = PhysicalConfig(R=R.tolist(), Z=[int(z) for z in Z])
    cfg = (ModelConfigDeepErwin4 if case["model"] == "dpe4" else ModelConfigFermiNet)(
        orbitals=OrbitalsConfigFermiNet(n_determinants=case["n_det"]))
    func, _, _, params, fixed = build_log_psi_squared(cfg, phys, rng_seed=seed, precision=case["precision"])
    rng = np.random.default_rng(seed + 1)
    for leaves in params.values():
        for k in leaves:
            if k == "b":
                leaves[k] = (0.3 * rng.standard_normal(leaves[k].shape)).astype(np.float32)
            elif k.startswith("alpha"):
                leaves[k] = rng.uniform(0.2, 2.0, leaves[k].shape).astype(np.float32)
            elif k.startswith("weights"):
                leaves[k] = (1.0 + 0.3 * rng.standard_normal(leaves[k].shape)).astype(np.float32)
    return func, params, fixed, phys, R, Z


def _walkers(case, seed, params, phys, R, Z):
    """Walkers after BURN_IN Metropolis steps from the Gaussian initialisation (float32)."""
    n, u, B = phys.n_electrons, phys.n_up, case["walkers"]
    r = torch.tensor(init_walkers_gaussian(np.random.default_rng(seed + 2), B, R, phys.el_ion_mapping),
                     dtype=torch.float32, device="cuda")
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 3)
    psi = _Psi(params, n, u, R, Z, torch.float32)
    lp = psi.log_psi_sqr(r)
    step = 0.45 / math.sqrt(n)
    for _ in range(BURN_IN):
        rn = r + step * torch.randn(r.shape, generator=gen, device="cuda")
        lpn = psi.log_psi_sqr(rn)
        take = torch.exp(lpn - lp) > torch.rand(B, generator=gen, device="cuda")
        r = torch.where(take[:, None, None], rn, r)
        lp = torch.where(take, lpn, lp)
    return r.contiguous()


def _proposal(case):
    return MCMCLangevinProposalConfig() if case["proposal"] == "langevin" else MCMCSimpleProposalConfig()


def _stepsize(case):
    return 0.1 if case["proposal"] == "langevin" else 0.02


def prepare(case, seed):
    func, params, fixed, phys, R, Z = _problem(case, seed)
    r = _walkers(case, seed, params, phys, R, Z)
    dev = dict(device="cuda", dtype=torch.float32)
    s = dict(case=case, func=func, params=params, fixed=fixed, spin=(phys.n_up, phys.n_dn), r=r,
             R=torch.tensor(R, **dev), Z=torch.tensor(Z, **dev))
    if case["op"] == "mcmc":
        gen = torch.Generator(device="cuda")
        gen.manual_seed(seed + 4)
        s["mc"] = MetropolisHastingsMonteCarlo(MCMCConfig(n_walkers=case["walkers"], proposal=_proposal(case),
                                                          stepsize_update_interval=7))
        s["state"] = MCMCState(r=r, R=s["R"], Z=s["Z"], log_psi_sqr=torch.full((case["walkers"],), -1000.0, **dev),
                               walker_age=torch.zeros(case["walkers"], dtype=torch.int32, device="cuda"),
                               rng_state=gen, chain=make_chain(_stepsize(case)))
    if case["op"] in ("eloc", "grad"):
        s["eloc"] = build_local_energy(func)
    if case["op"] == "grad":
        s["loss"] = build_value_and_grad_func(func, s["eloc"], ClippingConfig(from_previous_step=False))
    return s


def run(state):
    op, func, params, (up, dn) = state["case"]["op"], state["func"], state["params"], state["spin"]
    if op == "mcmc":
        new = state["mc"].run_mcmc_steps(func, state["state"], params, up, dn, state["fixed"], state["case"]["steps"])
        return dict(r=new.r, log_psi_sqr=new.log_psi_sqr, age=new.walker_age, acceptance=new.last_acceptance,
                    chain=new.chain)
    if op == "logpsi":
        phase, lp = func(params, up, dn, state["r"], state["R"], state["Z"], state["fixed"])
        return dict(phase=phase, log_psi_sqr=lp)
    if op == "eloc":
        e, flags = state["eloc"](params, (up, dn), state["r"], state["R"], state["Z"], state["fixed"],
                                 return_flags=True)
        return dict(E_loc=e, flags=flags)
    (loss, (clip, aux)), grads = state["loss"](params, None, (up, dn), (state["r"], state["R"], state["Z"],
                                                                         state["fixed"]))
    packed = torch.cat([g.reshape(-1) for leaves in grads.values() for g in leaves.values()])
    return dict(loss=loss, clip=clip, E_loc=aux["E_loc"], grads=packed)


# --------------------------------------------------------------------------------------------------------
# exact: the same quantities in 64 bits with plain torch
# --------------------------------------------------------------------------------------------------------

def exact(case, seed):
    _, params, _, phys, R, Z = _problem(case, seed)
    r32 = _walkers(case, seed, params, phys, R, Z)
    r = r32.double()
    psi = _Psi(params, phys.n_electrons, phys.n_up, R, Z, torch.float64)
    if case["op"] == "logpsi":
        lp, sign = psi.log_psi_sqr(r, with_sign=True)
        return dict(phase=torch.where(sign < 0, math.pi, 0.0).double(), log_psi_sqr=lp)
    if case["op"] == "mcmc":
        return _exact_chain(case, seed, psi, r32)
    e = psi.local_energy(r)
    if case["op"] == "eloc":
        return dict(E_loc=e, flags=None)
    center, width = e.mean(), 5.0 * e.std(unbiased=False)
    ec = center + torch.tanh((e - center) / width) * width
    loss = ec.mean()
    clip = torch.stack([loss, 5.0 * (ec - loss).square().mean().sqrt()])
    leaves = [(p, k) for p, lv in psi.params.items() for k in lv]
    for p, k in leaves:
        psi.params[p][k].requires_grad_(True)
    per = max(1, 20_000_000 // (phys.n_electrons ** 2 * 256))
    for b in range(0, len(r), per):
        ((ec - loss)[b:b + per] / len(r) * psi.log_psi_sqr(r[b:b + per])).sum().backward()
    return dict(loss=loss, clip=clip, E_loc=e, grads=torch.cat([psi.params[p][k].grad.reshape(-1) for p, k in leaves]))


def _exact_chain(case, seed, psi, r32):
    """The chain in 64 bits with the draws of the sampler's generator (per-electron normals of every step, then
    the uniforms); ages and the chain record are whole numbers and are compared as they are."""
    B, n, S = case["walkers"], case["n_el"], case["steps"]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed + 4)
    xi = torch.randn((S, B, n, 3), generator=gen, device="cuda", dtype=torch.float32).double()
    uni = torch.rand((S, B), generator=gen, device="cuda", dtype=torch.float32).double()
    r, step, rate, acc = r32.double(), float(np.float32(_stepsize(case))), 0.0, []
    lp = psi.log_psi_sqr(r)
    pc = _proposal(case)
    for k in range(S):
        if case["proposal"] == "langevin":
            def local(x):
                diff = x[:, :, None] - psi.R
                dist = diff.norm(dim=-1)
                s = step * dist.amin(-1).clamp(pc.r_min, pc.r_max)
                return s[..., None], -pc.langevin_scale * (psi.Z[:, None] * diff / dist[..., None]).sum(-2)
            s, g = local(r)
            rn = (r + xi[k] * s + g * s * s).float().double()
            sn, gn = local(rn)
            lq = (3 * torch.log(s / sn) + 0.5 * ((rn - r - g * s * s).square().sum(-1, True) / s ** 2
                                                  - (r - rn - gn * sn * sn).square().sum(-1, True) / sn ** 2))
            lq = lq.sum((1, 2))
        else:
            rn, lq = (r + xi[k] * step).float().double(), 0.0
        lpn = psi.log_psi_sqr(rn)
        take = torch.exp(lpn - lp + lq) > uni[k]
        r, lp = torch.where(take[:, None, None], rn, r), torch.where(take, lpn, lp)
        acc.append(take.double().mean())
        old, rate = rate, 0.9 * rate + 0.1 * float(acc[-1])
        if (k + 1) % 7 == 0:
            step = float(np.float32(min(1.0, max(1e-2, step / 1.05 if old < 0.5 else step * 1.05))))
    return dict(r=r, log_psi_sqr=lp, age=None, acceptance=torch.stack(acc), chain=None)


class _Psi:
    """log|psi|^2 and the local energy of both models in plain torch.

    Activations are [walker, electron, channel, feature]: channel 0 the value and, for a local energy, 3 n
    tangents (one per electron and axis) and the Laplacian.  What depends on one electron's position or on one
    pair's difference vector alone is held in 5 channels (value, 3 derivatives, Laplacian) until it is summed."""

    def __init__(self, params, n, n_up, R, Z, dtype):
        dev = dict(device="cuda", dtype=dtype)
        self.params = {p: {k: torch.as_tensor(np.asarray(v)).to(**dev) for k, v in lv.items()}
                       for p, lv in params.items()}
        self.R, self.Z = torch.tensor(R, **dev), torch.tensor(Z, **dev)
        self.n, self.u, self.dtype = n, n_up, dtype
        self.spin = (torch.arange(n, device="cuda") >= n_up).long()
        self.z = torch.tensor(np.asarray(Z) - int(np.min(Z)), device="cuda")
        self.dpe4 = any("symm_features_0" in p for p in params)
        self.L = sum(p.split("/")[-2].startswith("h_el_") and p.split("/")[-2].count("_") == 2 and
                     p.split("/")[-2][5:].isdigit() for p in params if p.endswith("linear_0"))

    def _leaf(self, suffix, leaf):
        return next(lv[leaf] for p, lv in self.params.items() if ("/" + p).endswith("/" + suffix))

    def _dense(self, module, x):
        """tanh(x W + b) along channels: [value, first derivatives..., Laplacian] at axis -2, or the value alone."""
        z = x @ self._leaf(module + "/linear_0", "w")
        z0 = z[..., :1, :] + self._leaf(module + "/linear_0", "b")
        t = torch.tanh(z0)
        if z.shape[-2] == 1:
            return t
        d1 = 1 - t * t
        zk = z[..., 1:-1, :]
        return torch.cat([t, d1 * zk, d1 * z[..., -1:, :] - 2 * t * d1 * zk.square().sum(-2, keepdim=True)], -2)

    @staticmethod
    def _distance(diff, lap, zero=None):
        """[|d|, d] of difference vectors [..., 3] in 1 or 5 channels (the Laplacian for one moving end)."""
        dist = diff.norm(dim=-1) if zero is None else torch.where(zero, 0.0, torch.where(zero[..., None], 1.0, diff).norm(dim=-1))
        value = torch.cat([dist[..., None], diff], -1)[..., None, :]
        if not lap:
            return value
        safe = dist if zero is None else torch.where(zero, 1.0, dist)
        unit = diff / safe[..., None]
        eye = torch.eye(3, dtype=diff.dtype, device=diff.device).expand(*diff.shape[:-1], 3, 3)
        second = torch.zeros_like(value)
        second[..., 0, 0] = 2.0 / safe if zero is None else torch.where(zero, 0.0, 2.0 / safe)
        if zero is not None:
            eye = torch.where(zero[..., None, None], torch.zeros_like(eye), eye)
        return torch.cat([value, torch.cat([unit[..., None], eye], -1), second], -2)

    def _own(self, x):
        """One electron's 5 channels [b, i, 5, f] at that electron's places among all channels."""
        if x.shape[-2] == 1:
            return x
        b, n, _, f = x.shape
        tan = torch.zeros(b, n, n, 3, f, dtype=x.dtype, device=x.device)
        i = torch.arange(n, device=x.device)
        tan[:, i, i] = x[:, :, 1:4]
        return torch.cat([x[:, :, :1], tan.reshape(b, n, 3 * n, f), x[:, :, 4:]], -2)

    def _pair_sum(self, x, weight):
        """sum_j weight_j x[i, j] of pair channels [b, i, j, 5, f] (r_j - r_i) in all channels of electron i."""
        x = x * weight[:, None, None]
        if x.shape[-2] == 1:
            return x.sum(2)
        b, n, _, _, f = x.shape
        tan = x[:, :, :, 1:4].clone()
        i = torch.arange(n, device=x.device)
        tan[:, i, i] -= x[:, :, :, 1:4].sum(2)
        return torch.cat([x[..., 0, :].sum(2)[:, :, None], tan.reshape(b, n, 3 * n, f),
                          2 * x[..., 4, :].sum(2)[:, :, None]], 2)

    def _convolve(self, w, hm):
        """sum_j w[i, j] * hm[j]: w in pair channels, hm [b, j, c, f] in all channels."""
        if hm.shape[-2] == 1:
            return (w * hm[:, None]).sum(2)
        b, n, c, f = hm.shape
        h0 = hm[:, None, :, 0]
        value = (w[..., 0, :] * h0).sum(2)
        tan = torch.einsum("bijf,bjcf->bicf", w[..., 0, :], hm[:, :, 1:-1]).reshape(b, n, n, 3, f)
        g = w[..., 1:4, :]
        gh = g * h0[..., None, :]
        i = torch.arange(n, device=hm.device)
        tan = tan + gh
        tan[:, i, i] -= gh.sum(2)
        ht = hm[:, :, 1:-1].reshape(b, n, n, 3, f)                          # [b, j, e, axis, f]
        cross = (g * (ht[:, i, i][:, None] - ht.transpose(1, 2))).sum((2, 3))
        lap = (w[..., 0, :] * hm[:, None, :, -1] + 2 * w[..., 4, :] * h0).sum(2) + 2 * cross
        return torch.cat([value[:, :, None], tan.reshape(b, n, 3 * n, f), lap[:, :, None]], 2)

    def _orbitals(self, r, lap):
        """Orbital matrices [b, channel, det, electron, orbital]."""
        b, n, u = r.shape[0], self.n, self.u
        ei = self._distance(r[:, :, None] - self.R, lap)                     # [b, i, I, 1 or 5, 4]
        h = self._own(ei.transpose(2, 3).reshape(b, n, ei.shape[3], -1))
        zero = torch.eye(n, dtype=torch.bool, device=r.device)
        ee = self._distance(r[:, None] - r[:, :, None], lap, zero)          # [b, i, j, ., 4], r_j - r_i
        one = torch.ones(n, dtype=self.dtype, device=r.device)
        up, dn = one * (self.spin == 0) / u, one * (self.spin == 1) / (n - u)
        same = (self.spin[:, None] == self.spin[None])[..., None, None]
        if self.dpe4:
            ee = ee[..., :1]
        for l in range(self.L):
            mean = [h[:, s].mean(1, keepdim=True).expand_as(h) for s in (slice(0, u), slice(u, n))]
            if self.dpe4:
                conv = "symm_features_%d/convolutional_features/" % l
                w = torch.where(same, self._dense(conv + "w_same", ee), self._dense(conv + "w_diff", ee))
                table = self._leaf("input/h_ion", "embeddings")[self.z]
                him = torch.tanh(table @ self._leaf(conv + "h_ion_map/linear_0", "w")
                                 + self._leaf(conv + "h_ion_map/linear_0", "b"))
                extra = [self._convolve(w, self._dense(conv + "h_map", h)), self._own((ei * him[:, None]).sum(2))]
            else:
                extra = [self._pair_sum(ee, up), self._pair_sum(ee, dn)]
            h = self._dense("h_el_%d" % l, torch.cat([h, *mean, *extra], -1))
            if l == self.L - 1:
                break

            def res(module, x):
                y = self._dense("%s_%d" % (module, l), x)
                return (x + y) / math.sqrt(2.0) if x.shape == y.shape else y
            if self.dpe4:
                ee, ei = torch.where(same, res("h_same", ee), res("h_diff", ee)), res("h_el_ion", ei)
            else:
                ee = res("h_el_el", ee)
        diff = r[:, :, None] - self.R
        dist = diff.norm(dim=-1)[..., None]
        out = []
        for s, sl in (("up", slice(0, u)), ("dn", slice(u, n))):
            bf = h[:, sl] @ self._leaf("bf_%s/linear_0" % s, "w")            # [b, i, c, D n]
            kap = torch.nn.functional.softplus(self._leaf("envelope_orbitals", "alpha_" + s))
            d = dist[:, sl]
            ex = self._leaf("envelope_orbitals", "weights_" + s) * torch.exp(-kap * d)
            env = ex.sum(2)[:, :, None]
            if lap:
                de = torch.einsum("bixf,bixa->biaf", -kap * ex, diff[:, sl] / d)
                le = (kap * (kap - 2 / d) * ex).sum(2)[:, :, None]
                i = torch.arange(n, device=r.device)[sl]
                k = torch.arange(len(i), device=r.device)
                tan = bf[:, :, 1:-1].reshape(b, len(i), n, 3, -1)
                own = tan[:, k, i]
                tan = tan * env[:, :, None]
                tan[:, k, i] += de * bf[:, :, :1]
                last = env * bf[:, :, -1:] + le * bf[:, :, :1] + 2 * (de * own).sum(2, keepdim=True)
                m = torch.cat([env * bf[:, :, :1], tan.reshape(b, len(i), 3 * n, -1), last], 2)
            else:
                m = env * bf
            out.append(m)
        m = torch.cat(out, 1)                                                # [b, i, c, D n]
        return m.reshape(b, n, m.shape[2], -1, n).permute(0, 2, 3, 1, 4)

    def log_psi_sqr(self, r, with_sign=False):
        sign, logdet = torch.linalg.slogdet(self._orbitals(r, False)[:, 0].contiguous())
        shift = logdet.amax(-1, keepdim=True)
        x = (sign * torch.exp(logdet - shift)).sum(-1)
        lp = 2 * (torch.log(x.abs() + 1e-8) + shift[:, 0])
        return (lp, x) if with_sign else lp

    def local_energy(self, r):
        per = max(1, 300_000_000 // (self.n * (3 * self.n + 2) * 832 * 8))
        return torch.cat([self._local_energy(r[b:b + per]) for b in range(0, len(r), per)])

    def _local_energy(self, r):
        n = self.n
        m = self._orbitals(r, True)
        m0 = m[:, 0].contiguous()
        sign, logdet = torch.linalg.slogdet(m0)
        inv = torch.linalg.inv(m0)
        y = inv[:, None] @ m[:, 1:].contiguous()                             # [b, c, D, n, n]
        tr = y.diagonal(dim1=-2, dim2=-1).sum(-1)
        g = tr[:, :-1]                                                       # [b, 3n, D]
        lam = tr[:, -1] - (y[:, :-1] * y[:, :-1].transpose(-1, -2)).sum((1, 3, 4))
        top = logdet.argmax(-1, keepdim=True)
        w = sign * torch.exp(logdet - logdet.gather(-1, top))
        gm, lm = g.gather(2, top[:, None].expand(-1, 3 * n, 1)), lam.gather(1, top)
        x = w.sum(-1)
        dx = (w[:, None] * (g - gm)).sum(-1)
        lx = (w * (lam - lm + (g - gm).square().sum(1))).sum(-1)
        s, a = torch.sign(x), x.abs() + 1e-8
        grad = 2 * (s[:, None] * dx / a[:, None] + gm[..., 0])
        lap = 2 * (s * lx / a - dx.square().sum(-1) / a ** 2 + lm[:, 0])
        kin = -0.5 * (lap / 2 + grad.square().sum(-1) / 4)
        d = lambda x, y: (x[..., :, None, :] - y[..., None, :, :]).norm(dim=-1)  # noqa: E731
        i, j = torch.triu_indices(n, n, 1, device=r.device)
        pot = (1 / d(r, r)[:, i, j]).sum(-1) - (self.Z / d(r, self.R)).sum((1, 2))
        a, b = torch.triu_indices(len(self.Z), len(self.Z), 1, device=r.device)
        return kin + pot + (self.Z[a] * self.Z[b] / d(self.R, self.R)[a, b]).sum()
