"""The Laplacian half of the tuner's sweep (CPU only): the library's choice is a candidate, fields that no kernel of the form
reads are left out, and a choice has to gain in both forms that share it."""
import pytest

from deeperwin_amd import _native, tuning
from deeperwin_amd.params import ModelShape

torch = pytest.importorskip("torch")


@pytest.mark.parametrize("precision,width1,mu", [("fp32", 256, None), ("fp32", 384, (-1, 0, 1, 2)), ("bf16x3", 256, (-1, 0)),
                                                 ("bf16", 256, None), ("fp64", 256, None)])
def test_search_space_follows_the_kernels(precision, width1, mu):
    space = {name: tuple(cands) for name, cands, _ in tuning.search_space(14, precision, width1)}
    assert space["lap_cols"][0] == 0 and space["lap_electrons"][0] == 0 and space["lap_orb_tile"][0] == -1
    assert space.get("lap_mu_tile") == mu
    assert set(space) <= set(_native.TUNING_FIELDS)


class Model:
    """Energies take as long as `cost` says for the fields set and the form."""
    precision, shape = "fp32", ModelShape(14, 7, 2, 4)

    def __init__(self, cost):
        self.cost, self.fields, self.took, self.forms = cost, dict(_native.TUNING_DEFAULT), 0.0, set()

    def get_tuning(self):
        return dict(self.fields)

    def set_tuning(self, **kw):
        self.fields.update(kw)

    def logpsi(self, r, R, Z, lp):
        self.took = 1.0

    def local_energy(self, r, R, Z, e):
        form = _native._lap_form.get()
        self.forms.add(form)
        self.took = self.cost(self.fields, form)


@pytest.mark.parametrize("split,fp32,expected", [(1.5, 0.5, 0), (0.9, 1.1, 0), (0.9, 0.95, 256), (1.0, 1.0, 0)])
def test_a_choice_has_to_gain_in_both_forms(monkeypatch, split, fp32, expected):
    def cost(f, form):
        return (fp32 if form == _native.LAP_FP32 else split) if f["lap_cols"] == 256 else 1.0

    m = Model(cost)

    def timed(fn, reps=3):
        fn()
        return m.took

    monkeypatch.setattr(tuning, "time_ms", timed)
    best, log = tuning.autotune_model(m, torch.zeros(3, 14, 3), None, None)
    assert best["lap_cols"] == expected and best["lap_electrons"] == 0 and best["lap_mu_tile"] == -1
    assert m.forms == {None, _native.LAP_FP32}
    assert "lap_mu_tile" not in {entry["field"] for entry in log}
