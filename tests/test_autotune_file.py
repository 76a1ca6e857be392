"""Autotune's parameter file: entries are found again only when the user
parameters match (floats to 1e-6, temperature to 10 %), and a new entry
replaces a matching one.  No GPU: the file logic is host code."""
from __future__ import annotations

import pytest

from rumd_amd.Autotune import Autotune, _same_user

USER = {"deviceName": "gfx950", "N": 1000, "numberEachType": [800, 200], "rho": 1.2, "T": 0.45,
        "potentialTypes": ["potLJ_12_6"], "pot_parameters": [[2.5, 4.0, -4.0]], "integratorType": "IntegratorNVT",
        "timeStep": 0.0025, "mixedPrecision": False}
TECH = {"pb": 32, "tp": 4, "skin": 0.3, "NB_method": "n2"}


def test_matching_rules():
    assert _same_user(USER, dict(USER))
    assert _same_user(USER, dict(USER, T=0.48))          # within 10 %
    assert not _same_user(USER, dict(USER, T=0.6))
    assert not _same_user(USER, dict(USER, N=1001))
    assert _same_user(USER, dict(USER, rho=1.2000002))      # float noise
    assert not _same_user(USER, dict(USER, rho=1.2001))
    assert not _same_user(USER, dict(USER, pot_parameters=[[2.5, 4.0, -4.1]]))
    assert not _same_user(USER, dict(USER, deviceName="other"))


def test_file_round_trip(tmp_path):
    at = Autotune(auto_filename=tmp_path / "autotune.json")
    assert at.CompareSavedParameters(USER) is None
    at.WriteParametersToFile(USER, TECH)
    assert at.CompareSavedParameters(USER) == TECH
    other = dict(USER, N=2000)
    at.WriteParametersToFile(other, dict(TECH, tp=1))
    at.WriteParametersToFile(USER, dict(TECH, skin=0.4))     # replaces the first entry
    assert at.CompareSavedParameters(USER)["skin"] == 0.4
    assert at.CompareSavedParameters(other)["tp"] == 1
    assert len(at._read_file()) == 2


def test_fixed_parameters_validated():
    with pytest.raises(ValueError):
        Autotune(tp=3)
    with pytest.raises(ValueError):
        Autotune(NB_method="cells")
    with pytest.raises(TypeError):
        Autotune(bogus=1)


def test_batch_entries_match_only_batches(tmp_path):
    """Batch user parameters (lists per replica) compare element by element
    and never match a single-sample entry."""
    from rumd_amd.Autotune import _same_user
    batch = {"deviceName": "d", "kind": "ReplicaBatch", "N": [300, 1200], "L": [6.3, 10.0],
             "thermostats": [[0.5, 0.2], [1.5, 0.2]], "timeStep": 0.0025, "skin": 0.3, "cutoffMethod": 2,
             "params": [2.5, 4.0, -4.0]}
    assert _same_user(batch, dict(batch))
    other = dict(batch, N=[300, 1201])
    assert not _same_user(batch, other)
    assert not _same_user(batch, dict(batch, thermostats=[[0.5, 0.2], [1.6, 0.2]]))
    single = {"deviceName": "d", "N": 1500}
    assert not _same_user(batch, single)


class _Timed(Autotune):
    """Autotune over a made-up clock: the list method alone decides."""

    def __init__(self, fastest, current, **kwargs):
        super().__init__(**kwargs)
        self.fastest, self.current = fastest, current

    def GetCurrentTechnicalParameters(self, sim):
        return {"pb": 64, "tp": self.current, "skin": 0.3, "NB_method": "default", "waves": 5}

    @staticmethod
    def _save(sim):
        return {}

    @staticmethod
    def _restore(sim, saved):
        pass

    def _trial_steps(self, sim, params, saved):
        return 40

    def _time(self, sim, params, saved, nsteps):
        return 1.0 if params["NB_method"] == self.fastest else 2.0


@pytest.mark.parametrize("n,fastest,searched", [(500, "none", ["sort"]), (16384, "n2", ["sort"]),
                                                (16385, "n2", ["n2", "sort"]), (40000, "sort", ["sort"])])
def test_lanes_are_timed_only_where_they_make_a_difference(tmp_path, n, fastest, searched):
    sim = type("Sim", (), {"sample": type("S", (), {"GetNumberOfParticles": lambda self: n})()})()
    at = _Timed(fastest, 4, auto_filename=tmp_path / "autotune.json")
    best = at.OptimizeTechnicalParameters(sim)
    assert best["NB_method"] == fastest
    tried = [t["params"] for t in at.trials if t["params"]["skin"] == 0.3]
    for method in ("none", "n2", "sort"):
        lanes = {p["tp"] for p in tried if p["NB_method"] == method}
        if lanes:
            assert lanes == ({1, 2, 4, 8} if method in searched else {4}), method
    fixed = _Timed(fastest, 4, auto_filename=tmp_path / "autotune.json", tp=2)
    assert fixed.OptimizeTechnicalParameters(sim)["tp"] == 2
    assert {t["params"]["tp"] for t in fixed.trials} == {2}
