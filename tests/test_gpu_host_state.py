"""What the host classes keep between calls: after calls that are refused, when
list flags are read, and for objects that serve more than one sample."""
from __future__ import annotations

import numpy as np
import pytest

from capi import gpu_available
from rumd_amd import conf_io, configs, rumd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


def _sample(pos, box, velocity=0.5):
    n = len(pos)
    s = rumd.Sample(0, 0)
    s.SetVerbose(False)
    s.SetConfiguration(conf_io.Configuration(
        n=n, box=np.full(3, float(box)), types=np.zeros(n, np.int32), positions=np.asarray(pos, np.float64),
        masses=np.ones(1), velocities=np.full((n, 3), velocity), images=np.zeros((n, 3))))
    return s


def _lj(rcut, method="n2", max_nbrs=None):
    pot = rumd.Pot_LJ_12_6(cutoff_method=rumd.ShiftedPotential)
    pot.SetVerbose(False)
    pot.SetParams(0, 0, Sigma=1.0, Epsilon=1.0, Rcut=rcut)
    pot.SetNbListSkin(0.3)
    pot.SetNB_Method(method)
    if max_nbrs:
        pot.SetNbMaxNumNbrs(max_nbrs)
    return pot


@pytest.mark.parametrize("method", ["n2", "none"])
def test_a_step_without_degrees_of_freedom_moves_nothing(method):
    """One particle has none (3 N - 3) for its thermostat: refused, as it was."""
    s = _sample([[0.25, -1.0, 2.0]], 20.0)
    pot, itg = _lj(2.5, method), rumd.IntegratorNVT(timeStep=0.005, targetTemperature=1.0,
                                                    thermostatRelaxationTime=0.2)
    s.SetPotential(pot)
    s.SetIntegrator(itg)
    r, v = s.GetPositions(), s.GetVelocities()
    print(f"[case] no degrees of freedom {method}", flush=True)
    s.CalcF()
    for step in (itg.Integrate, lambda: s.RunSteps(0, 1, 1, 0), lambda: s.RunSteps(0, 4, 4, 0)):
        with pytest.raises(RuntimeError, match="degrees of freedom"):
            step()
        np.testing.assert_array_equal(s.GetPositions(), r)
        np.testing.assert_array_equal(s.GetVelocities(), v)
        assert itg.GetThermostatState() == 0.0


def test_list_flags_are_read_anew_after_an_exception():
    """Synchronize reads every list's flags and then acts on them; when acting
    on the first list's throws, the second's are still to be read."""
    n = 66000
    k = 41  # 41^3 sites
    box = 2.0 * k
    site = np.arange(n)
    pos = (np.stack([site // (k * k), site // k % k, site % k], axis=1) + 0.5) * 2.0 - 0.5 * box
    s = _sample(pos, box, velocity=0.0)
    # the first twenty are 0.2 apart after one step
    together = pos[0] + 0.2 * np.stack([np.arange(20) % 3, np.arange(20) // 3 % 3, np.arange(20) // 9], axis=1)
    vel = np.zeros((n, 3), np.float32)
    vel[:20] = (together - pos[:20]) / 0.01
    s.SetVelocities(vel)
    itg = rumd.IntegratorNVE(timeStep=0.01)
    s.SetIntegrator(itg)
    # all pairs in reach: the list overflows, and cannot grow to 66,000 x 66,048 entries
    a, b = _lj(1.2, max_nbrs=8), _lj(0.9 * box, max_nbrs=44000)
    s.SetPotential(a)
    s.AddPotential(b)  # ahead of the first
    print("[case] flags after an exception", flush=True)
    s.CalcF()
    with pytest.raises(ValueError, match="2\\^32"):
        s.Synchronize()
    b.SetParams(0, 0, Sigma=1.0, Epsilon=1.0, Rcut=1.2)
    b.SetNbMaxNumNbrs(64)
    itg.Integrate()
    s.CalcF()
    s.Synchronize()  # the list of eight grows
    s.CalcF()
    assert np.diff(a.GetNeighborListCSR(s)[0])[:20].tolist() == [19] * 20


def test_list_flags_of_a_potential_given_to_another_sample():
    """The first sample's Synchronize may find work of the second's in flight;
    an overflow in that work is still acted upon."""
    rng = np.random.default_rng(3)
    n, box = 150001, 60.0
    pos = rng.uniform(-0.5 * box, 0.5 * box, size=(n, 3))  # some 8 within 1.4 on average, some particles more than 16
    first, second = _sample(pos[:1000], box), _sample(pos, box)
    pot = _lj(1.1, max_nbrs=8)
    first.SetPotential(pot)
    first.CalcF()
    first.Synchronize()
    second.SetPotential(pot)
    print("[case] flags of a shared potential", flush=True)
    second.CalcF()
    first.Synchronize()
    second.Synchronize()
    second.CalcF()
    cnt = np.diff(pot.GetNeighborListCSR(second)[0])
    assert cnt.max() == pot.GetActualMaxNumNbrs() > 16


@pytest.mark.parametrize("kind", ["BondHarmonic", "BondFENE", "AngleCosSq", "AngleSq", "DihedralRyckaert",
                                  "PeriodicDihedral"])
def test_no_steps_with_molecular_parameters_unset(kind):
    """A run of no steps asks nothing of the potentials; one of a step names what is missing."""
    s = _sample([[0.9 * i, 0.0, 0.1 * (i % 2)] for i in range(6)], 20.0)
    pot, term, itg = _lj(2.5), getattr(rumd, kind)(), rumd.IntegratorNVE(timeStep=0.001)
    md = s.CreateMoleculeData()
    md.SetBonds([0, 1, 0, 1, 2, 0])
    md.SetAngles([0, 1, 2, 0])
    md.SetDihedrals([0, 1, 2, 3, 0])
    s.SetPotential(pot)
    s.AddPotential(term)
    s.SetIntegrator(itg)
    print(f"[case] parameters unset {kind}", flush=True)
    s.RunSteps(0, 0, 10, 0)
    assert s.PrepareRunSteps(0, 0, 10, 0) == 0
    for steps in (1, 4):
        with pytest.raises(RuntimeError, match="parameters"):
            s.RunSteps(0, steps, steps, 0)
