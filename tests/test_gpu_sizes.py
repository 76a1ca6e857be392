"""Kernels at the sizes where their work split changes: remainders of a wave or
workgroup, both sides of a size rule, the smallest and larger samples."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
from capi import GpuSystem, check, gpu_available, lib
from helpers import FORCE_TOL_GUARDED, force_errors, ka_table, load_golden, sorted_rows, unsort
from test_gpu_batch import make_batch
from test_gpu_potentials import PE_ATOL, _forms, _table
from rumd_amd import conf_io, configs, rumd

pytestmark = pytest.mark.gpu

SP, SF, NS = 1, 2, 0


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


def _ka(n, seed=7, jitter=0.02, density=1.2):
    s = configs.ka_random_lattice(n, density=density, seed=seed)
    rng = np.random.default_rng(seed + 1)
    pos = s.positions + rng.uniform(-jitter, jitter, size=s.positions.shape)
    pos -= s.box * np.rint(pos / s.box)
    return s, configs.pack_pos4(pos.astype(np.float32), s.types)


def _gpu(s, pos4, method, **kw):
    return GpuSystem(pos4, configs.pack_vel4(s.velocities, s.types, s.masses), configs.box8(s.box), 2, ka_table(),
                     method=method, **kw)


# a wave per particle, sixteen per workgroup, candidates 1,024 at a time
@pytest.mark.parametrize("n", [2, 16, 17, 1023, 1024, 1025, 4099])
def test_n2_lists_at_the_edges_of_the_wave_split(n):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, "n2", max_nbrs=n + 1)
    print(f"[case] n2 lists n={n}", flush=True)
    g.update_nblist()
    # a second build starts from the counters the first one left
    check(lib().rumdx_nblist_request_rebuild(C.byref(g.nb), None))
    g.update_nblist()
    cnt, nbl = g.neighbor_lists()
    off, idx = oracle.nblist_brute_f32(pos4, configs.box8(s.box), 2, configs.cut_skin2_table(ka_table(), 0.3))
    for i in range(n):
        assert np.array_equal(nbl[: cnt[i], i], np.sort(idx[off[i]:off[i + 1]])), i
    flags = g.flags_host()
    # (no rebuild pending, no overflow, two builds, the longest list, counter at zero)
    assert flags[:5].tolist() == [0, 0, 2, cnt.max(), 0]


# more groups of sixteen particles than workgroups: some take two in turn
@pytest.mark.parametrize("n", [32768, 32769, 32785])
def test_n2_lists_beyond_one_group_per_workgroup(n):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, "n2", max_nbrs=160)
    print(f"[case] n2 lists n={n}", flush=True)
    for builds in (1, 2):
        g.update_nblist()
        cnt, nbl = g.neighbor_lists()
        off, idx = oracle.nblist_brute_f32(pos4, configs.box8(s.box), 2, configs.cut_skin2_table(ka_table(), 0.3))
        assert np.array_equal(cnt, np.diff(off))
        lists = np.where(np.arange(nbl.shape[0])[:, None] < cnt, nbl[:, :n], np.uint32(0xffffffff))
        assert np.array_equal(lists.T[:, : cnt.max()].astype(np.int64) & 0x7fffffff, sorted_rows(off, idx))
        assert g.flags_host()[:5].tolist() == [0, 0, builds, cnt.max(), 0]
        check(lib().rumdx_nblist_request_rebuild(C.byref(g.nb), None))


# a wave per particle, four per workgroup, partners 512 at a time
@pytest.mark.parametrize("n", [2, 3, 65, 511, 513, 1027])
@pytest.mark.parametrize("stress", [False, True])
def test_all_pairs_at_the_edges_of_the_partner_tiles(n, stress):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, "none", with_sts=stress)
    print(f"[case] all pairs n={n} stress={stress}", flush=True)
    f_ref, _ = oracle.forces_brute(pos4, s.box, 2, ka_table(), SF)
    g.calc_f(SF, stress=stress)
    f = g.get("f")[:n]
    assert force_errors(f[:, :3], f_ref[:, :3])["guarded_max"] <= FORCE_TOL_GUARDED
    g.calc_f(SF, initialize=False, stress=stress)  # added to the first call's
    np.testing.assert_allclose(g.get("f")[:n], 2 * f, rtol=0, atol=2e-6 * np.abs(f).max())


# one, two and four workgroups per tile (27, 125 and 512 tiles), wrapping tiles
# with and without the shifted frame, FP64 positions
@pytest.mark.parametrize("n,cutoff,stress", [(2500, SF, False), (2500, SP, True), (19001, NS, False),
                                             (19001, SF, True), (95003, SF, False)])
def test_fp64_tiles_at_each_split(n, cutoff, stress):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, "sorted", max_nbrs=200, with_sts=stress)
    print(f"[case] fp64 tiles n={n} tiles={g.nb.ntiles} cutoff={cutoff} stress={stress}", flush=True)
    g.calc_f(cutoff, fp64=True, stress=stress)
    uidx = g.unsorted_index()
    f = unsort(g.get("f"), uidx)
    f_ref, _ = oracle.forces_cells(pos4, s.box, 2, ka_table(), cutoff)
    # the output's rounding (2^-24) and the float parameters the oracle shares
    assert force_errors(f[:, :3], f_ref[:, :3])["guarded_max"] <= 2e-7
    if stress:
        sts = unsort(g.get("sts"), uidx)
        sts_ref = oracle.stress_brute(pos4, s.box, 2, ka_table(), cutoff) if n < 5000 else None
        if sts_ref is not None:
            np.testing.assert_allclose(sts[:, :3], sts_ref[:, :3], rtol=0, atol=2e-7 * np.abs(sts_ref).max())


# all six components, kept in sts and in the middle of w, at each split and list kind
@pytest.mark.parametrize("method,n,cutoff", [("sorted", 2500, SP), ("sorted", 19001, SF), ("sorted", 95003, NS),
                                             ("n2", 1003, SF), ("none", 333, SP)])
def test_fp64_stress_components(method, n, cutoff):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, method, with_sts=True, **({"max_nbrs": 200} if method != "none" else {}))
    print(f"[case] fp64 stress {method} n={n} cutoff={cutoff}", flush=True)
    g.calc_f(cutoff, fp64=True, stress=True)
    uidx = g.unsorted_index()
    sts, w = unsort(g.get("sts"), uidx), unsort(g.get("w"), uidx)
    ref = oracle.stress_brute(pos4, s.box, 2, ka_table(), cutoff)
    # the output's rounding (2^-24) and the float parameters the oracle shares, as for the forces
    np.testing.assert_allclose(np.column_stack([sts, w[:, 1:3]]), ref, rtol=0, atol=2e-7 * np.abs(ref).max())


# list lanes and the all-pairs wave of the FP64 slot kernel
@pytest.mark.parametrize("method,n", [("n2", 3), ("n2", 17), ("n2", 1003), ("none", 3), ("none", 333)])
def test_fp64_slots_with_shared_lanes(method, n):
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, method)
    print(f"[case] fp64 slots {method} n={n}", flush=True)
    g.calc_f(SF, fp64=True)
    f = unsort(g.get("f"), g.unsorted_index())
    f_ref, _ = oracle.forces_brute(pos4, s.box, 2, ka_table(), SF)
    assert force_errors(f[:, :3], f_ref[:, :3])["guarded_max"] <= 2e-7


# the kernels compiled per form (no stresses, initialising), every cut-off and list method
@pytest.mark.parametrize("case", _forms(), ids=lambda c: c[0])
def test_forms_without_stresses(golden_dir, case):
    name, form, make, rows = case
    c = load_golden(golden_dir / "KA_N1000_T0.466.xyz.gz")
    pos4 = configs.pack_pos4(c.positions, c.types)
    for cutoff in (NS, SP, SF):
        table = _table(make, cutoff, rows)
        f_ref, _ = oracle.forces_form_brute(pos4, c.box, 2, table, form, cutoff)
        for method in ("sorted", "n2", "none"):
            g = GpuSystem(pos4, configs.pack_vel4(c.velocities, c.types, c.masses), configs.box8(c.box), 2, table,
                          method=method)
            print(f"[case] form {name} cutoff={cutoff} method={method}", flush=True)
            g.calc_f(cutoff, form=form)
            f = unsort(g.get("f"), g.unsorted_index())
            assert force_errors(f[:, :3], f_ref[:, :3])["guarded_max"] <= FORCE_TOL_GUARDED
            pe_tol = max(PE_ATOL, 2e-6 * np.abs(f_ref[:, 3]).max())
            np.testing.assert_allclose(f[:, 3], f_ref[:, 3], rtol=0, atol=pe_tol)


def test_new_padding_keeps_the_fp64_positions():
    """SetPB_TP reallocates the particle arrays; in mixed-precision mode the
    low-order position parts stay with the configuration."""
    s, _ = _ka(500)
    sample = rumd.Sample(0, 0)
    sample.SetVerbose(False)
    sample.SetMixedPrecisionPositions(True)
    sample.SetConfiguration(conf_io.Configuration(
        n=s.n, box=s.box, types=s.types, positions=s.positions, masses=s.masses, velocities=s.velocities,
        images=np.zeros_like(s.positions)))
    pos64 = s.positions.astype(np.float64) * (1.0 + 1e-8)
    sample.SetPositionsFP64(pos64)
    before = sample.GetPositionsFP64()
    assert np.abs(before - pos64).max() < 1e-12
    sample.SetPB_TP(64, 8)
    np.testing.assert_array_equal(sample.GetPositionsFP64(), before)


def _stepping_sample(n, method, thermo, mixed, T=2.0):
    s, _ = _ka(n, jitter=0.0)
    sample = rumd.Sample(0, 0)
    sample.SetVerbose(False)
    sample.SetMixedPrecisionPositions(mixed)
    sample.SetConfiguration(conf_io.Configuration(
        n=s.n, box=s.box, types=s.types, positions=s.positions, masses=s.masses,
        velocities=2.0 * s.velocities, images=np.zeros_like(s.positions)))
    pot = rumd.Pot_LJ_12_6(cutoff_method=rumd.ShiftedForce)
    pot.SetVerbose(False)
    for (i, j, sg, ep, rc) in configs.ka_params(2.5):
        pot.SetParams(i, j, Sigma=sg, Epsilon=ep, Rcut=rc)
    pot.SetNbListSkin(0.3)
    pot.SetNB_Method(method)
    sample.SetPotential(pot)
    itg = rumd.IntegratorNVT(timeStep=0.0025, targetTemperature=T, thermostatRelaxationTime=0.2) if thermo else \
        rumd.IntegratorNVE(timeStep=0.0025)
    if thermo:
        itg.SetTemperatureChangePerTimeStep(1e-4)
    sample.SetIntegrator(itg)
    return sample, pot, itg


# one-kernel steps in chains of 7, 1, 2 and more against CalcF and Integrate:
# remainders of the 16-particle groups, the largest size, rebuilds inside chains
@pytest.mark.parametrize("n,method,thermo,mixed", [(40, "none", True, False), (531, "none", False, True),
                                                   (203, "n2", True, False), (1003, "n2", False, False),
                                                   (4099, "n2", True, True), (16384, "n2", True, False)])
def test_one_kernel_steps_equal_the_separate_calls(n, method, thermo, mixed):
    print(f"[case] small steps n={n} {method} thermo={thermo} mixed={mixed}", flush=True)
    a, pot_a, itg_a = _stepping_sample(n, method, thermo, mixed)
    b, pot_b, itg_b = _stepping_sample(n, method, thermo, mixed)
    i = 0
    for steps, block in ((7, 7), (1, 5), (2, 2), (23, 8)):
        a.RunSteps(i, steps, block, 20)
        for k in range(i, i + steps):
            if k % 20 == 0:
                itg_b.SetMomentumToZero()
            b.CalcF()
            itg_b.Integrate()
        i += steps
        for get in ("GetPositionsFP64", "GetVelocities", "GetImages", "GetForcesAndEnergies", "GetVirials"):
            np.testing.assert_array_equal(getattr(a, get)(), getattr(b, get)(), err_msg=f"{get} after {i} steps")
        assert itg_a.GetThermostatState() == itg_b.GetThermostatState()
        assert itg_a.GetKineticEnergy() == itg_b.GetKineticEnergy()
    if thermo:
        assert itg_a.GetTargetTemperature() == itg_b.GetTargetTemperature()
    if method == "n2":
        assert pot_a.GetNumberOfNbListBuilds() == pot_b.GetNumberOfNbListBuilds() > 1


# the largest N2 sample that steps in chains, and the smallest that does not
@pytest.mark.parametrize("n", [5000, 5001])
def test_steps_on_both_sides_of_the_chain_rule(n):
    test_one_kernel_steps_equal_the_separate_calls(n, "n2", True, True)


def test_one_kernel_steps_with_an_overflowed_list():
    """Lists that overflow inside a chain take all pairs, and grow afterwards."""
    a, pot_a, _ = _stepping_sample(1003, "n2", True, False)
    b, _, _ = _stepping_sample(1003, "n2", True, False)
    pot_a.SetNbMaxNumNbrs(40)
    print("[case] small steps, overflowed lists", flush=True)
    a.RunSteps(0, 10, 10, 0)
    b.RunSteps(0, 10, 10, 0)
    # the overflowed particles' sums run in another order: rounding apart after ten steps
    np.testing.assert_allclose(a.GetVelocities(), b.GetVelocities(), rtol=0, atol=1e-4)
    a.CalcF()  # builds in the grown lists
    assert pot_a.GetActualMaxNumNbrs() > 40


def _short_ranged(n, rcut, temperature=0.8):
    """An LJ liquid at density 0.8442 cut off at rcut, sorted lists, constant energy."""
    rng = np.random.default_rng(n)
    k = int(np.ceil(n ** (1.0 / 3.0)))
    box = (n / 0.8442) ** (1.0 / 3.0)
    site = np.sort(rng.permutation(k ** 3)[:n])
    pos = (np.stack([site // (k * k), site // k % k, site % k], axis=1) + 0.5) * (box / k) - 0.5 * box
    pos = (pos + rng.uniform(-0.1, 0.1, size=pos.shape)).astype(np.float32)
    sample = rumd.Sample(0, 0)
    sample.SetVerbose(False)
    sample.SetConfiguration(conf_io.Configuration(
        n=n, box=np.full(3, box), types=np.zeros(n, np.int32), positions=pos, masses=np.ones(1),
        velocities=rng.normal(size=(n, 3)) * np.sqrt(temperature), images=np.zeros((n, 3))))
    pot = rumd.Pot_LJ_12_6(cutoff_method=rumd.ShiftedForce)
    pot.SetVerbose(False)
    pot.SetParams(0, 0, Sigma=1.0, Epsilon=1.0, Rcut=rcut)
    pot.SetNbListSkin(0.3)
    pot.SetNB_Method("sort")
    sample.SetPotential(pot)
    itg = rumd.IntegratorNVE(timeStep=0.002)
    sample.SetIntegrator(itg)
    return sample, pot, itg, configs.pack_pos4(sample.GetPositions(), np.zeros(n, np.int32)), np.full(3, box)


# tiles of few particles: up to eight, two and one lane per list (1,331, 3,375 and
# 4,913 tiles of 34 to 41), two lanes for the larger ones of many (4,913 of 66 to 81)
@pytest.mark.parametrize("n,rcut,tiles", [(30001, 1.5, 729), (45001, 1.5, 1331), (130001, 1.5, 3375),
                                          (200001, 1.5, 4913), (90001, 2.0, 1331), (400001, 2.0, 4913)])
def test_forces_at_each_number_of_lanes(n, rcut, tiles):
    s, pot, _itg, pos4, box = _short_ranged(n, rcut)
    print(f"[case] lanes n={n} rcut={rcut}", flush=True)
    s.CalcF()
    assert pot.GetNbTileStats()["tiles"] == tiles
    f = s.GetForcesAndEnergies()
    table = configs.lj_param_table([(0, 0, 1.0, 1.0, rcut)], 1)
    f_ref, _ = oracle.forces_cells(pos4, box, 1, table, SF)
    assert force_errors(f[:, :3], f_ref[:, :3])["guarded_max"] <= FORCE_TOL_GUARDED


# axes of five cells, where a tile's halo holds the box once and its stencils still
# wrap, of six and seven, alone and with long ones, in every shape of tile
@pytest.mark.parametrize("box", [(6.9, 6.9, 6.9), (8.5, 8.5, 8.5), (9.9, 9.9, 9.9), (7.0, 8.5, 9.9),
                                 (56.0, 56.0, 7.0), (56.0, 7.0, 56.0), (7.0, 56.0, 56.0), (56.0, 56.0, 8.5),
                                 (30.0, 7.0, 7.5), (140.0, 140.0, 7.0), (17.0, 17.0, 7.0)])
def test_sorted_lists_and_forces_in_boxes_of_few_cells(box):
    rng = np.random.default_rng(17)
    box = np.array(box)
    k = np.floor(box / 1.12).astype(int)
    n = int(k.prod())
    site = np.stack(np.meshgrid(*[np.arange(m) for m in k], indexing="ij"), axis=-1).reshape(-1, 3)
    pos = ((site + 0.5) * (box / k) - 0.5 * box + rng.uniform(-0.15, 0.15, size=(n, 3))).astype(np.float32)
    sample = rumd.Sample(0, 0)
    sample.SetVerbose(False)
    sample.SetConfiguration(conf_io.Configuration(
        n=n, box=box, types=np.zeros(n, np.int32), positions=pos, masses=np.ones(1),
        velocities=rng.normal(size=(n, 3)), images=np.zeros((n, 3))))
    pot = rumd.Pot_LJ_12_6(cutoff_method=rumd.ShiftedForce)
    pot.SetVerbose(False)
    pot.SetParams(0, 0, Sigma=1.0, Epsilon=1.0, Rcut=2.5)
    pot.SetNbListSkin(0.3)
    pot.SetNB_Method("sort")
    sample.SetPotential(pot)
    itg = rumd.IntegratorNVE(timeStep=0.002)
    sample.SetIntegrator(itg)
    table = configs.lj_param_table([(0, 0, 1.0, 1.0, 2.5)], 1)
    b8 = configs.box8(box)
    print(f"[case] few cells {box.tolist()} n={n}", flush=True)
    for steps in (0, 12):  # the full sort and, with a rebuild asked for, the tile re-sort
        sample.RunSteps(0, steps, 6, 0)
        if steps:
            sample.SortParticles()
        sample.CalcF()
        pos4 = configs.pack_pos4(sample.GetPositions(), np.zeros(n, np.int32))
        off, idx = oracle.nblist_brute_f32(pos4, b8, 1, configs.cut_skin2_table(table, 0.3))
        got_off, got_idx = pot.GetNeighborListCSR(sample)
        assert np.array_equal(sorted_rows(got_off, got_idx), sorted_rows(off, idx))
        f_ref, _ = oracle.forces_nl(pos4, box, 1, table, SF, off, idx)
        assert force_errors(sample.GetForces(), f_ref[:, :3])["guarded_max"] <= FORCE_TOL_GUARDED


# both sides of the fused steps' rule: at most 1,024 tiles, or 64 particles a tile;
# the same bits either way
@pytest.mark.parametrize("n,rcut,fused", [(20000, 2.0 ** (1.0 / 6.0), True), (30000, 2.0 ** (1.0 / 6.0), False),
                                          (65000, 1.7, False), (90000, 2.0, True)])
def test_fused_steps_on_both_sides_of_their_rule(n, rcut, fused):
    print(f"[case] fused rule n={n} rcut={rcut:.3f}", flush=True)
    a, pot_a, _ia, _, _ = _short_ranged(n, rcut)
    b, _pb, _ib, _, _ = _short_ranged(n, rcut)
    b.SetFusedSteps(False)
    a.RunSteps(0, 40, 10, 0)  # rebuilds inside
    b.RunSteps(0, 40, 10, 0)
    tiles = pot_a.GetNbTileStats()["tiles"]
    assert a.UsesFusedSteps() == fused == (tiles <= 1024 or 64 * tiles <= n)
    assert pot_a.GetNumberOfNbListBuilds() > 1
    for get in ("GetPositions", "GetVelocities", "GetImages", "GetForcesAndEnergies", "GetVirials"):
        np.testing.assert_array_equal(getattr(a, get)(), getattr(b, get)(), err_msg=get)


# the FP64 tile kernel's workgroups of 64 to 512 lanes: few tiles (864, 729 and 512)
# and many (1,331 or more), by the particles in a tile
@pytest.mark.parametrize("n,rcut,tiles", [(9000, 1.5, 864), (30001, 1.5, 729), (130001, 2.5, 1000),
                                          (30001, 1.2, 1331), (45001, 1.5, 1331), (90001, 2.0, 1331),
                                          (200001, 2.5, 1331)])
def test_fp64_forces_at_each_number_of_lanes(n, rcut, tiles):
    s, pot, _itg, pos4, box = _short_ranged(n, rcut)
    pot.SetFP64Forces(True)
    print(f"[case] fp64 lanes n={n} rcut={rcut}", flush=True)
    s.CalcF()
    assert pot.GetNbTileStats()["tiles"] == tiles
    table = configs.lj_param_table([(0, 0, 1.0, 1.0, rcut)], 1)
    f_ref, _ = oracle.forces_cells(pos4, box, 1, table, SF)
    assert force_errors(s.GetForces(), f_ref[:, :3])["guarded_max"] <= 2e-7  # as for all FP64 forces


# tiles of 2x2x2, 4x2x2, 4x4x2 and 4x4x4 cells
@pytest.mark.parametrize("n", [9001, 33001, 66001, 130001])
def test_sorted_lists_and_steps_at_each_tile_shape(n):
    print(f"[case] tile shapes n={n}", flush=True)
    a, pot, itg_a = _stepping_sample(n, "sort", True, False)
    b, _, itg_b = _stepping_sample(n, "sort", True, False)
    b.SetFusedSteps(False)
    a.RunSteps(0, 30, 10, 0)  # rebuilds inside
    b.RunSteps(0, 30, 10, 0)
    assert pot.GetNumberOfNbListBuilds() > 1
    # the kinetic-energy sum runs per tile in one and per 256 slots in the
    # other (Ps agrees to 1e-12), so bits may differ where ps rounds to float
    np.testing.assert_allclose(itg_a.GetThermostatState(), itg_b.GetThermostatState(), rtol=1e-6)
    np.testing.assert_allclose(a.GetVelocities(), b.GetVelocities(), rtol=0, atol=2e-4)
    a.CalcF()
    off, ids = pot.GetNeighborListCSR(a)
    pos4 = configs.pack_pos4(a.GetPositions(), a.GetTypes())
    box = np.array([a.GetSimulationBox().GetLength(k) for k in range(3)])
    f_ref, _ = oracle.forces_cells(pos4, box, 2, ka_table(), SF)
    assert force_errors(a.GetForces(), f_ref[:, :3])["guarded_max"] <= FORCE_TOL_GUARDED
    # the list holds every pair within rc of the current positions (it was
    # built within half a skin of them): check a sample of particles
    x = pos4[:, :3].astype(np.float64)
    for i in range(0, n, n // 50):
        d = x - x[i]
        d -= box * np.rint(d / box)
        near = np.flatnonzero((d * d).sum(axis=1) < (2.5 * 0.8) ** 2)
        assert set(near) - {i} <= set(ids[off[i]:off[i + 1]].tolist())


@pytest.mark.parametrize("tp", [1, 2])
def test_batch_steps_at_the_edges_of_the_passes(tp):
    """Batched steps in one launch (a captured block: its inner steps without
    energies) against separate calls: the same bits at the edges of the 256-slot
    blocks and 1024-slot passes, with complete lists and with lists of which
    all but a few overflow (partners then come from the cells)."""
    sizes = [256, 257, 1024, 1025, 2049]
    systems = [configs.ka_random_lattice(n, density=1.2, temperature=0.9, seed=300 + n) for n in sizes]
    for cap in (None, 40):
        out = []
        for fused in (False, True):
            b = make_batch(systems, [0.8, 1.5, 0.6, 1.0, 0.9], max_nbrs=cap)
            b.SetThermostat(2, 0.6, 0.0)  # NVE
            b.SetLanesPerParticle(tp)
            b.SetFusedSteps(fused)
            print(f"[case] batch passes fused={fused} lanes={tp} cap={cap}", flush=True)
            b.RunSteps(10, 10)
            out.append([(b.GetPositions(r), b.GetVelocities(r), b.GetForcesAndEnergies(r)) for r in range(len(sizes))]
                       + [b.GetThermostatStates(), b.GetEnergies()])
        for r in range(len(sizes)):
            for k in range(3):
                np.testing.assert_array_equal(out[0][r][k], out[1][r][k], err_msg=f"replica {r} array {k}")
        np.testing.assert_array_equal(np.asarray(out[0][-2]), np.asarray(out[1][-2]))
        np.testing.assert_array_equal(np.asarray(out[0][-1]), np.asarray(out[1][-1]))


def _melt(golden_dir, chains, copies, method, kinds):
    """`chains` five-bead chains of the pentamer melt, the box repeated `copies`
    times per axis, with the potentials named in `kinds`."""
    c = load_golden(golden_dir / "pentamer200_rho0.85_T0.5.xyz.gz")
    box = np.asarray(c.box, np.float64)
    shifts = np.array([[x, y, z] for x in range(copies) for y in range(copies) for z in range(copies)])
    mid = (copies - 1) / 2.0
    pos = np.concatenate([c.positions[:5 * chains] + (sh - mid) * box for sh in shifts])
    total = copies ** 3 * chains
    n, big = 5 * total, box * copies
    pos -= big * np.rint(pos / big)
    rng = np.random.default_rng(5)
    s = rumd.Sample(0, 0)
    s.SetVerbose(False)
    s.SetConfiguration(conf_io.Configuration(
        n=n, box=big, types=np.zeros(n, np.int32), positions=pos, masses=np.ones(1),
        velocities=rng.normal(size=(n, 3)), images=np.zeros((n, 3))))
    pot = rumd.Pot_LJ_12_6(cutoff_method=rumd.ShiftedPotential)
    pot.SetVerbose(False)
    pot.SetParams(0, 0, Sigma=1.0, Epsilon=1.0, Rcut=2.5)
    pot.SetNbListSkin(0.3)
    pot.SetNB_Method(method)
    s.SetPotential(pot)
    md = s.CreateMoleculeData()
    first = 5 * np.arange(total)
    md.SetBonds([int(x) for f in first for k in range(4) for x in (f + k, f + k + 1, k % 2)])
    md.SetAngles([int(x) for f in first for k in range(3) for x in (f + k, f + k + 1, f + k + 2, 0)])
    md.SetDihedrals([int(x) for f in first[::2] for k in range(2) for x in (f + k, f + k + 1, f + k + 2, f + k + 3, 0)])
    for kind in kinds:
        p = getattr(rumd, kind)()
        p.SetVerbose(False)
        if kind == "BondHarmonic":
            p.SetParams(bond_type=0, bond_length=1.0, stiffness=100.0, exclude=False)
        elif kind == "BondFENE":
            p.SetParams(1, 2.5, 30.0, False)
        elif kind.startswith("Angle"):
            p.SetParams(angle_type=0, theta0=2.0, ktheta=20.0)
        else:
            p.SetParams(dihedral_type=0, coeffs=[1.0, -0.5, 0.3, 0.2, 0.1, -0.2][:4 if kind.startswith("P") else 6])
        s.AddPotential(p)
    itg = rumd.IntegratorNVT(timeStep=0.002, targetTemperature=1.0, thermostatRelaxationTime=0.2)
    s.SetIntegrator(itg)
    return s, itg, (pot, md)


# one to four terms, every kind; remainders of the 256-slot workgroups; both
# groupings of the kinetic energy
@pytest.mark.parametrize("chains,copies,method,kinds", [
    (51, 1, "none", ("BondHarmonic",)), (52, 1, "n2", ("BondFENE", "AngleSq")),
    (200, 1, "n2", ("BondHarmonic", "AngleCosSq", "DihedralRyckaert")),
    (200, 2, "sort", ("BondHarmonic", "BondFENE", "AngleSq", "PeriodicDihedral")),
    (199, 3, "sort", ("BondHarmonic", "AngleCosSq"))])
def test_bonded_steps_equal_the_separate_calls(golden_dir, chains, copies, method, kinds):
    print(f"[case] bonded steps {5 * chains * copies ** 3} {method} {kinds}", flush=True)
    a, itg_a, keep_a = _melt(golden_dir, chains, copies, method, kinds)
    b, itg_b, keep_b = _melt(golden_dir, chains, copies, method, kinds)
    i = 0
    for steps, block in ((7, 7), (1, 5), (24, 8)):
        a.RunSteps(i, steps, block, 20)
        for k in range(i, i + steps):
            if k % 20 == 0:
                itg_b.SetMomentumToZero()
            b.CalcF()
            itg_b.Integrate()
        i += steps
        b.Synchronize()
        for get in ("GetPositions", "GetVelocities", "GetImages", "GetForcesAndEnergies", "GetVirials"):
            np.testing.assert_array_equal(getattr(a, get)(), getattr(b, get)(), err_msg=f"{get} after {i} steps")
        assert itg_a.GetThermostatState() == itg_b.GetThermostatState()
        assert itg_a.GetKineticEnergy() == itg_b.GetKineticEnergy()
    if method != "none":
        assert keep_a[0].GetNumberOfNbListBuilds() == keep_b[0].GetNumberOfNbListBuilds() > 1


# the fused bonded step, the slot index that rebuilds keep and exclusions struck
# out by the build, together in captured blocks
@pytest.mark.parametrize("chains,copies,method,kinds", [
    (200, 1, "n2", ("BondHarmonic", "AngleCosSq", "DihedralRyckaert")),
    (200, 2, "sort", ("BondHarmonic", "AngleSq", "PeriodicDihedral")),
    (199, 3, "sort", ("BondHarmonic", "AngleCosSq"))])
def test_bonded_steps_with_exclusions_equal_the_separate_calls(golden_dir, chains, copies, method, kinds):
    print(f"[case] bonded steps with exclusions {5 * chains * copies ** 3} {method} {kinds}", flush=True)
    both = []
    for _ in range(2):
        s, itg, (pot, md) = _melt(golden_dir, chains, copies, method, kinds)
        for p in s.GetPotentials():
            if isinstance(p, rumd.BondHarmonic):
                p.SetParams(bond_type=0, bond_length=1.0, stiffness=100.0, exclude=True)
                p.SetParams(bond_type=1, bond_length=1.0, stiffness=100.0, exclude=True)
            if hasattr(p, "SetExclusions"):
                p.SetExclusions(pot)
        both.append((s, itg, pot, md))
    (a, itg_a, pot_a, _), (b, itg_b, pot_b, _) = both
    total = chains * copies ** 3
    gone = {(k, k + 1) for k in range(4)} | {(k, k + 2) for k in range(3)}  # bonds and the ends of angles
    ends = {(k, k + 3) for k in range(2)} if len(kinds) == 3 else set()     # and of every other chain's dihedrals
    assert pot_a.GetNumberOfExclusions() == total * len(gone) + (total + 1) // 2 * len(ends)
    i = 0
    for steps, block in ((7, 7), (1, 5), (24, 8), (16, 16)):
        a.RunSteps(i, steps, block, 20)
        for k in range(i, i + steps):
            if k % 20 == 0:
                itg_b.SetMomentumToZero()
            b.CalcF()
            itg_b.Integrate()
        i += steps
        b.Synchronize()
        for get in ("GetPositions", "GetVelocities", "GetImages", "GetForcesAndEnergies", "GetVirials"):
            np.testing.assert_array_equal(getattr(a, get)(), getattr(b, get)(), err_msg=f"{get} after {i} steps")
        assert itg_a.GetThermostatState() == itg_b.GetThermostatState()
    assert pot_a.GetNumberOfNbListBuilds() == pot_b.GetNumberOfNbListBuilds() > 1
    off, ids = pot_a.GetNeighborListCSR(a)
    first = np.repeat(np.arange(off.size - 1), np.diff(off))
    same = first // 5 == ids // 5
    lo, hi = np.minimum(first, ids)[same] % 5, np.maximum(first, ids)[same] % 5
    near = {(int(x), int(y)) for x, y in zip(lo, hi)}
    assert not near & gone
    even = (first[same] // 5) % 2 == 0
    assert not {(int(x), int(y)) for x, y in zip(lo[even], hi[even])} & ends


# the FP64 tile kernel's two workgroup sizes (small tiles and 4x4x4 cells)
@pytest.mark.parametrize("n", [9001, 33001, 130001])
def test_fp64_forces_at_each_workgroup_size(n):
    print(f"[case] fp64 tile shapes n={n}", flush=True)
    a, pot, _ = _stepping_sample(n, "sort", True, False)
    pot.SetFP64Forces(True)
    a.CalcF()
    pos4 = configs.pack_pos4(a.GetPositions(), a.GetTypes())
    box = np.array([a.GetSimulationBox().GetLength(k) for k in range(3)])
    f_ref, _ = oracle.forces_cells(pos4, box, 2, ka_table(), SF)
    # the output's rounding (2^-24) and the float parameters the oracle shares
    assert force_errors(a.GetForces(), f_ref[:, :3])["guarded_max"] <= 2e-7


def test_small_batches_are_cut_into_slot_ranges():
    """A batch of few large replicas takes slot ranges by default and whole
    replicas when asked, with the same bits."""
    systems = [configs.ka_random_lattice(n, density=1.2, temperature=0.9, seed=400 + n) for n in (4100, 3000)]
    out = []
    for fused in (False, True):
        b = make_batch(systems, [0.8, 1.5])
        if fused:
            b.SetFusedSteps(True)
        print(f"[case] small batch fused={fused}", flush=True)
        b.RunSteps(12, 10)
        assert b.UsesFusedSteps() == fused and b.GetFusedSteps()
        out.append([(b.GetPositions(r), b.GetVelocities(r), b.GetForcesAndEnergies(r)) for r in range(2)])
    for r in range(2):
        for k in range(3):
            np.testing.assert_array_equal(out[0][r][k], out[1][r][k], err_msg=f"replica {r} array {k}")
