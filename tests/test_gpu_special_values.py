"""Pair terms at the values a run can meet when it goes wrong: positions that are
infinite or not a number, and particles at the same place."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import oracle
from capi import GpuSystem, check, gpu_available, lib
from helpers import force_errors, ka_table, unsort
from test_gpu_potentials import PE_ATOL, _forms, _table
from rumd_amd import configs

pytestmark = pytest.mark.gpu

NS, SP, SF = 0, 1, 2


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    if not gpu_available():
        pytest.fail("no GPU visible: the gpu tests must run on an MI355X")


def _ka(n):
    s = configs.ka_random_lattice(n, density=1.2, seed=7)
    rng = np.random.default_rng(8)
    pos = s.positions + rng.uniform(-0.02, 0.02, size=s.positions.shape)
    pos -= s.box * np.rint(pos / s.box)
    return s, configs.pack_pos4(pos.astype(np.float32), s.types)


def _gpu(s, pos4, method, table, **kw):
    return GpuSystem(pos4, configs.pack_vel4(s.velocities, s.types, s.masses), configs.box8(s.box), 2, table,
                     method=method, **kw)


# tiles in FP64 displacements (2500) and in the shifted frame (19001), slot lists, all pairs
@pytest.mark.parametrize("method,n", [("sorted", 2500), ("sorted", 19001), ("n2", 1003), ("none", 333)])
@pytest.mark.parametrize("cutoff", [NS, SP, SF])
def test_fp64_forces_leave_out_particles_without_a_position(method, n, cutoff):
    """Particles that leave the finite numbers after the list was built act on
    none of their listed neighbours, nor these on them."""
    s, pos4 = _ka(n)
    g = _gpu(s, pos4, method, ka_table(), with_sts=True, **({"max_nbrs": 200} if method != "none" else {}))
    print(f"[case] fp64 {method} n={n} cutoff={cutoff} lost positions", flush=True)
    if g.nb is not None:
        g.update_nblist()
    r = g.r.download(np.float32, (g.nvp, 4))
    lost = {int(n // 3): (np.nan, 0), int(n // 2): (np.inf, 1), int(n - 1): (-np.inf, 2)}
    for slot, (x, axis) in lost.items():
        r[slot, axis] = x
    g.r.upload(r)
    check(lib().rumdx_pair_lj_fp64(C.byref(g.p), C.byref(g.nb) if g.nb is not None else None, g.d_params.value, 2,
                                   g.box8, cutoff, 1, 1, None))
    kept = np.setdiff1d(np.arange(n), list(lost))
    f_ref, _ = oracle.forces_brute(r[kept], s.box, 2, ka_table(), cutoff) if n < 5000 else \
        oracle.forces_cells(r[kept], s.box, 2, ka_table(), cutoff)
    f, w, sts = g.get("f"), g.get("w"), g.get("sts")
    for a in (f, w, sts):
        assert np.isfinite(a).all()
        assert not a[list(lost)].any()
    assert force_errors(f[kept, :3], f_ref[:, :3])["guarded_max"] <= 2e-7  # as for all FP64 forces
    np.testing.assert_allclose(f[kept, 3], f_ref[:, 3], rtol=0, atol=2e-7 * np.abs(f_ref[:, 3]).max())


@pytest.mark.parametrize("method", ["sorted", "n2", "none"])
@pytest.mark.parametrize("cutoff", [NS, SP, SF])
def test_fp64_energy_of_coincident_particles(method, cutoff):
    s, pos4 = _ka(1003)
    j = int(np.flatnonzero(s.types == s.types[0])[1])
    pos4[j] = pos4[0]
    g = _gpu(s, pos4, method, ka_table())
    print(f"[case] fp64 {method} cutoff={cutoff} coincident particles", flush=True)
    g.calc_f(cutoff, fp64=True)
    u = unsort(g.get("f"), g.unsorted_index())[:, 3]
    assert np.isposinf(u[[0, j]]).all()
    assert np.isfinite(np.delete(u, [0, j])).all()


# forms that have a value or an infinity of one sign at zero distance
_AT_ZERO = ["smooth_2_4", "Gauss", "Buckingham", "IPL_18", "Yukawa", "Exp", "LJ_Gauss", "IPL_12", "IPL_9",
            "IPL_18_class", "Dzugutov", "Fermi_Jagla", "Repulsive_Shoulder", "SAAP", "SF_Coulomb"]


@pytest.mark.parametrize("stress", [False, True])  # compiled per form, and with the form as an argument
@pytest.mark.parametrize("method", ["sorted", "n2", "none"])
@pytest.mark.parametrize("case", [c for c in _forms() if c[0] in _AT_ZERO], ids=lambda c: c[0])
def test_form_energy_of_coincident_particles(case, method, stress):
    name, form, make, rows = case
    table = _table(make, NS, rows)
    s, pos4 = _ka(1003)
    j = int(np.flatnonzero(s.types == s.types[0])[1])
    pos4[j] = pos4[0]
    # of the pair alone, at a distance where the form has reached its limit (or is beyond any float)
    near = np.stack([pos4[0], pos4[0]])
    near[:, :3] = 0.0
    near[1, 0] = 1e-8
    pair = 2.0 * oracle.forces_form_brute(near, s.box, 2, table, form, NS)[0][0, 3]
    rest = oracle.forces_form_brute(np.delete(pos4, j, axis=0), s.box, 2, table, form, NS)[0]
    g = _gpu(s, pos4, method, table, with_sts=stress)
    print(f"[case] form {name} {method} stress={stress} coincident particles", flush=True)
    g.calc_f(NS, form=form, stress=stress)
    u = unsort(g.get("f"), g.unsorted_index())[:, 3]
    if name in ("Gauss", "Exp"):
        want = rest[0, 3] + 0.5 * pair
        np.testing.assert_allclose(u[[0, j]], want, rtol=0, atol=max(PE_ATOL, 2e-6 * abs(want)))
    else:
        assert (u[[0, j]] == np.copysign(np.inf, pair)).all(), (u[[0, j]], pair)
    assert np.isfinite(np.delete(u, [0, j])).all()
