"""Caller's arrays through the packed transfers and the device expansion of the
half lists (forces.cpp:489 reads the half rows; the device sums full rows):
ragged sizes, rows with more than a wave of incoming partners, packed sizes of
several chunks, and the host path beyond 1024 molecules."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

pytestmark = pytest.mark.gpu


def _system(nside, P):
    L = [3.107 * n for n in nside]
    q0, box = cfg.lattice_water_box(nside, L, seed=4, jitter_bohr=0.1)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=5) if P > 1 else q0
    return q, cfg.sample_momenta(n, P, beta_n, seed=6), box, cfg.lj_rcut_for(min(L)), n


@pytest.mark.parametrize("nside,P", [
    ((4, 4, 4), 2), ((4, 4, 5), 4), ((5, 5, 5), 8), ((6, 6, 6), 4), ((7, 8, 9), 16), ((9, 10, 11), 2),
    ((10, 11, 10), 2)])
def test_caller_lists_give_the_resident_forces(nside, P):
    """The lists a resident state holds, handed back by the caller: the same
    full rows in the same order, so the same forces to the last bit."""
    from qtip4pf_water_amd import Water
    q, p, box, lj, n = _system(nside, P)
    with Water(n, P, box, lj_rcut=lj) as w:
        w.set_state(q, p)
        q1, p1, F, fph, disp = w.get_state()
        assert np.array_equal(q1.ravel(), q) and np.array_equal(p1.ravel(), p)
        assert not disp.any()
        point, lst = w.get_lists()
        F2, fph2 = np.zeros_like(q), np.zeros_like(q)
        w.force_eval_sc_nospline(q, F2, None, None, point, lst, fph2)
        assert np.array_equal(F2, F.ravel()) and np.array_equal(fph2, fph.ravel())


def test_caller_lists_in_any_row_order(oracle_mod):
    """Rows in any order, entries that start past list[0], against the oracle
    with the same arrays."""
    from qtip4pf_water_amd import Water
    q, _, box, lj, n = _system((6, 5, 7), 1)
    o = oracle_mod.Oracle(n, 1, box, lj_rcut=lj)
    point, lst, _ = o.all_lists(q)
    rng = np.random.default_rng(8)
    for i in range(n - 1):
        rng.shuffle(lst[point[i]:point[i + 1]])
    used = point[n - 1]
    lst[3:used + 3] = lst[:used].copy()
    point += 3
    Fr, F = np.zeros_like(q), np.zeros_like(q)
    o.get_forces(q, Fr, point, lst, 0)
    with Water(n, 1, box, lj_rcut=lj) as w:
        w.get_forces_nospline(q, F, o.charge, point, lst, 0)
        d = np.linalg.norm((F - Fr).reshape(-1, 3), axis=1)
        assert np.max(d / np.linalg.norm(Fr.reshape(-1, 3), axis=1)) < 1e-10
        # refused as before, and the context goes on
        for at, what in ((0, n), (used, -1)):
            bad = lst.copy()
            bad[point[0] + at - (at > 0)] = what
            with pytest.raises(Exception, match="entry out of range"):
                w.get_forces_nospline(q, F, o.charge, point, bad, 0)
        bad = point.copy()
        bad[n // 2] = lst.size + 1
        with pytest.raises(Exception, match="point"):
            w.get_forces_nospline(q, F, o.charge, bad, lst, 0)
        F3 = np.zeros_like(q)
        w.get_forces_nospline(q, F3, o.charge, point, lst, 0)
        w.get_forces_nospline(q, F, o.charge, point, lst, 0)
        assert np.array_equal(F, F3)


def test_caller_lists_with_repeated_entries(oracle_mod):
    """Lists the caller may pass though no builder writes them: a pair listed
    twice counts twice, a row that many others list, rows left empty."""
    from qtip4pf_water_amd import Water
    q, _, box, lj, n = _system((4, 5, 6), 1)
    o = oracle_mod.Oracle(n, 1, box, lj_rcut=lj)
    point, lst, _ = o.all_lists(q)
    full = [list(lst[point[i]:point[i + 1]]) for i in range(n - 1)]
    rows = [r + r if i % 3 == 0 else [] if i % 7 == 1 else r for i, r in enumerate(full)]
    # every pair of the second half of the molecules with the last one, often
    rows = [r + [n - 1] * (20 if i >= n // 2 else 0) for i, r in enumerate(rows)]
    flat = [j for r in rows for j in r]
    assert len(flat) <= lst.size and flat.count(n - 1) > 1024
    lst[:] = 0
    lst[:len(flat)] = flat
    point[:] = np.concatenate([[0], np.cumsum([len(r) for r in rows])])
    Fr, F = np.zeros_like(q), np.zeros_like(q)
    o.get_forces(q, Fr, point, lst, 0)
    with Water(n, 1, box, lj_rcut=lj) as w:
        w.get_forces_nospline(q, F, o.charge, point, lst, 0)
    d = np.linalg.norm((F - Fr).reshape(-1, 3), axis=1)
    assert np.max(d / np.linalg.norm(Fr.reshape(-1, 3), axis=1)) < 1e-10
