"""The force phase's launch forms: the one-stream form of the resident steps
(k_phase_pairs, k_phase_reduce) against the kernels launched one by one, and
the pieces they share (fixed-point pair test of the real-space tiles,
structure-factor slot groups) against the oracle (forces.cpp:468-630) where
they can go wrong: boxes that are not cubic, molecules whole boxes away,
ragged last blocks, k-sets around the n-tile edges (2 k_max + 2 = 16, 32)."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

from energy_tol import single

pytestmark = pytest.mark.gpu

A = cfg.ANGS2BOHR


def _box(nside, seed, edge=3.107):
    L = [edge * n for n in nside]
    q, box = cfg.lattice_water_box(nside, L, seed=seed, jitter_bohr=0.1)
    return q, box, L


def rel_atom_err(F, Fr):
    d = np.linalg.norm((F - Fr).reshape(-1, 3), axis=1)
    return float(np.max(d / np.linalg.norm(Fr.reshape(-1, 3), axis=1)))


@pytest.mark.parametrize("nside,n_max", [
    ((4, 4, 4), 5), ((4, 5, 6), 7), ((7, 3, 5), 8), ((5, 5, 5), 15), ((6, 6, 7), 16), ((6, 6, 6), 23)])
def test_forces_follow_the_oracle(nside, n_max, oracle_mod):
    """Per-atom forces to 1e-10 and energies to 1e-12 of V, molecules moved by
    whole box vectors (the fixed-point wrap, the factor tables' reduction)."""
    from qtip4pf_water_amd import Water
    q, box, L = _box(nside, 5)
    n = q.size // 9
    rng = np.random.default_rng(7)
    q = (q.reshape(n, 3, 3) + rng.integers(-3, 4, (n, 1, 3)) * np.array(box)).reshape(-1)
    rc = min(9.0, 0.4999 * min(L)) * A
    ew = {"kappa": 2.9 / rc, "rcut": rc, "k_max": n_max,
          "k_cut": 2.0 * np.pi * n_max / max(box) * (1.0 + 1e-9)}
    lj = cfg.lj_rcut_for(min(L))
    o = oracle_mod.Oracle(n, 1, box, ewald=ew, lj_rcut=lj)
    point, lst, _ = o.all_lists(q)
    Fr = np.zeros_like(q)
    with oracle_mod.exact_energy():
        er = o.get_forces(q, Fr, point, lst, 0)
    with Water(n, 1, box, ewald=ew, lj_rcut=lj) as w:
        F = np.zeros_like(q)
        e = w.get_forces_nospline(q, F, o.charge, point, lst, 0)
        assert rel_atom_err(F, Fr) < 1e-10
        # terms of a few hundred Eh cancel here: a floor of epsilons of their size
        assert single(e, er) or abs(e - er) < 1e-11
        w.set_state(q, np.zeros_like(q))
        F2, W = w.get_state()[2], w.virial()
        assert rel_atom_err(F2, Fr) < 1e-10 and np.isfinite(W[0]).all()


@pytest.mark.parametrize("nside,P,thermo", [
    ((4, 4, 4), 1, None), ((6, 6, 6), 1, "pile_l"), ((4, 5, 6), 8, "pile_l"), ((6, 6, 6), 8, "pile_g"),
    ((7, 7, 8), 8, None)])
def test_one_stream_form_is_bitwise_the_kernels_one_by_one(nside, P, thermo):
    """Steps with per-kernel timing on launch the kernels one by one; without
    it the phase takes the one-stream form.  Same sums in the same order."""
    from qtip4pf_water_amd import Water
    q0, box, L = _box(nside, 11)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=12)
    p = cfg.sample_momenta(n, P, beta_n, seed=13)
    out = []
    for timing in (False, True):
        with Water(n, P, box, lj_rcut=cfg.lj_rcut_for(min(L))) as w:
            if thermo:
                w.set_thermostat(thermo, 100.0)
            # rebuilds on some steps, inside the phase's first launch
            w.set_lists("auto", 4)
            w.set_tuning(rs_registers=1)
            w.set_seed(3)
            w.enable_timing(timing)
            w.set_state(q, p)
            w.run(10, is_nvt=thermo is not None)
            s = w.scalars()
            assert s["status"] == 0 and s["rebuilds"] >= 2 * P
            out.append((w.get_state(), w.get_lists(), s, w.virial()))
    a, b = out
    assert all(np.array_equal(x, y) for x, y in zip(a[0], b[0]))
    assert all(np.array_equal(x, y) for x, y in zip(a[1], b[1]))
    assert a[2] == b[2]
    assert all(np.array_equal(x, y) for x, y in zip(a[3], b[3]))


@pytest.mark.parametrize("nside,P", [
    ((4, 4, 4), 4), ((4, 4, 5), 2), ((8, 8, 8), 1), ((8, 9, 9), 2), ((9, 10, 11), 2), ((8, 8, 16), 1)])
def test_spread_rebuild_is_the_one_block_rebuild(nside, P):
    """Lists rebuilt inside the one-stream phase (bitmaps, then offsets and
    rows, over many blocks) against k_nlist_bead's: rows up to the largest
    molecule count, whole and ragged words and blocks of rows."""
    from qtip4pf_water_amd import Water
    q0, box, L = _box(nside, 21)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=22) if P > 1 else q0
    p = cfg.sample_momenta(n, P, beta_n, seed=23)
    out = []
    for timing in (False, True):
        with Water(n, P, box, lj_rcut=cfg.lj_rcut_for(min(L))) as w:
            w.set_lists("allpairs", 2)
            w.set_tuning(rs_registers=1)
            w.set_seed(3)
            w.enable_timing(timing)
            w.set_state(q, p)
            w.run(5)
            s = w.scalars()
            # every second step, and where the beads moved far enough
            assert s["status"] == 0 and s["rebuilds"] >= 2 * P
            out.append((w.get_lists(), w.get_state(), s))
    a, b = out
    assert a[2] == b[2]
    for x, y in zip(a[0] + a[1], b[0] + b[1]):
        assert np.array_equal(x, y)


def _ewald(box, rc_angs, n_max=6):
    rc = rc_angs * A
    return {"kappa": 2.9 / rc, "rcut": rc, "k_max": n_max,
            "k_cut": 2.0 * np.pi * n_max / max(box) * (1.0 + 1e-9)}


@pytest.mark.parametrize("nside,edge,P", [((7, 10, 14), 3.107, 32), ((8, 8, 8), 2.6, 2), ((6, 7, 8), 3.107, 4)])
def test_culled_tiles_in_groups(nside, edge, P, oracle_mod):
    """Boxes past the culling threshold: several tiles a block with a ragged
    last group (980 H2O x 32: 1081 tiles, two a block; one bead alone: one a
    block), boxes that are and are not cubic, and more pairs in a wave's half
    of a tile than its queue holds (512 at 2.6 A a molecule)."""
    from qtip4pf_water_amd import Water
    q0, box, L = _box(nside, 31, edge)
    n = q0.size // 9
    rc = min(L) / 2.51
    lj = cfg.lj_rcut_for(min(L))
    if edge < 3.0:  # molecules in lattice order: close blocks of 64 sites
        x = q0.reshape(3 * n, 3)
        most = 0
        for J in range(1, 8):
            d = x[64 * (J - 1):64 * J, None] - x[None, 64 * J:64 * J + 32]
            d -= np.array(box) * np.rint(d / np.array(box))
            most = max(most, int(np.count_nonzero((d * d).sum(-1) < (rc * A) ** 2)))
        assert most > 1024
    q = cfg.replicate_beads(q0, P) + np.random.default_rng(32).normal(0, 0.03, P * 9 * n)
    o = oracle_mod.Oracle(n, P, box, ewald=_ewald(box, rc), lj_rcut=lj)
    point, lst, _ = o.all_lists(q)
    with Water(n, P, box, ewald=_ewald(box, rc), lj_rcut=lj) as w:
        F, f = np.zeros_like(q), np.zeros_like(q)
        w.force_eval_sc_nospline(q, F, o.charge, o.mass, point, lst, fphys=f)
        for b in (0, P - 1):
            sl = slice(9 * n * b, 9 * n * (b + 1))
            F1, Fr = np.zeros_like(q), np.zeros_like(q)
            w.get_forces_nospline(q, F1, o.charge, point, lst, b)
            o.get_forces(q, Fr, point, lst, b)
            assert rel_atom_err(F1[sl], Fr[sl]) < 1e-10
            assert rel_atom_err(f[sl], F1[sl]) < 1e-10


@pytest.mark.parametrize("nside,P,thermo,mode", [
    ((4, 4, 4), 2, "pile_l", None), ((4, 4, 5), 6, None, None), ((6, 6, 6), 32, "pile_l", None),
    ((4, 5, 6), 64, "pile_l", "pacmd"), ((5, 5, 5), 8, "pile_g", "centroid_fixed")])
def test_propagation_forms_agree_bitwise(nside, P, thermo, mode):
    """One launch with a thread per (mode, dof) (the default of small systems)
    against the two-kernel form: same operations in the same
    order, the heat included."""
    from qtip4pf_water_amd import Water
    q0, box, L = _box(nside, 41)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=42)
    p = cfg.sample_momenta(n, P, beta_n, seed=43)
    out = []
    for fused in (-1, 0, 1):
        with Water(n, P, box, dtfs=0.1, lj_rcut=cfg.lj_rcut_for(min(L))) as w:
            if thermo:
                w.set_thermostat(thermo, 100.0)
            if mode:
                w.set_pimd_mode(mode)
            w.set_tuning(fused_propagation=fused, rs_registers=1)
            w.set_seed(5)
            w.set_state(q, p)
            w.run(4, is_nvt=thermo is not None)
            out.append((w.get_state(), w.scalars()))
    for st, sc in out[1:]:
        assert all(np.array_equal(x, y) for x, y in zip(st, out[0][0]))
        assert sc == out[0][1]
