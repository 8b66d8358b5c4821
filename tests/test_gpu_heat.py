"""The thermostat's heat (pile_g's return value, thermostat.cpp:86-129), which
is summed over groups of sixteen dofs and then over the modes: bead counts
around multiples of sixteen, up to those that one block of the one-launch
propagation takes and beyond."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

pytestmark = pytest.mark.gpu


def _system(nside, P, seed):
    L = [3.107 * n for n in nside]
    q0, box = cfg.lattice_water_box(nside, L, seed=seed, jitter_bohr=0.05)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    return n, cfg.free_ring_polymer_beads(q0, P, beta_n, seed=seed + 1), \
        cfg.sample_momenta(n, P, beta_n, seed=seed + 2), box, cfg.lj_rcut_for(min(L))


@pytest.mark.parametrize("nside,P", [
    ((3, 3, 3), 2), ((3, 4, 3), 14), ((3, 3, 3), 16), ((3, 3, 3), 18), ((4, 3, 3), 34), ((3, 3, 3), 64),
    ((3, 3, 3), 66)])
def test_heat_of_a_step_follows_the_oracle(nside, P, oracle_mod):
    """pile_g steps with the caller's random numbers.  Momenta agree to 1e-10
    of their size at worst (the parity bound), so the heat to twice that of
    the kinetic energy."""
    from qtip4pf_water_amd import HostRng, Water
    n, q, p, box, lj = _system(nside, P, 3)
    o = oracle_mod.Oracle(n, P, box, lj_rcut=lj)
    point, lst, disp = o.all_lists(q)
    F, fph = np.zeros(P * o.n_dof), np.zeros(P * o.n_dof)
    o.force_eval_sc(q, F, fph, point, lst)
    ref = [q.copy(), p.copy(), F.copy(), fph.copy(), point.copy(), lst.copy(), disp.copy()]
    gpu = [a.copy() for a in ref]
    rng = HostRng(5)
    hr = hg = 0.0
    with Water(n, P, box, lj_rcut=lj) as w:
        for _ in range(2):
            ke = float(np.sum(0.5 * ref[1].reshape(P, -1) ** 2 / o.mass))
            dev = rng.draw_pile(o.n_atoms, P)
            _, hr, _, _ = o.update_sc(*ref, True, dev, hr)
            _, hg, _ = w.update_sc_nospline(gpu[0], gpu[1], o.mass, gpu[2], gpu[3], o.charge, gpu[4],
                                            gpu[5], gpu[6], dev, True, hg)
            assert abs(hr) > 1e-3 * ke
            assert abs(hg - hr) <= 2e-10 * ke


@pytest.mark.parametrize("nside,P", [((3, 4, 3), 14), ((3, 3, 3), 18), ((4, 4, 4), 34), ((10, 11, 10), 18)])
def test_heat_is_the_same_in_both_forms(nside, P):
    """One launch for the propagation against two: the same bits, whichever
    kernel adds the groups (the list check's up to 1024 molecules, k_heat's)."""
    from qtip4pf_water_amd import Water
    n, q, p, box, lj = _system(nside, P, 7)
    out = []
    for fused in (-1, 0):
        with Water(n, P, box, lj_rcut=lj) as w:
            w.set_thermostat("pile_l", 100.0)
            w.set_tuning(fused_propagation=fused)
            w.set_seed(5)
            w.set_state(q, p)
            w.run(3, is_nvt=True)
            out.append((w.scalars(), w.get_state()))
    assert out[0][0] == out[1][0] and out[0][0]["heat"] != 0.0
    assert all(np.array_equal(a, b) for a, b in zip(out[0][1], out[1][1]))
