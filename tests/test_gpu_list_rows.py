"""Half-list rows as the host-array calls leave them: a rebuilt row is its
entries and zeros behind them, as neighbour.cpp:23-32 writes it, whichever
call rebuilt it, and a row that was not rebuilt is left alone."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

pytestmark = pytest.mark.gpu


def _system(nside, P, edge=3.107, seed=4):
    L = [edge * n for n in nside]
    q0, box = cfg.lattice_water_box(nside, L, seed=seed, jitter_bohr=0.1)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=seed + 1) if P > 1 else q0
    return n, q, box, cfg.lj_rcut_for(min(L))


def _lists(w, q, P, n):
    point, lst = np.zeros(P * n, np.int32), np.zeros(P * w.list_size, np.int32)
    for b in range(P):
        w.neighbour_list(q, point, lst, None, b)
    return point, lst


@pytest.mark.parametrize("nside,P", [
    ((4, 4, 4), 1), ((4, 4, 5), 2), ((6, 6, 6), 4), ((9, 10, 11), 1), ((10, 11, 10), 1), ((10, 11, 10), 2)])
def test_rebuilt_rows_come_back_whole(nside, P):
    """Every other bead's displacements ask for a rebuild; the caller's rows
    are full to the end before the step."""
    from qtip4pf_water_amd import Water
    n, q, box, lj = _system(nside, P)
    with Water(n, P, box, lj_rcut=lj) as w:
        N = w.list_size
        point, lst = _lists(w, q, P, n)
        for b in range(P):
            assert point[(b + 1) * n - 1] < N
            lst[b * N + point[(b + 1) * n - 1]:(b + 1) * N] = n - 1
        point0, lst0 = point.copy(), lst.copy()
        disp = np.zeros(P * 3 * n)
        for b in range(0, P, 2):
            disp[3 * n * b:3 * n * b + 6] = 100.0
        p, F, fph = np.zeros_like(q), np.zeros_like(q), np.zeros_like(q)
        if P == 1:
            w.update_trajectory_class_nospline(q, p, None, F, None, point, lst, disp)
        else:
            w.update_sc_nospline(q, p, None, F, fph, None, point, lst, disp, None, False, 0.0)
        got_p, got_l = w.get_lists()
        want_p, want_l = _lists(w, q, P, n)
        for b in range(P):
            rp, rl = slice(b * n, (b + 1) * n), slice(b * N, (b + 1) * N)
            if b % 2 == 0:
                assert np.array_equal(point[rp], want_p[rp]) and np.array_equal(lst[rl], want_l[rl])
                assert np.array_equal(got_p[rp], want_p[rp]) and np.array_equal(got_l[rl], want_l[rl])
                assert not disp[3 * n * b:3 * n * (b + 1)].any()
            else:
                assert np.array_equal(point[rp], point0[rp]) and np.array_equal(lst[rl], lst0[rl])


@pytest.mark.parametrize("nside,P", [((4, 4, 4), 1), ((4, 4, 5), 4), ((9, 10, 11), 2), ((10, 11, 10), 2)])
def test_lists_held_are_the_callers(nside, P):
    """A call on host arrays replaces the rows that the context held, the part
    before and behind the entries with them: here rows of half the entries,
    from list[3] on."""
    from qtip4pf_water_amd import Water
    n, q, box, lj = _system(nside, P)
    with Water(n, P, box, lj_rcut=lj) as w:
        N = w.list_size
        point, lst = _lists(w, q, P, n)
        for b in range(P):
            pt, row = point[b * n:(b + 1) * n], lst[b * N:(b + 1) * N]
            rows = [row[pt[i]:(pt[i] + pt[i + 1]) // 2] for i in range(n - 1)]
            flat = np.concatenate(rows)
            assert flat.size + 13 < pt[n - 1]
            row[:] = 0
            row[3:3 + flat.size] = flat
            pt[:] = 3 + np.concatenate([[0], np.cumsum([r.size for r in rows])])
        F = np.zeros_like(q)
        if P == 1:
            w.get_forces_nospline(q, F, None, point, lst, 0)
        else:
            w.force_eval_sc_nospline(q, F, None, None, point, lst)
        got_p, got_l = w.get_lists()
        assert np.array_equal(got_p, point)
        assert np.array_equal(got_l, lst)
