"""The autotuner (qtp_autotune; no counterpart in the reference) over the kinds
of context it may be called on."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

pytestmark = pytest.mark.gpu


def _state(n_side, L_angs, P, seed):
    q0, box = cfg.lattice_water_box(n_side, L_angs, seed=seed, jitter_bohr=0.05)
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=seed + 1) if P > 1 else q0
    return q, cfg.sample_momenta(q0.size // 9, P, beta_n, seed=seed + 2), box


@pytest.mark.parametrize("P", [1, 2])
def test_autotune_without_matrix_kspace(P):
    """k_max 24: the vector k-space kernels only, so no slot groups of the
    matrix-core structure factors to split over blocks."""
    from qtip4pf_water_amd import Water
    q, p, box = _state(6, 18.64, P, 51)
    ew = {"kappa": 0.3 / cfg.ANGS2BOHR, "rcut": 9.0 * cfg.ANGS2BOHR,
          "k_cut": 2.0 * np.pi * 24.0 / float(box[0]) * (1.0 + 1e-9), "k_max": 24}
    with Water(216, P, box, ewald=ew) as w:
        w.set_state(q, p)
        F = w.get_state()[2]
        r = w.autotune(retime=True)
        assert r["timed"] >= 8 and r["chosen"]["matrix_kspace"] == 0
        assert r["best_ms"] <= r["default_ms"] * 1.001
        F2 = w.get_state()[2]
        assert np.max(np.abs(F2 - F)) < 1e-9 * np.max(np.abs(F))
        w.run(5)
        assert w.scalars()["status"] == 0


@pytest.mark.parametrize("start", [{}, {"rs_waves": 2}, {"ksum_blocks_per_chunk": 1}])
@pytest.mark.parametrize("P", [1, 4])
def test_autotune_times_the_one_stream_form(P, start):
    """From any starting configuration: the one-stream force phase with both
    lane counts and both force-block widths is among the candidates."""
    from qtip4pf_water_amd import Water
    q, p, box = _state(5, 15.54, P, 61)
    with Water(125, P, box, lj_rcut=cfg.lj_rcut_for(15.54)) as w:
        w.set_tuning(**start)
        w.set_state(q, p)
        a = w.timing("one_stream_phase")[1]
        F = w.get_state()[2]
        r = w.autotune(retime=True)
        # captured once a candidate: the four, each with every phase of a step
        assert w.timing("one_stream_phase")[1] - a >= 4 * (2 if P > 1 else 1)
        assert r["best_ms"] <= r["default_ms"] * 1.001
        F2 = w.get_state()[2]
        assert np.max(np.abs(F2 - F)) < 1e-9 * np.max(np.abs(F))
