"""Which form of the force phase a context takes: the systems whose one-stream
form test_gpu_phase_forms.py compares with the kernels one by one do take it,
and what the form does not cover takes the two streams."""
import numpy as np
import pytest

from qtip4pf_water_amd import config as cfg

pytestmark = pytest.mark.gpu


def _run(nside, P, method="auto", every=0, timing=False, tuning=None, ewald=None):
    """Phases queued in the one-stream form by set_state and by a run."""
    from qtip4pf_water_amd import Water
    L = [3.107 * n for n in nside]
    q0, box = cfg.lattice_water_box(nside, L, seed=11, jitter_bohr=0.1)
    n = q0.size // 9
    beta_n = 1.0 / (cfg.K2AU * 298.0) / P
    q = cfg.free_ring_polymer_beads(q0, P, beta_n, seed=12) if P > 1 else q0
    p = cfg.sample_momenta(n, P, beta_n, seed=13)
    with Water(n, P, box, lj_rcut=cfg.lj_rcut_for(min(L)), ewald=ewald(L) if ewald else None) as w:
        w.set_lists(method, every)
        if tuning:
            w.set_tuning(**tuning)
        w.enable_timing(timing)
        w.set_state(q, p)
        a = w.timing("one_stream_phase")[1]
        w.run(3)
        s = w.scalars()
        assert s["status"] == 0
        return a, w.timing("one_stream_phase")[1] - a


@pytest.mark.parametrize("nside,P,method,every", [
    # the steps compared bit for bit
    ((4, 4, 4), 1, "auto", 4), ((6, 6, 6), 1, "auto", 4), ((4, 5, 6), 8, "auto", 4),
    ((6, 6, 6), 8, "auto", 4), ((7, 7, 8), 8, "auto", 4),
    # the rebuilds compared with one block's
    ((4, 4, 4), 4, "allpairs", 2), ((4, 4, 5), 2, "allpairs", 2), ((8, 8, 8), 1, "allpairs", 2),
    ((8, 9, 9), 2, "allpairs", 2), ((9, 10, 11), 2, "allpairs", 2), ((8, 8, 16), 1, "allpairs", 2)])
def test_one_stream_form_is_taken(nside, P, method, every):
    phases = 2 if P > 1 else 1
    tuning = {"rs_registers": 1}
    # the run queues one step, captured once
    assert _run(nside, P, method, every, tuning=tuning) == (phases, phases)
    assert _run(nside, P, method, every, timing=True, tuning=tuning) == (0, 0)


def _narrow(L):
    """r_c so short that tiles are culled (the box is 2.51 r_c wide)."""
    rc = min(L) / 2.51 * cfg.ANGS2BOHR
    return {"kappa": 2.9 / rc, "rcut": rc, "k_max": 6,
            "k_cut": 2.0 * np.pi * 6 / (max(L) * cfg.ANGS2BOHR) * (1.0 + 1e-9)}


@pytest.mark.parametrize("kw", [
    {"tuning": {"rs_waves": 2}}, {"tuning": {"rs_registers": 0}}, {"tuning": {"rs_split": 1}},
    {"tuning": {"matrix_kspace": 0}}, {"tuning": {"ksum_blocks_per_chunk": 1}},
    {"tuning": {"ksum_chunks_per_block": 2}}, {"ewald": _narrow}])
def test_two_streams_otherwise(kw):
    assert _run((6, 6, 6), 2, **kw) == (0, 0)


@pytest.mark.parametrize("lanes,w16", [(16, 0), (16, 1), (64, 0), (64, 1), (64, -1)])
def test_choices_within_the_one_stream_form(lanes, w16):
    assert _run((6, 6, 6), 2, tuning={"lanes": lanes, "kforce_16_waves": w16}) == (2, 2)
