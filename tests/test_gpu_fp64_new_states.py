"""FP64 trajectories that find a new state on nearly every hop: events selected without
a record, tags that come back, and what keeping them may cost."""
import ctypes as C

import numpy as np
import pytest

import oracle
from kmc_dn_amd import _lib, engine
from tests.netgen import fixture_network, random_network

pytestmark = pytest.mark.gpu

DIFFUSE = dict(I_0=1.0, a=1.0, vmax=1.0)


@pytest.mark.parametrize("N,P", [(3, 2), (5, 0), (16, 4), (30, 8), (63, 12), (64, 16), (80, 0)])
def test_events_equal_oracle(gpu_engine, N, P):
    """From networks whose few states all come back (N = 3) to ones where none does."""
    net = random_network(21, N, P, M=max(1, N // 3), **DIFFUSE)
    hops = 2000
    print(f"[gpu] FP64 new states N={N} P={P}: {hops} hops", flush=True)
    u = oracle.stream_uniforms(7, 0, hops)
    args = (N, P, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"], net["E_constant"])
    ref = oracle.numba_simulate(*args, net["site_energies"].copy(), net["transitions_constant"], net["occupation"].copy(),
                                np.zeros(P, np.int64), hops, record=True, uniforms=np.asarray(u).ravel(), log=True)
    se, occ, eo = net["site_energies"].copy(), net["occupation"].copy(), np.zeros(P, np.int64)
    t, traffic, oit, ev, tot = engine.simulate_discrete(*args, se, net["transitions_constant"], occ, eo, hops, record=True,
                                                        seed=7, log=True)
    assert np.array_equal(ev, ref.events)
    assert np.array_equal(eo, ref.electrode_occupation) and np.array_equal(occ, ref.occupation)
    assert np.array_equal(traffic, ref.traffic)
    # the device's exp is within an ulp of the host's
    assert abs(t - ref.time) <= 1e-12 * ref.time
    assert np.allclose(tot, ref.totals, rtol=1e-13, atol=0)
    assert np.allclose(oit, ref.occupations_in_time, rtol=1e-12, atol=0)


def test_new_states_cost_little_besides_their_evaluation(gpu_engine):
    """The phases of a hop besides the evaluation (energies, pair lists with the lookup,
    rates, prefix chain) take less than a seventh of it (storing every record: a fifth)."""
    net = random_network(7, 30, 8, **DIFFUSE)
    lay = engine.Layout(30, 8, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"], net["transitions_constant"])
    es = lay.energy_sets(net["E_constant"], net["site_energies"][30:])
    b = engine.Batch(engine.make_trajs(1, lay.id, int(es[0]), np.arange(1, dtype=np.uint64), 4000, net["occupation"]))
    print("[gpu] FP64 phases of new states", flush=True)
    c = (C.c_uint64 * 7)()
    for _ in range(2):
        _lib.check(_lib.load().kmc_probe_fp64_phases(b.id, c, 7))
    b.close()
    lay.close()
    assert sum(c[4:]) < sum(c[:4]) / 7, list(c)


def test_records_beyond_a_trajectory_per_cu(gpu_engine, fixtures):
    """One trajectory fewer than CUs and two more, of a fixture network at +-300 kT: as many
    records each (64 instead, and the evicted states evaluated again, take 1.5 times
    as long)."""
    net = fixture_network(fixtures, "rnd", 4)
    lay = engine.Layout(30, 8, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"], net["transitions_constant"])
    es = lay.energy_sets(net["E_constant"], net["site_energies"][30:])
    cus = engine.device_info()["cu_count"]
    ms = []
    for K in (cus - 1, cus + 2):
        b = engine.Batch(engine.make_trajs(K, lay.id, int(es[0]), np.arange(K, dtype=np.uint64), 4000, net["occupation"]))
        print(f"[gpu] FP64 records: {K} trajectories", flush=True)
        took = []
        for _ in range(3):
            b.run(precision=_lib.FP64_DENSE)
            took.append(b.sync())
        ms.append(min(took[1:]))
        b.close()
    lay.close()
    assert ms[1] < 1.2 * ms[0], ms
