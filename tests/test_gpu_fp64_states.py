"""State records of the FP64 kernel: hops from a recorded state and runs of hops
between two states take the events, totals and clock of evaluating every state.

Networks at +-300 kT visit many states (records are evicted, chunks of 64
entries are searched), low-bias ones few (leaps); sizes lie at the edges of the
site words, the record's search chunks and the kernel's limit.
"""
import numpy as np
import pytest

import oracle
from kmc_dn_amd import _lib, engine
from tests.netgen import random_network
from tests.test_zz_no_alloc import _call

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P,vmax", [(2, 2, 1.0), (8, 0, 1.0), (30, 8, 300.0), (63, 12, 300.0), (64, 16, 300.0),
                                      (65, 15, 2.0), (80, 0, 1.0)])
def test_events_equal_oracle(gpu_engine, N, P, vmax):
    net = random_network(11, N, P, M=max(1, N // 3), I_0=100.0 if vmax > 10 else 50.0, a=0.25, vmax=vmax)
    hops = 3000
    print(f"[gpu] FP64 records N={N} P={P} vmax={vmax}: {hops} hops", flush=True)
    u = oracle.stream_uniforms(99, 0, hops)
    args = (N, P, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"], net["E_constant"])
    ref = oracle.numba_simulate(*args, net["site_energies"].copy(), net["transitions_constant"], net["occupation"].copy(),
                                np.zeros(P, np.int64), hops, record=True, uniforms=np.asarray(u).ravel(), log=True)
    se, occ, eo = net["site_energies"].copy(), net["occupation"].copy(), np.zeros(P, np.int64)
    t, traffic, oit, ev, tot = engine.simulate_discrete(*args, se, net["transitions_constant"], occ, eo, hops, record=True,
                                                        seed=99, log=True)
    assert np.array_equal(ev, ref.events)
    assert np.array_equal(eo, ref.electrode_occupation) and np.array_equal(occ, ref.occupation)
    assert np.array_equal(traffic, ref.traffic)
    # the device's exp is within an ulp of the host's, as in the replay test
    assert abs(t - ref.time) <= 1e-12 * ref.time
    assert np.allclose(tot, ref.totals, rtol=1e-13, atol=0)
    assert np.allclose(oit, ref.occupations_in_time, rtol=1e-12, atol=0)
    assert np.allclose(se[:N], ref.site_energies[:N], rtol=1e-13, atol=1e-12)
    # fewer records (the allocation-free entry point's scratch): the same bits
    a, b = (_call(f, net, hops, None, 99) for f in ("kmc_simulate_discrete", "kmc_simulate_discrete_noalloc"))
    for k in a:
        assert np.array_equal(np.asarray(a[k]), np.asarray(b[k])), k


@pytest.mark.parametrize("N,P,K", [(10, 4, 9000), (60, 12, 700)])
def test_queued_batch_equals_single_runs(gpu_engine, N, P, K):
    """More trajectories than workgroups fit: those taken from the queue run as alone."""
    net = random_network(3, N, P, I_0=50.0, a=0.1, vmax=1.0)
    print(f"[gpu] FP64 queue: {K} trajectories of N={N}", flush=True)
    lay = engine.Layout(N, P, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"], net["transitions_constant"])
    es = lay.energy_sets(net["E_constant"], net["site_energies"][N:])
    b = engine.Batch(engine.make_trajs(K, lay.id, int(es[0]), np.arange(K, dtype=np.uint64), 150, net["occupation"],
                                       prehops=30))
    try:
        for _ in range(2):
            b.run(precision=_lib.FP64_DENSE, record=True)
            b.sync()
        r = b.results()
        one = engine.Batch(engine.make_trajs(40, lay.id, int(es[0]), np.arange(K - 40, K, dtype=np.uint64), 150,
                                             net["occupation"], prehops=30))
        one.run(precision=_lib.FP64_DENSE, record=True)
        one.sync()
        q = one.results()
        one.close()
        assert (r.status == 0).all() and (r.hops_done == 150).all()
        for f in ("time", "eo", "occ_bits", "occ_time"):
            assert np.array_equal(getattr(r, f)[-40:], getattr(q, f)), f
    finally:
        b.close()
        lay.close()
