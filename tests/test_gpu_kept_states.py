"""How the FP32 kernels take a hop changes no bit of a trajectory.

Hops by kept transitions, leaps and looked-up states, intervals of general steps
(for trajectories that find a new state on most hops), and the kernels that give
each trajectory one wave per site chunk all produce the same clock, tallies,
occupation and records.  The tests compare runs that take the same hops in
different ways, bit for bit: a launch capped by grid_limit gives every trajectory
one wave; each resumed range of one recompute interval starts with kept
transitions whatever the interval before found; and state_store sets how many
states a one-chunk trajectory keeps (-1: two, so states are taken over all the
time).
"""
import numpy as np
import pytest

from kmc_dn_amd import _lib, engine
from tests.netgen import random_network
from tests.test_gpu_fp32 import _positions

pytestmark = pytest.mark.gpu

LOCAL = dict(I_0=50.0, a=0.1)    # few states, many returns
DIFFUSE = dict(I_0=1.0, a=1.0)   # nearly every hop finds a new state


def _layout(N, P, **kw):
    net = random_network(N + P, N, P, vmax=1.0, **kw)
    lay = engine.Layout(N, P, net["nu"], net["kT"], net["I_0"], net["R"], net["distances"],
                        net["transitions_constant"])
    lay.set_positions(kw["a"] * net["R"], _positions(net))
    es = lay.energy_sets(net["E_constant"], net["site_energies"][N:])
    return net, lay, es[0]


def _run(trajs, chunk=None, sizes=None, **opts):
    """Results (and traffic) of the trajectories, whole or in resumed ranges of `chunk` hops."""
    b = engine.Batch(trajs)
    total = int((trajs["prehops"] + trajs["hops"]).max())
    if chunk is None:
        b.run(precision=_lib.FP32_BATCHED, **opts)
        b.sync()
    else:
        for h in range(0, total, chunk):
            ends = np.minimum(h + chunk, trajs["prehops"] + trajs["hops"])
            b.set_state(h_begin=np.minimum(h, ends), h_end=ends)
            b.run(precision=_lib.FP32_BATCHED, resume=True, **opts)
            b.sync()
    r = b.results()
    assert (r.status == 0).all()
    out = [r.time.view(np.uint64), r.eo, r.occ_bits, r.hops_done]
    if opts.get("record"):
        out.append(r.occ_time.view(np.uint64))
    if opts.get("traffic"):
        out += b.traffic(sizes)
    out = [np.array(x) for x in out]
    b.close()
    return out


def _same(x, y, what):
    assert len(x) == len(y)
    for i, (a, b) in enumerate(zip(x, y)):
        assert np.array_equal(a, b), (what, i)


@pytest.mark.parametrize("N,P,form", [(57, 8, 1), (57, 8, 2), (57, 8, 3), (120, 8, 2), (121, 8, 3),
                                      (180, 12, 3)])
@pytest.mark.parametrize("kind", [LOCAL, DIFFUSE])
def test_a_wave_per_chunk_equals_one_wave(gpu_engine, N, P, form, kind):
    """S = 65, 128, 129 and 192 beside a network of one chunk (S = 24)."""
    print(f"[gpu] one wave per chunk: S={N + P} form {form} {kind}", flush=True)
    big, lb, eb = _layout(N, P, **kind)
    small, ls, e_small = _layout(16, 8, **kind)
    t = np.concatenate([
        engine.make_trajs(5, lb.id, eb, np.arange(5, dtype=np.uint64), 3000, big["occupation"],
                          prehops=100),
        engine.make_trajs(3, ls.id, e_small, np.arange(3, dtype=np.uint64), 4000,
                          small["occupation"])])
    sizes = [N + P] * 5 + [24] * 3
    for rec in (False, True):
        opts = dict(table_form=form, record=rec, traffic=rec)
        one = _run(t, sizes=sizes, grid_limit=64, **opts)
        _same(one, _run(t, sizes=sizes, **opts), (N, form, rec))
    _same(_run(t, table_form=form), _run(t, chunk=1024, table_form=form), (N, form, "resumed"))
    lb.close()
    ls.close()


@pytest.mark.parametrize("N,P,form,team", [(16, 4, 1, 1), (56, 8, 2, 1), (57, 8, 1, 1), (121, 8, 3, 1),
                                           (40, 8, 1, 2), (57, 8, 1, 4), (121, 8, 3, 4)])
def test_general_steps_equal_kept_transitions(gpu_engine, N, P, form, team):
    """Diffuse networks of one to three chunks, solo and in teams."""
    print(f"[gpu] general steps: S={N + P} form {form} team {team}", flush=True)
    net, lay, es = _layout(N, P, **DIFFUSE)
    t = engine.make_trajs(4, lay.id, es, np.arange(4, dtype=np.uint64), 6000, net["occupation"],
                          prehops=1500)
    for rec in (False, True):
        opts = dict(table_form=form, team=team, record=rec)
        _same(_run(t, **opts), _run(t, chunk=1024, **opts), (N, form, team, rec))
    lay.close()


@pytest.mark.parametrize("K", [1024, 1 << 20])
@pytest.mark.parametrize("kind", [LOCAL, DIFFUSE])
def test_states_taken_over_change_no_bits(gpu_engine, K, kind):
    """More states than a wave keeps, 64 or two, with and without recomputes."""
    net, lay, es = _layout(30, 8, **kind)
    t = engine.make_trajs(8, lay.id, es, np.arange(8, dtype=np.uint64), 20_000, net["occupation"])
    print(f"[gpu] states taken over: recompute every {K} hops, {kind}", flush=True)
    for rec in (False, True):
        opts = dict(record=rec, recompute_interval=K)
        ref = _run(t, state_store=-1, **opts)
        for store in (0, 1, 4):
            _same(ref, _run(t, state_store=store, **opts), (K, store, rec))
    lay.close()
