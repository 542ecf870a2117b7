"""Kept transitions, kept states and leaps give the general steps' trajectories.

The probe runs a batch by general steps alone: every hop selects its row and its
partner from the state's rates, and a state is evaluated unless it is the one before
the last hop.  The ordinary run of the same batch keeps transitions and states, takes
runs of hops back at once, changes between both ways by what it finds and, where a
launch leaves SIMDs idle, gives each trajectory a wave per site chunk.  Every result is
the same to the bit.
"""
import ctypes as C

import numpy as np
import pytest

from kmc_dn_amd import _lib, engine
from tests.test_gpu_kept_states import DIFFUSE, LOCAL, _layout, _same

pytestmark = pytest.mark.gpu

STRONG = dict(I_0=100.0, a=0.25, E_spread=100.0)   # many states, some returns


def _general(b, record, traffic, table_form, team=1):
    o = _lib.kmc_run_opts(_lib.FP32_BATCHED, 0, 0, int(record) | 2 * int(traffic), 0, 0, 0, table_form, 0, team, 0, 0)
    _lib.check(_lib.load().kmc_probe_fp32_general(b.id, C.byref(o)))
    b.recorded = bool(record)


def _results(b, record, S):
    b.sync()
    r = b.results()
    assert (r.status == 0).all()
    out = [r.time.view(np.uint64), r.eo, r.occ_bits, r.hops_done]
    return out + [r.occ_time.view(np.uint64)] + b.traffic(S) if record else out


@pytest.mark.parametrize("N,P,form", [(30, 8, 1), (54, 8, 2), (40, 8, 3), (56, 8, 1), (57, 8, 1), (92, 8, 2),
                                      (120, 8, 3), (121, 8, 2), (124, 8, 2), (140, 12, 3)])
@pytest.mark.parametrize("kind", [LOCAL, DIFFUSE, STRONG], ids=["local", "diffuse", "strong"])
def test_kept_paths_equal_general_steps(gpu_engine, N, P, form, kind):
    """S = 38 to 64 in one chunk, 65 to 128 in two, 129 to 152 in three; solo launches
    that leave SIMDs idle (a wave per chunk) and that do not; budgets over several
    recomputes that end within an interval and within a uniform block."""
    net, lay, es = _layout(N, P, **kind)
    for K, hops in ((6, 9001), (700, 1503)):
        b = engine.Batch(engine.make_trajs(K, lay.id, es, np.arange(K, dtype=np.uint64), hops, net["occupation"],
                                           prehops=100))
        for rec in (False, True):
            print(f"[gpu] general steps: S={N + P} form {form} K={K} record {rec}", flush=True)
            b.run(precision=_lib.FP32_BATCHED, table_form=form, record=rec, traffic=rec)
            kept = [np.array(x) for x in _results(b, rec, N + P)]
            _general(b, rec, rec, form)
            _same(kept, _results(b, rec, N + P), (N, form, K, rec))
        b.close()
    lay.close()


@pytest.mark.parametrize("N,P,form,team", [(40, 8, 1, 2), (56, 8, 2, 4), (50, 8, 3, 4), (57, 8, 2, 4)])
@pytest.mark.parametrize("kind", [LOCAL, DIFFUSE, STRONG], ids=["local", "diffuse", "strong"])
def test_teams_equal_general_steps(gpu_engine, N, P, form, team, kind):
    net, lay, es = _layout(N, P, **kind)
    b = engine.Batch(engine.make_trajs(5, lay.id, es, np.arange(5, dtype=np.uint64), 6001, net["occupation"],
                                       prehops=100))
    for rec in (False, True):
        print(f"[gpu] general steps: S={N + P} form {form} team {team} record {rec}", flush=True)
        b.run(precision=_lib.FP32_BATCHED, table_form=form, team=team, record=rec, traffic=rec)
        kept = [np.array(x) for x in _results(b, rec, N + P)]
        _general(b, rec, rec, form, team)
        _same(kept, _results(b, rec, N + P), (N, form, team, rec))
    b.close()
    lay.close()
