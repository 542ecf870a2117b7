"""Runs of one batch that group its trajectories differently (waves per workgroup, a wave
per site chunk or a grid limit instead), one after the other without a wait between them
and around a captured graph."""
import numpy as np
import pytest

from kmc_dn_amd import _lib, engine
from tests.test_gpu_kept_states import LOCAL, _layout, _same

pytestmark = pytest.mark.gpu


def _results(b):
    b.sync()
    r = b.results()
    assert (r.status == 0).all()
    return [np.array(x) for x in (r.time.view(np.uint64), r.eo, r.occ_bits)]


def test_a_graph_survives_other_groups(gpu_engine):
    """64 groups of eight; then 512 of one, for which the buffer grows and moves."""
    net, lay, es = _layout(30, 8, **LOCAL)
    b = engine.Batch(engine.make_trajs(512, lay.id, es, np.arange(512, dtype=np.uint64), 2000, net["occupation"]))
    print("[gpu] graph around other groups", flush=True)
    b.run(precision=_lib.FP32_BATCHED, waves_per_group=8)
    ref = _results(b)
    for _ in range(3):
        b.run(precision=_lib.FP32_BATCHED, waves_per_group=8, use_graph=True)
        _same(ref, _results(b), "graph")
        b.run(precision=_lib.FP32_BATCHED, waves_per_group=1)
        _same(ref, _results(b), "groups of one")
    b.close()
    lay.close()


def test_groups_change_behind_a_run_in_flight(gpu_engine):
    net, lay, es = _layout(57, 8, **LOCAL)
    b = engine.Batch(engine.make_trajs(512, lay.id, es, np.arange(512, dtype=np.uint64), 20_000, net["occupation"]))
    print("[gpu] groups change behind a run in flight", flush=True)
    ref = None
    for opts in (dict(waves_per_group=4), dict(waves_per_group=1), dict(table_form=2, waves_per_group=8),
                 dict(waves_per_group=4, grid_limit=64)):
        b.run(precision=_lib.FP32_BATCHED, waves_per_group=2)
        b.run(precision=_lib.FP32_BATCHED, **opts)
        b.run(precision=_lib.FP32_BATCHED, waves_per_group=2)
        out = _results(b)
        if ref is not None:
            _same(ref, out, opts)
        ref = out
    b.close()
    lay.close()
