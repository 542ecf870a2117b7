"""Launches whose trajectories may get a wave per site chunk: they do while all fit
beside each other, and a bucket entry's run that takes the solo kernel after all (a
grid limit) has full workgroups."""
import numpy as np
import pytest

from kmc_dn_amd import _lib, engine
from tests.test_gpu_kept_states import DIFFUSE, LOCAL, _layout, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P", [(57, 8), (100, 9)])
def test_grid_limit_runs_full_workgroups(gpu_engine, N, P):
    """64 trajectories of two chunks on 8 workgroups of four waves, by a plan's entry and
    without a plan: the same kernel on the same groups, the same bits and the same time
    (with one wave of four at work it takes more than twice as long)."""
    net, lay, es = _layout(N, P, **LOCAL)
    t = engine.make_trajs(64, lay.id, es, np.arange(64, dtype=np.uint64), 20_000, net["occupation"])
    print(f"[gpu] plan entry under a grid limit: S={N + P}", flush=True)
    out, ms = [], []
    for plan in ([], [(192, 2, 4, 1, 0)]):
        b = engine.Batch(t)
        b.set_buckets(plan)
        took = []
        for _ in range(4):
            b.run(precision=_lib.FP32_BATCHED, table_form=2, waves_per_group=4, grid_limit=8)
            took.append(b.sync())
        r = b.results()
        out.append([r.time, r.eo, r.occ_bits])
        ms.append(min(took[1:]))
        b.close()
    lay.close()
    _same(out[0], out[1], (N, P))
    assert ms[1] < 1.5 * ms[0], ms


@pytest.mark.parametrize("record", [False, True])
def test_a_wave_per_chunk_only_while_all_fit(gpu_engine, record):
    """560 trajectories of three chunks: three of their workgroups do not fit a CU, so
    one would wait and double the launch; it is no longer than one wave each (a grid
    limit that limits nothing)."""
    net, lay, es = _layout(140, 8, **DIFFUSE)
    t = engine.make_trajs(560, lay.id, es, np.arange(560, dtype=np.uint64), 2000, net["occupation"])
    print(f"[gpu] 560 trajectories of S = 148, record {record}", flush=True)
    ms = []
    b = engine.Batch(t)
    for grid in (1 << 20, 0):
        took = []
        for _ in range(4):
            b.run(precision=_lib.FP32_BATCHED, table_form=3, record=record, grid_limit=grid)
            took.append(b.sync())
        ms.append(min(took[1:]))
    b.close()
    lay.close()
    assert ms[1] < 1.1 * ms[0], ms
