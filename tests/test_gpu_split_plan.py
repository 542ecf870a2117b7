"""Bucket entries whose trajectories may get a wave per site chunk: a run that takes
their solo kernel after all (a grid limit) has full workgroups."""
import pytest

from kmc_dn_amd import _lib, engine
from tests.test_gpu_kept_states import LOCAL, _layout, _same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,P", [(57, 8), (100, 9)])
def test_grid_limit_runs_full_workgroups(gpu_engine, N, P):
    """64 trajectories of two chunks on 8 workgroups of four waves, by a plan's entry and
    without a plan: the same kernel on the same groups, the same bits and the same time
    (with one wave of four at work it takes more than twice as long)."""
    import numpy as np
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
