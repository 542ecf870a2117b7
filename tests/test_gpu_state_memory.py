"""Device memory of the kept states: launches that keep none reserve none, and a refused
allocation leaves no error for a later call."""
import numpy as np
import pytest
import torch

from kmc_dn_amd import _lib, engine
from tests.test_gpu_general_steps import _general
from tests.test_gpu_kept_states import LOCAL, _layout

pytestmark = pytest.mark.gpu


def _taken(run):
    """Device bytes that run() takes for good, from an engine that holds none."""
    engine.reset()
    net, lay, es = _layout(92, 8, **LOCAL)
    b = engine.Batch(engine.make_trajs(256, lay.id, es, np.arange(256, dtype=np.uint64), 200, net["occupation"]))
    before = torch.cuda.mem_get_info()[0]
    run(b)
    b.sync()
    taken = before - torch.cuda.mem_get_info()[0]
    assert (b.results().status == 0).all()
    b.close()
    lay.close()
    return taken


def test_runs_that_keep_no_states_reserve_none(gpu_engine):
    print("[gpu] memory of kept states", flush=True)
    opts = dict(precision=_lib.FP32_BATCHED, table_form=2)
    for _ in range(2):   # (the first run of each kernel loads its code)
        kept = _taken(lambda b: b.run(**opts))
        team = _taken(lambda b: b.run(team=4, **opts))
        general = _taken(lambda b: _general(b, False, False, 2))
    # 256 workgroups of two waves, two chunks of 32 KiB each
    assert kept >= 32 << 20
    assert team < 8 << 20 and general < 8 << 20, (kept, team, general)
    engine.reset()


def test_a_refused_allocation_leaves_no_error(gpu_engine):
    """Traffic matrices of 2^21 trajectories of S = 192 (618 GB) are refused; the mean-field
    run after it, which asks the runtime for launch errors, is not."""
    net, lay, es = _layout(176, 16, **LOCAL)
    b = engine.Batch(engine.make_trajs(1 << 21, lay.id, es, np.arange(1 << 21, dtype=np.uint64), 1, net["occupation"]))
    print("[gpu] a refused allocation", flush=True)
    with pytest.raises(_lib.KmcError) as e:
        b.run(precision=_lib.FP32_BATCHED, table_form=3, traffic=True)
    assert e.value.code == _lib.ERR_NOMEM
    r = engine.meanfield_simulate([lay], [int(es)], 2, net["occupation"][None].astype(float))
    assert (r.time > 0).all()
    b.close()
    lay.close()
