"""Spells of general steps: a trajectory that finds many new states leaves its kept
transitions within the recompute interval, whatever its energies follow from, and
stays with general steps for the intervals it has to."""
import ctypes as C

import numpy as np
import pytest

from kmc_dn_amd import _lib, engine
from tests.test_gpu_kept_states import DIFFUSE, _layout

pytestmark = pytest.mark.gpu


def _times(b, record, form, team):
    """Best of four kernel times: the ordinary run's and by general steps alone."""
    o = _lib.kmc_run_opts(_lib.FP32_BATCHED, 0, 0, int(record), 0, 0, 0, form, 0, team, 0, 0)
    kept, general = [], []
    for _ in range(4):
        b.run(precision=_lib.FP32_BATCHED, table_form=form, team=team, record=record)
        kept.append(b.sync())
        _lib.check(_lib.load().kmc_probe_fp32_general(b.id, C.byref(o)))
        general.append(b.sync())
    return min(kept), min(general)


@pytest.mark.parametrize("N,P,form,team,K", [(100, 9, 2, 1, 512), (62, 8, 2, 1, 1024), (50, 8, 2, 4, 32)])
@pytest.mark.parametrize("record", [False, True])
def test_new_states_on_most_hops(gpu_engine, N, P, form, team, K, record):
    """Nearly every hop new, four recompute intervals: an eighth of an interval with
    transitions costs at most a fifth of the whole (whole intervals of them cost a third)."""
    net, lay, es = _layout(N, P, **DIFFUSE)
    b = engine.Batch(engine.make_trajs(K, lay.id, es, np.arange(K, dtype=np.uint64), 4000, net["occupation"]))
    print(f"[gpu] spells of general steps: S={N + P} team {team} record {record}", flush=True)
    kept, general = _times(b, record, form, team)
    b.close()
    lay.close()
    assert kept < 1.2 * general, (kept, general)
