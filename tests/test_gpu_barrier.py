"""tj_set_dt and tj_begin_run return after the work queued before them."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["set_dt", "begin_run"])
def test_call_waits_for_earlier_work(call):
    import torch

    from tenjin_amd import GpuLevel, configs

    pb = configs.shock_inclusion_2d(nx=1024, ny=512)
    print(f"\n[case] {call} after 40 queued steps", flush=True)
    g = GpuLevel(pb)
    g.init_from_prims(pb.prims)
    g.begin_run()
    g.advance(2)
    g.sync()
    stream = torch.cuda.ExternalStream(g.lib.tj_stream(g.ctx))
    g.advance(40)
    done = stream.record_event()
    if call == "set_dt":
        g.set_dt(1e-9)
    else:
        g.begin_run()
    assert done.query()
    assert g.status() == 0
