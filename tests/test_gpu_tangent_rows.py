"""Direction groups of the tangent-linear form side by side (grid rows): a last
group that is not full, and more groups than run at once, must give the traces
and derivative states of one group of six."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,ndir,chunk", [(24, 5, 2), (24, 1, 1), (40, 4, 3), (216, 6, 1)])
def test_group_rows_match_one_group(n, ndir, chunk):
    from tenjin_amd import configs, tangent

    pb = configs.plate_impact_differentiated(n=n, box=32)
    dirs = tangent.ALL_DIRECTIONS[:ndir]
    probe = (pb.layout.comp(configs.VELOCITY, 0, 0), n // 2 + 2, n // 2, 0)
    print(f"\n[case] tangent rows n {n} directions {ndir} chunk {chunk}", flush=True)
    runs = []
    for k in (chunk, 6):
        t = tangent.TangentRun(pb, dirs, chunk=k)
        trace, done = t.run(4, probe)
        d = ndir - 1  # in the last group of both
        runs.append((trace, done, t.state(), t.state_derivative(d), t.g.clock(), t.status()))
        t.close()
    a, b = runs
    assert a[1] == b[1] == 4 and a[4] == b[4] and a[5] == b[5] == 0
    for q in (0, 2, 3):
        assert np.array_equal(a[q], b[q])
    assert np.abs(a[0][:, 1:]).max() > 0.0
