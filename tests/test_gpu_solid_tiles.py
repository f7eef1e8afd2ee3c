"""Solid flux passes at the edges of their tiles: segments of 64 or 32 lanes
along x, tiles of 16 columns by 15 faces along y and z (14 cells where stage 1
updates them in the same launch), ragged rows, and reflective ends.  The FP64 state must equal the oracle's bit for bit."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plate(n, bc_lo=(0, 0, 0), bc_hi=(0, 0, 0), box=16):
    """The plate impact cut down to n cells of the same size."""
    from tenjin_amd import configs

    dim = len(n)
    m = max(n)
    pb = configs.plate_impact(dim=dim, n=m, box=box, length=25.6e-3 * m / 256)
    nx, ny, nz = (tuple(n) + (1,))[:3]
    lo = [(m - q) // 2 for q in (nx, ny)] + [0]
    prims = pb.prims[:, lo[2]:lo[2] + nz, lo[1]:lo[1] + ny, lo[0]:lo[0] + nx]
    return dataclasses.replace(pb, n=(nx, ny, nz), L=tuple(1e-4 * q for q in (nx, ny, nz)), bc_lo=bc_lo, bc_hi=bc_hi,
                               prims=np.ascontiguousarray(prims))


CASES = [
    ((14, 15), 0), ((15, 14), 1), ((16, 16), 0), ((17, 29), 1), ((30, 30), 0), ((31, 31), 1), ((62, 13), 0),
    ((63, 32), 1), ((64, 44), 0), ((95, 3), 0), ((3, 46), 1), ((16, 14, 15), 0), ((33, 17, 14), 1), ((5, 31, 16), 0)]


@pytest.mark.parametrize("n,bc", CASES)
def test_solid_tiles_match_oracle(n, bc):
    from oracle.oracle import Oracle
    from tenjin_amd import GpuLevel

    pb = _plate(n, bc_lo=(bc, 0, bc), bc_hi=(0, bc, bc))
    print(f"\n[case] solid tiles {n} bc {bc}", flush=True)
    # f: the y pass and the update of stage 1 as two launches
    o, g, f = Oracle(pb), GpuLevel(pb), GpuLevel(pb)
    f.set_tuning(fuse=0)
    for q in (g, f):
        q.init_from_prims(pb.prims, pb.shift_pressure)
    for step in range(4):
        dt = o.driver_dt(step, 0.0)
        assert g.compute_dt() * (0.2 if step < 5 else 1.0) == dt
        o.step(dt)
        ref = o.get()
        for q in (g, f):
            q.set_dt(dt, reset_clock=1)
            q.step()
            got = q.get_state()
            for c in pb.layout.state_comps():
                assert np.array_equal(ref[c], got[c]), (step, pb.layout.names[c])
    assert g.status() == f.status() == 0


# of the largest value of a component's kind: an FP32 flux is off by some 1e-6 of
# its terms (24-bit operands, a few dozen roundings), of which a step adds a CFL
# number's part; four steps stay below 1e-5, and a misplaced face is of order 1
MIXED_TOL = 1e-4


@pytest.mark.parametrize("n,bc", CASES)
def test_solid_tiles_mixed(n, bc):
    """The FP32 instantiations: both stage forms give the same bits in every
    component, and all stay by the FP64 state but the phase densities, quotients
    by volume fractions of 1e-6."""
    from tenjin_amd import TJ_PREC_MIXED, GpuLevel

    pb = _plate(n, bc_lo=(bc, 0, bc), bc_hi=(0, bc, bc))
    print(f"\n[case] solid tiles, mixed, {n} bc {bc}", flush=True)
    d, g, f = GpuLevel(pb), GpuLevel(pb), GpuLevel(pb)
    f.set_tuning(fuse=0)
    for q in (d, g, f):
        q.init_from_prims(pb.prims, pb.shift_pressure)
    kinds = {}
    for c in pb.layout.state_comps():
        kinds.setdefault(pb.layout.names[c].rstrip("0123456789_"), []).append(c)
    for step in range(4):
        dt = d.compute_dt() * 0.2
        d.set_dt(dt, reset_clock=1)
        d.step()
        for q in (g, f):
            q.set_dt(dt, reset_clock=1)
            q.step(TJ_PREC_MIXED)
        ref, got, planes = d.get_state(), g.get_state(), f.get_state()
        for kind, comps in kinds.items():
            scale = max(np.abs(ref[comps]).max(), 1.0 if kind == "epsilon" else 0.0)
            if kind == "alphaRhoEpsilon":
                scale = np.abs(ref[kinds["alphaRho"]]).max()
            for c in comps:
                assert np.array_equal(got[c], planes[c]), (step, pb.layout.names[c])
                err = np.abs(got[c] - ref[c]).max()
                assert kind == "rho_k" or err <= MIXED_TOL * scale, (step, pb.layout.names[c], err, scale)
    assert g.status() == f.status() == 0
