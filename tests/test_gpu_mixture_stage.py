"""Two-dimensional levels with a mixture material on the stage kernels: at the
edges of their tiles (60 / 62 cells along x, 12 / 14 rows along y) against the
oracle, bit for bit; against the flux-plane passes; and tj_run_static of a
level whose scratch holds the flux planes but not the stage planes."""
from __future__ import annotations

import ctypes
import dataclasses

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tube(nx, ny, thinc, box=16):
    from tenjin_amd import configs

    pb = configs.reactive_tube(dim=2, n=max(nx, 2 * ny), box=box, thinc=thinc)
    prims = np.ascontiguousarray(pb.prims[:, :, :ny, :nx])
    return dataclasses.replace(pb, n=(nx, ny, 1), prims=prims)


CASES = [(12, 11, 1), (59, 12, 1), (60, 13, 1), (61, 25, 1), (62, 14, 0), (63, 15, 0), (17, 29, 0), (33, 24, 1)]


@pytest.mark.parametrize("nx,ny,thinc", CASES)
def test_mixture_stage_tiles_match_oracle(nx, ny, thinc):
    from oracle.oracle import Oracle
    from tenjin_amd import GpuLevel

    pb = _tube(nx, ny, thinc)
    print(f"\n[case] mixture stage tiles {nx} x {ny} thinc {thinc}", flush=True)
    o, g, f = Oracle(pb), GpuLevel(pb), GpuLevel(pb)
    f.set_tuning(fuse=0)
    for q in (g, f):
        q.init_from_prims(pb.prims)
    for step in range(4):
        dt = o.driver_dt(step, 0.0)
        o.step(dt)
        for q in (g, f):
            q.set_dt(dt, reset_clock=1)
            q.step()
        ref = o.get()
        for q in (g, f):
            got = q.get_state()
            for c in pb.layout.state_comps():
                assert np.array_equal(ref[c], got[c]), (step, pb.layout.names[c])
    assert g.status() == f.status() == o.status()


@pytest.mark.parametrize("nx,ny,thinc", CASES)
def test_mixture_stage_tiles_mixed(nx, ny, thinc):
    """The FP32 instantiations: the stage kernels and the flux-plane passes give
    the same bits in every component."""
    from tenjin_amd import TJ_PREC_MIXED, GpuLevel

    pb = _tube(nx, ny, thinc)
    print(f"\n[case] mixture stage tiles, mixed, {nx} x {ny} thinc {thinc}", flush=True)
    g, f = GpuLevel(pb), GpuLevel(pb)
    f.set_tuning(fuse=0)
    for q in (g, f):
        q.init_from_prims(pb.prims)
    for step in range(4):
        dt = g.compute_dt() * 0.2
        assert f.compute_dt() * 0.2 == dt
        for q in (g, f):
            q.set_dt(dt, reset_clock=1)
            q.step(TJ_PREC_MIXED)
        got, planes = g.get_state(), f.get_state()
        for c in pb.layout.state_comps():
            assert np.array_equal(got[c], planes[c]), (step, pb.layout.names[c])
    assert g.status() == f.status()


@pytest.mark.parametrize("seed,energy,negative", [(1, 0.0, 0), (2, 0.5, 0), (3, 4.0, 0), (4, 0.5, 1), (5, 4.0, 1)])
def test_bisection_signs_match_oracle(seed, energy, negative):
    """rootFind's known signs: cells whose mass fraction, density, pressure and
    (for energy > 0) total energy are drawn over decades, brackets without a
    sign change among them, and (negative) half the cells with a partial density
    below 0, against the oracle's plain bisection, bit for bit."""
    from oracle.oracle import Oracle
    from tenjin_amd import GpuLevel
    from tenjin_amd.configs import ALPHA, ALPHARHO, ALPHARHOLAMBDA, LAMBDA, P, RHO_K, TOTAL_E

    rng = np.random.default_rng(seed)
    pb = _tube(37, 29, 0)
    L, U, shape = pb.layout, pb.prims.copy(), pb.prims.shape[1:]
    al = 10.0 ** rng.uniform(-6.0, 0.0, shape)
    print(f"\n[case] bisection seed {seed} energy {energy}", flush=True)
    for m in range(2):
        U[L.comp(ALPHA, m)] = (al, 1.0 - al)[m]
        U[L.comp(RHO_K, m)] = 10.0 ** rng.uniform(0.0, 3.8, shape)
    U[L.comp(LAMBDA)] = rng.uniform(0.0, 1.0, shape)
    U[L.comp(P)] = 10.0 ** rng.uniform(4.0, 11.0, shape)
    pb = dataclasses.replace(pb, prims=U)
    o, g = Oracle(pb), GpuLevel(pb)
    g.init_from_prims(pb.prims)
    s = o.get()
    assert np.array_equal(s[L.comp(ALPHARHO)], g.get_state()[L.comp(ALPHARHO)])
    s[L.comp(TOTAL_E)] *= 10.0 ** (energy * rng.uniform(-1.0, 1.0, shape))
    if negative:
        flip = rng.choice([-1.0, 1.0], shape)
        for c in [L.comp(ALPHARHO, m) for m in range(2)] + [L.comp(ALPHARHOLAMBDA)]:
            s[c] *= flip
    o.set(s)
    g.set_state(s)
    o.c2p()
    g.c2p()
    ref, got = o.get(), g.get_state()
    for c in L.state_comps():
        assert np.array_equal(ref[c], got[c], equal_nan=True), L.names[c]
    assert g.status() == o.status()


def test_static_scratch_without_stage_planes():
    import torch

    from tenjin_amd import GpuLevel, LevelDesc, MFView, level_desc, load_library

    pb = _tube(832, 416, 0, box=64)  # flux planes 53 MiB, stage planes 24 MiB more, of 64 MiB
    print("\n[case] static run, flux planes only", flush=True)
    L = load_library()
    mfp = ctypes.POINTER(MFView)
    L.tj_run_static.argtypes = [ctypes.POINTER(LevelDesc), mfp, mfp, ctypes.c_double, ctypes.c_int, ctypes.c_int,
                                ctypes.c_int, ctypes.c_void_p, ctypes.POINTER(ctypes.c_double),
                                ctypes.POINTER(ctypes.c_int)]
    g = GpuLevel(pb)
    g.init_from_prims(pb.prims)
    S, T = g.S.clone(), torch.zeros_like(g.S)
    torch.cuda.synchronize()
    n, t = g.run(float("inf"), max_steps=2)
    vS, vT, d = g._view(S), g._view(T), level_desc(pb)
    tt, nn = ctypes.c_double(), ctypes.c_int()
    assert L.tj_run_static(ctypes.byref(d), ctypes.byref(vS), ctypes.byref(vT), float("inf"), 2, 0, 8, None,
                           ctypes.byref(tt), ctypes.byref(nn)) == 0
    torch.cuda.synchronize()
    assert (nn.value, tt.value) == (n, t)
    assert torch.equal(S, g.S)
