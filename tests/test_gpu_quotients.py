"""The FP64 quotients that share a divisor's reciprocal against a / b over the
operands that they are used for, bit for bit; and solid levels whose
transverse velocities, shear and plastic strains vanish ahead of a wave (down to
subnormal numbers) against the oracle, bit for bit."""
from __future__ import annotations

import ctypes
import dataclasses
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "host", "libquotients.so")


def _ordinary(rng, n, lo, hi):
    return rng.choice([-1.0, 1.0], n) * np.ldexp(rng.uniform(1.0, 2.0, n), rng.integers(lo, hi, n))


def _hard(rng, n):
    """Divisors next to a power of two and few-bit dividends: quotients close to
    the middle of two numbers."""
    b = np.ldexp(2.0 - rng.integers(1, 64, n) * 2.0 ** -52, rng.integers(-40, 40, n))
    a = np.ldexp(1.0 + rng.integers(0, 1 << 10, n) * 2.0 ** -rng.choice([10, 52], n), rng.integers(-40, 40, n))
    return a, b


def _run(a, b):
    """(qdiv, qdiv0) of the pairs."""
    import torch

    L = ctypes.CDLL(LIB)
    vp = ctypes.c_void_p
    L.quotients.argtypes = [vp, vp, vp, ctypes.c_int]
    n = len(a)
    ta, tb = torch.from_numpy(a).cuda(), torch.from_numpy(b).cuda()
    out = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert L.quotients(ta.data_ptr(), tb.data_ptr(), out.data_ptr(), n) == 0
    return out.cpu().numpy().reshape(2, n)


def _same(got, a, b):
    with np.errstate(all="ignore"):
        want = a / b
    bad = ~((got.view(np.int64) == want.view(np.int64)) | (np.isnan(got) & np.isnan(want)))
    assert not bad.any(), [tuple(v.hex() for v in t) for t in zip(*(q[bad][:3].tolist() for q in (a, b, got, want)))]


SPECIAL = [0.0, -0.0, 1.0, -3.0, np.inf, -np.inf, np.nan, 2.0 ** -900, 2.0 ** 499, 1e5]


@pytest.mark.parametrize("which,lo,n", [("qdiv", -900, 1 << 21), ("qdiv0", -1074, 1 << 21)])
def test_quotients_equal_division(which, lo, n):
    """Dividends from 2^lo to 2^500 (0, infinities and NaN among them) and
    divisors from 2^-500 to 2^500, spread over their exponents, next to 1, at
    the dividends' lower end, and hard to round."""
    rng = np.random.default_rng(5)
    h = _hard(rng, n)
    s = np.repeat(SPECIAL, 5)
    a = np.concatenate([_ordinary(rng, n, lo, 500), _ordinary(rng, n, -60, 60), _ordinary(rng, n, lo, lo + 60),
                        np.ldexp(h[0], lo // 2), h[0], s])
    b = np.concatenate([_ordinary(rng, n, -500, 500), _ordinary(rng, n, -60, 60), _ordinary(rng, n, -60, 60),
                        np.ldexp(h[1], lo // 4), h[1], np.tile([0.0, 1.0, 3.0, -np.inf, np.nan], len(SPECIAL))])
    print(f"\n[case] {which} on {len(a)} pairs", flush=True)
    _same(_run(a, b)[("qdiv", "qdiv0").index(which)], a, b)


@pytest.mark.parametrize("n,lo,hi,strain", [((30, 33), 290, 323, 1), ((30, 33), 306, 310, 0), ((62, 17), 300, 312, 0),
                                            ((17, 15, 14), 304, 316, 0)])
def test_vanishing_shear_matches_oracle(n, lo, hi, strain):
    """Transverse velocities, off-diagonal V and (strain) plastic strains of
    1e-lo to 1e-hi in every cell."""
    from oracle.oracle import Oracle
    from tenjin_amd import GpuLevel
    from tenjin_amd.configs import EPSILON, V_TENSOR, VELOCITY
    from test_gpu_solid_tiles import _plate

    pb = _plate(n)
    L, U, shape = pb.layout, pb.prims.copy(), pb.prims.shape[1:]
    rng = np.random.default_rng(lo)

    def tiny():
        return rng.choice([-1.0, 1.0], shape) * 10.0 ** -rng.uniform(lo, hi, shape)

    print(f"\n[case] vanishing shear {n} 1e-{lo} to 1e-{hi} strain {strain}", flush=True)
    for q in range(1, 3):
        U[L.comp(VELOCITY, 0, q)] = tiny()
    for q in range(9):
        if q % 4:
            U[L.comp(V_TENSOR, 0, q // 3, q % 3)] = tiny()
    for m in range(2):
        if strain:
            U[L.comp(EPSILON, m)] = np.abs(tiny())
    pb = dataclasses.replace(pb, prims=U)
    o, g = Oracle(pb), GpuLevel(pb)
    g.init_from_prims(pb.prims, pb.shift_pressure)
    for step in range(4):
        dt = o.driver_dt(step, 0.0)
        o.step(dt)
        g.set_dt(dt, reset_clock=1)
        g.step()
        ref, got = o.get(), g.get_state()
        for c in L.state_comps():
            assert np.array_equal(ref[c], got[c]), (step, L.names[c], np.abs(ref[c] - got[c]).max())
    assert g.status() == o.status()


@pytest.mark.parametrize("n,least", [(33, 1e-310), (33, 4e-320), (30, 1e-200)])
def test_vanishing_volume_fraction_matches_oracle(n, least):
    """A material whose volume fraction is next to nothing, down to subnormal
    numbers, where the other one fills the cell."""
    from oracle.oracle import Oracle
    from tenjin_amd import GpuLevel
    from tenjin_amd.configs import ALPHA
    from test_gpu_solid_tiles import _plate

    pb = _plate((n, n))
    L, U = pb.layout, pb.prims.copy()
    U[L.comp(ALPHA, 0)][U[L.comp(ALPHA, 0)] < 1e-3] = least
    U[L.comp(ALPHA, 1)][U[L.comp(ALPHA, 1)] < 1e-3] = least
    print(f"\n[case] volume fractions of {least} on {n} x {n}", flush=True)
    pb = dataclasses.replace(pb, prims=U)
    o, g = Oracle(pb), GpuLevel(pb)
    g.init_from_prims(pb.prims, pb.shift_pressure)
    for step in range(2):
        dt = o.driver_dt(step, 0.0)
        o.step(dt)
        g.set_dt(dt, reset_clock=1)
        g.step()
        ref, got = o.get(), g.get_state()
        assert not np.isnan(ref[: len(L.names)]).any()
        for c in L.state_comps():
            assert np.array_equal(ref[c], got[c]), (step, L.names[c], np.abs(ref[c] - got[c]).max())
