"""Division and square root of the kernels (csrc/physics.hpp: recip, quot, sqrt_) against IEEE's,
at the ends of the ranges in which they promise the same bits, a little beyond, and for zeros,
infinities and NaN.  Beyond: a remainder that falls off the subnormal grid leaves a quotient
within half a unit of its last place besides the rounding, so one step of it; a square root's
remainder is below that grid and its estimate good to half a unit, so likewise one step."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cxx", "libidfx_arith.so")
N = 3000


def _call(op, a, b=None):
    import torch
    assert torch.cuda.is_available()  # its HIP runtime first: the library uses the one loaded
    b = a if b is None else b
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b, dtype=a.dtype)
    assert a.dtype == (np.float32 if op == 1 else np.float64) and a.shape == b.shape
    out = np.empty_like(a)
    p = ctypes.c_void_p
    assert ctypes.CDLL(LIB).arith(op, a.ctypes.data_as(p), b.ctypes.data_as(p), out.ctypes.data_as(p),
                                  a.size) == 0
    return out


def _mantissas(rng, t):
    """In [1, 2): random ones, and those next to both ends."""
    eps = np.finfo(t).eps
    m = 1.0 + rng.integers(0, int(1 / eps), N) * eps
    m[:4] = 1.0, 1.0 + eps, 2.0 - eps, 2.0 - 2 * eps
    return (m * rng.choice([-1.0, 1.0], N)).astype(t)


def _pairs(t, ea, eb, lo, hi):
    rng = np.random.default_rng(7)
    A, B = [], []
    for x in ea:
        for y in eb:
            if lo <= x - y <= hi:
                A.append(np.ldexp(_mantissas(rng, t), x))
                B.append(np.ldexp(rng.permutation(_mantissas(rng, t)), y))
    return np.concatenate(A).astype(t), np.concatenate(B).astype(t)


def _same(got, want):
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan)
    bits = np.int32 if want.dtype == np.float32 else np.int64
    assert np.array_equal(got.view(bits)[~nan], want.view(bits)[~nan])


RANGES = {0: (np.float64, [-969, -968, -700, -1, 0, 1, 700, 1022], [-1022, -1021, -500, -1, 0, 1, 500, 1021], 1021),
          1: (np.float32, [-102, -101, -60, -1, 0, 1, 60, 126], [-126, -125, -60, -1, 0, 1, 60, 125], 125)}


@pytest.mark.parametrize("op", [0, 1])
def test_quotients_to_the_last_bit(op):
    t, ea, eb, top = RANGES[op]
    a, b = _pairs(t, ea, eb, 1 - top, top - 1)
    _same(_call(op, a, b), a / b)


@pytest.mark.parametrize("op", [0, 1])
def test_quotients_of_small_numerators(op):
    t, ea, eb, top = RANGES[op]
    low = -1022 if op == 0 else -126
    a, b = _pairs(t, [low, low + 1, low + 20, ea[0] - 1], [-60, -1, 0], 1 - top, top - 1)
    want = a / b
    assert (np.abs(_call(op, a, b) - want) <= np.spacing(np.abs(want))).all()


@pytest.mark.parametrize("op", [0, 1])
def test_quotients_of_special_operands(op):
    t, _, _, top = RANGES[op]
    tiny, big = np.finfo(t).tiny, np.ldexp(t(1.25), top)
    v = np.array([0.0, -0.0, np.inf, -np.inf, np.nan, 1.0, -1.0, 3.0, -3.0, tiny, -tiny, big, -big], dtype=t)
    a, b = (x.ravel().astype(t) for x in np.meshgrid(v, v))
    with np.errstate(all="ignore"):
        want = a / b
        wide = np.abs(a.astype(np.longdouble) / b.astype(np.longdouble))
        # without the quotients that overflow or underflow, and the numerators near the end of the
        # range (a remainder of theirs is not exact)
        end = np.isfinite(wide) & (wide != 0) & ((wide > np.finfo(t).max) | (wide < tiny) | (np.abs(a) <= tiny))
    keep = ~end
    assert keep.sum() > 100
    _same(_call(op, a[keep], b[keep]), want[keep])


def test_square_roots():
    rng = np.random.default_rng(8)
    x = np.concatenate([np.ldexp(np.abs(_mantissas(rng, np.float64)), e)
                        for e in (-767, -766, -400, -399, -1, 0, 1, 2, 500, 501, 1022, 1023)] +
                       [np.array([0.0, -0.0, np.inf, np.nan, -1.0, -np.inf])])
    with np.errstate(all="ignore"):
        _same(_call(2, x), np.sqrt(x))
    y = np.concatenate([np.ldexp(np.abs(_mantissas(rng, np.float64)), e) for e in (-1074, -1073, -1050, -1022, -900, -768)])
    y = y[y > 0]
    want = np.sqrt(y)
    assert (np.abs(_call(2, y) - want) <= np.spacing(want)).all()
