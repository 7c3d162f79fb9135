"""The evaluations that hold in a range of operands against the plain ones, bit for bit: division by a
shared reciprocal, the limiter's minimum from its smallest slope, and HLLL's norm from an exact sum of
squares (pyhype_amd/csrc/phx_numerics.hpp; tests/native/inrange_numerics.hip holds both).  On the host
every element takes its own path; on the GPU a wave takes one path, so the classes lie in runs of 64."""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest

LIB = Path(__file__).resolve().parent / "native" / "libinrange_numerics.so"
DIV, INV, LIMIT, NORM = range(4)


def _signed(rng, n, lo, hi):
    return rng.choice([-1.0, 1.0], n) * rng.uniform(1.0, 2.0, n) * 2.0 ** rng.uniform(lo, hi, n)


def _next(x, k):
    return (np.asarray(x).view(np.int64) + k).view(np.float64)


def divisions(rng):
    n, d = [_signed(rng, 64 * 400, -600, 600)], [_signed(rng, 64 * 400, -100, 100)]
    n.append(_signed(rng, 64 * 400, -1, 1)); d.append(_signed(rng, 64 * 400, -1, 1))
    k = rng.integers(1, 1 << 20, 64 * 100).astype(float)                    # exact and nearly exact quotients
    n.append(k * rng.integers(1, 1 << 20, k.size)); d.append(k)
    n.append(_next(n[-1], rng.integers(-2, 3, k.size))); d.append(k)
    n.append(np.repeat([0.0, -0.0], 64)); d.append(np.tile(np.abs(_signed(rng, 64, -100, 100)), 2))
    return np.stack([np.concatenate(n), np.concatenate(d)], axis=1)


def limiters(rng):
    out = []

    def add(u, dmax, dmin, h):
        out.append(np.column_stack(np.broadcast_arrays(u, dmax, dmin, *h)).reshape(-1, 7))

    n = 64 * 200
    u = _signed(rng, n, -2, 2)
    span = lambda lo, hi: [_signed(rng, n, lo, hi) for _ in range(4)]  # noqa: E731
    up, dn = np.abs(_signed(rng, n, -8, 0)), -np.abs(_signed(rng, n, -8, 0))
    add(u, up, dn, span(-12, 1))                                             # slopes on both sides of 2
    add(u, up, dn, span(-60, -48))                                           # increments of a few last places, and 0
    add(u, up * 0.0, dn, span(-12, 1))                                       # a local maximum
    add(u, up * 0.0, dn * 0.0, span(-12, 1))
    h = span(-6, -1)
    add(u, up, dn, [h[0], h[0], h[2], h[2]])                                 # equal slopes
    for k in (-3, -1, 1, 3, 4096, 1 << 16):                                  # slopes a few last places apart
        add(u * 0 + 1.0, up, dn, [h[0], _next(h[0], k), -h[0], _next(-h[0], -k)])
        add(u * 0 + 2.0 ** -30, up, -up, [h[0], -_next(h[0], k), h[0], -h[0]])
    s = up / (2.0 * (1.0 + rng.integers(-3, 4, n) * 2.0 ** -52))             # slopes next to 2
    add(u * 0 + 2.0 ** -40, up, dn, [s, -2.0 * s, s * 0.5, _next(s, 1)])
    add(u * 0 + 2.0 ** -40, up, -up, [s * 0.3, -s * 0.2, s * 0.1, -s * 0.4])  # all slopes above 2
    add(u * 0.0, up, dn, span(-12, 1))                                       # the value is zero
    add(u * 0.0, up, dn, span(-1060, 1))                                     # ... and slopes overflow
    add(u * 0.0, up * 0.0, dn * 0.0, [u * 0.0] * 4)
    add(u * 2.0 ** -400, up * 2.0 ** -400, dn * 2.0 ** -400, span(-420, -399))
    add(u * 2.0 ** 300, up * 2.0 ** 300, dn * 2.0 ** 300, span(280, 301))
    add(u, up * 2.0 ** 120, dn, span(-12, 1))
    bad = rng.choice([np.nan, np.inf, -np.inf, 0.0, 1.0], (64 * 20, 7))
    out.append(bad)
    mixed = np.concatenate(out)                                              # every class within one wave
    out.append(mixed[rng.permutation(mixed.shape[0])])
    return np.concatenate(out)


def norms(rng):
    n = 64 * 500
    out = [np.stack([_signed(rng, n, -3, 3) for _ in range(4)], axis=1),
           np.stack([_signed(rng, n, -40, 3) for _ in range(4)], axis=1),
           np.stack([_signed(rng, n, -700, 700) for _ in range(4)], axis=1),
           rng.integers(-64, 65, (n, 4)).astype(float),                      # many exact roots and powers of two
           np.zeros((64, 4)), np.ldexp(1.0, rng.integers(-500, 400, (n, 4)))]
    a = np.stack([_signed(rng, n, -1, 1) for _ in range(4)], axis=1)
    a[:, 1:] *= 2.0 ** -27                                                   # roots next to a midpoint of two doubles
    out.append(a)
    out.append(np.where(rng.random((n, 4)) < 0.4, 0.0, out[0]))
    return np.concatenate(out)


CASES = {"division": (DIV, divisions), "reciprocal": (INV, lambda r: _signed(r, 64 * 800, -100, 100)[:, None]),
         "limiter": (LIMIT, limiters), "norm": (NORM, norms)}


def _same_bits(a, b):
    both_nan = np.isnan(a) & np.isnan(b)
    return both_nan | (a.view(np.int64) == b.view(np.int64))


def _check(x, fast, plain):
    bad = np.nonzero(~_same_bits(fast, plain))[0]
    assert bad.size == 0, f"{bad.size} of {fast.size} differ, e.g. {x[bad[0]]}: {fast[bad[0]]!r} {plain[bad[0]]!r}"


def _load():
    if not LIB.exists():
        pytest.fail(f"missing {LIB.name}: run __graft_entry__.build()")
    return C.CDLL(str(LIB))


@pytest.mark.parametrize("name", list(CASES))
def test_in_range_evaluation_on_the_host(name):
    what, make = CASES[name]
    x = np.ascontiguousarray(make(np.random.default_rng(20)))
    fast, plain = np.empty(x.shape[0]), np.empty(x.shape[0])
    p = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    with np.errstate(all="ignore"):
        _load().inr_host(what, p(x), p(fast), p(plain), x.shape[0])
    _check(x, fast, plain)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_in_range_evaluation_on_the_device(name):
    import torch

    what, make = CASES[name]
    x = np.ascontiguousarray(make(np.random.default_rng(21)))
    d = torch.from_numpy(x).cuda()
    fast, plain = (torch.empty(x.shape[0], dtype=torch.float64, device="cuda") for _ in range(2))
    fn = _load().inr_device
    fn.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    assert fn(what, d.data_ptr(), fast.data_ptr(), plain.data_ptr(), x.shape[0],
              torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    _check(x, fast.cpu().numpy(), plain.cpu().numpy())
