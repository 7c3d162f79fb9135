"""Functions with a short evaluation for operands in range, on both sides of each range: quotients of a shared
divisor, the inverse area, the primitive states of a face, the averages of both fluxes, Barth-Jespersen's
value, and Venkatakrishnan's on a block whose geometry is out of range (pyhype_amd/csrc/phx_numerics.hpp;
tests/native/guards_numerics.hip holds both evaluations).  Bit for bit, on the host element by element and
on the device by waves, with every class in waves of its own and all classes within one wave."""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest

from tests.test_inrange_numerics import _check, _signed, limiters

LIB = Path(__file__).resolve().parent / "native" / "libguards_numerics.so"
N = 64 * 40
ODD = [0.0, -0.0, np.inf, -np.inf, np.nan, 5e-324, 2.0 ** -1030, 2.0 ** -700, 2.0 ** 700, -1.0]


def _mixed(classes):
    """Every class in waves of its own, then all of them shuffled."""
    x = np.concatenate([np.asarray(c, dtype=float)[:c.shape[0] // 64 * 64] for c in classes])
    return np.ascontiguousarray(np.concatenate([x, x[np.random.default_rng(1).permutation(x.shape[0])]]))


def _out_of_range(rng, base, columns):
    """base as it is; with values at and beyond the ends of the range, and special ones, in some of the columns."""
    out = [base]
    for c in columns:
        for lo, hi in ((-1000, -101), (-101, -99), (99, 101), (101, 600), (599, 602), (602, 1000)):
            x = base.copy()
            x[:, c] = np.abs(_signed(rng, base.shape[0], lo, hi))
            out.append(x)
        x = base.copy()
        x[:, c] = rng.choice(ODD, base.shape[0])
        out.append(x)
    x = base.copy()
    hit = rng.random(x.shape) < 0.1
    x[:, columns] = np.where(hit, rng.choice(ODD, x.shape), x)[:, columns]
    out.append(x)
    return _mixed(out)


def divisions(rng):
    d = _signed(rng, 40 * N, -1000, 999)
    q = _signed(rng, 40 * N, -759, 758)
    with np.errstate(all="ignore"):
        n = d * q
    ok = (np.abs(n) >= 2.0 ** -900) & (np.abs(n) <= 2.0 ** 1020)
    return _mixed([np.column_stack([n, d])[ok]])


def slopes(rng):
    s = 2.0 * (1.0 + rng.integers(-64, 65, N) * 2.0 ** -52)
    return _mixed([np.abs(_signed(rng, 8 * N, -680, 494))[:, None], np.abs(_signed(rng, 8 * N, -4, 3))[:, None], s[:, None],
                   np.zeros((64, 1)), np.full((64, 1), np.nan)])


def quotients(rng):
    base = np.column_stack([_signed(rng, N, -2, 2) for _ in range(4)] + [np.abs(_signed(rng, N, -2, 2))])
    return _out_of_range(rng, base, [0, 2, 4])


def areas(rng):
    return _out_of_range(rng, np.abs(_signed(rng, N, -20, 20))[:, None], [0])


def _states(rng):
    return np.column_stack([f(_signed(rng, N, -3, 3)) for _ in range(2) for f in (np.abs, np.array, np.array, np.abs)])


def states(rng):
    x = _states(rng)
    x[:, 3::4] += x[:, 1::4] ** 2 / x[:, 0::4] + x[:, 2::4] ** 2 / x[:, 0::4]
    return _out_of_range(rng, x, list(range(8)))


def averages(rng):
    x = np.column_stack([_states(rng), np.full(N, 1.4), np.zeros(N)])
    odd = x.copy()
    odd[:, 8], odd[:, 9] = 1.0 + 2.0 ** -rng.integers(21, 40, N), 1.0     # a gas out of range, marked as such
    same = x[:64].copy()
    same[:, 4:8] = same[:, 0:4]
    return np.concatenate([_out_of_range(rng, x, list(range(8))), _mixed([odd, same, odd[:64]])])


def cells(rng):
    x = limiters(rng)
    # extrema of a stencil that holds the cell: dmin <= 0 <= dmax
    return np.ascontiguousarray(x[~(x[:, 1] < 0) & ~(x[:, 2] > 0)])


KINDS = {"division": (0, divisions), "venkat": (1, slopes), "quotients": (2, quotients), "area": (3, areas),
         "states": (4, states), "roe": (5, averages), "hlll": (6, averages), "barth-jespersen": (7, cells),
         "odd geometry": (8, cells)}


def _load():
    if not LIB.exists():
        pytest.fail(f"missing {LIB.name}: run __graft_entry__.build()")
    return C.CDLL(str(LIB))


def _inputs(name, seed):
    what, make = KINDS[name]
    with np.errstate(all="ignore"):
        x = make(np.random.default_rng(seed))
    lib = _load()
    assert x.flags.c_contiguous and x.shape[1] == lib.rg_in(what)
    return lib, what, x, (x.shape[0], lib.rg_out(what))


def _compare(x, fast, plain):
    for k in range(fast.shape[1]):
        _check(x, np.ascontiguousarray(fast[:, k]), np.ascontiguousarray(plain[:, k]))


@pytest.mark.parametrize("name", list(KINDS))
def test_guarded_evaluation_on_the_host(name):
    lib, what, x, shape = _inputs(name, 30)
    fast, plain = np.empty(shape), np.empty(shape)
    p = lambda a: a.ctypes.data_as(C.POINTER(C.c_double))  # noqa: E731
    lib.rg_host(what, p(x), p(fast), p(plain), shape[0])
    _compare(x, fast, plain)


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(KINDS))
def test_guarded_evaluation_on_the_device(name):
    import torch

    lib, what, x, shape = _inputs(name, 31)
    d = torch.from_numpy(x).cuda()
    fast, plain = (torch.empty(shape, dtype=torch.float64, device="cuda") for _ in range(2))
    fn = lib.rg_device
    fn.argtypes = [C.c_int, C.c_void_p, C.c_void_p, C.c_void_p, C.c_int, C.c_void_p]
    assert fn(what, d.data_ptr(), fast.data_ptr(), plain.data_ptr(), shape[0],
              torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    _compare(x, fast.cpu().numpy(), plain.cpu().numpy())
