"""quot_plain (gw_math.h) on the device against a / b, bit for bit: operands over
the whole range it asks for, 2^+-310, its edges among them, and a zero numerator."""
import ctypes as C
import importlib.util
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gw-model_amd")


@pytest.fixture(scope="module")
def quot():
    spec = importlib.util.spec_from_file_location("gw_build_ext", os.path.join(PKG, "build_ext.py"))
    be = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(be)
    path = os.path.join(be.LIBDIR, "libgwprobe.so")
    if not os.path.exists(path):
        be.build_probe()
    fn = C.CDLL(path).gw_probe_quot_plain
    fn.argtypes = [C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64]

    def run(a, b):
        a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
        q = np.empty_like(a)
        assert fn(a.ctypes.data, b.ctypes.data, q.ctypes.data, a.size) == 0
        return q

    return run


def _mantissas(rng, n):
    """[1, 2): random, with few bits set, and at both ends."""
    m = rng.integers(0, 1 << 52, n, dtype=np.uint64)
    kind = rng.integers(0, 6, n)
    m = np.where(kind == 1, np.uint64(0), m)
    m = np.where(kind == 2, np.uint64((1 << 52) - 1), m)
    m = np.where(kind == 3, m & np.uint64(7), m)
    m = np.where(kind == 4, ~(m & np.uint64(7)) & np.uint64((1 << 52) - 1), m)
    return (m | np.uint64(1023 << 52)).view(np.float64)


def _same(quot, a, b):
    got, want = quot(a, b), a / b
    bad = np.flatnonzero(got.view(np.uint64) != want.view(np.uint64))
    assert bad.size == 0, [(a[i].hex(), b[i].hex(), got[i].hex(), want[i].hex()) for i in bad[:4]]


@pytest.mark.parametrize("lo,hi", [(-310, 309), (-1, 1), (300, 309), (-310, -300)])
def test_quotients_have_the_bits_of_a_division(quot, lo, hi):
    rng = np.random.default_rng(hi - lo)
    n = 4_000_000
    a = np.ldexp(_mantissas(rng, n), rng.integers(lo, hi + 1, n)) * rng.choice((-1.0, 1.0), n)
    b = np.ldexp(_mantissas(rng, n), rng.integers(lo, hi + 1, n)) * rng.choice((-1.0, 1.0), n)
    _same(quot, a, b)


@pytest.mark.parametrize("ea", [-310, 309])
@pytest.mark.parametrize("eb", [-310, 309])
def test_quotients_at_the_corners_of_the_range(quot, ea, eb):
    rng = np.random.default_rng(ea * 1000 + eb + 400_000)
    _same(quot, np.ldexp(_mantissas(rng, 1_000_000), ea), np.ldexp(_mantissas(rng, 1_000_000), eb))


def test_quotients_of_the_logarithm(quot):
    """f / (2 + f), f = m - 1 for m in [sqrt(2)/2, sqrt(2)], zero among them."""
    rng = np.random.default_rng(3)
    f = np.concatenate([rng.uniform(0.5 ** 0.5, 2 ** 0.5, 4_000_000) - 1.0, [0.0],
                        np.ldexp(rng.integers(1, 1 << 20, 100_000).astype(float), -53) * rng.choice((-1.0, 1.0), 100_000)])
    _same(quot, f, 2.0 + f)
