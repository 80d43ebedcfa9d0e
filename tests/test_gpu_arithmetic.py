"""rcp_rn, div_rn and sqrt_rn of lum_amd/csrc/march.hpp on the GPU against IEEE
division and square root (numpy, on the host), bit for bit: every significand
for the reciprocal and (both parities of the exponent) the root, seeded pairs
and the ends of the declared range for the quotient."""
import ctypes as C
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.abspath(__file__)), "libmarch_device.so")
RCP, DIV, SQRT = 0, 1, 2


@pytest.fixture(scope="module")
def md():
    import torch  # noqa: F401  (its HIP runtime is the process's, loaded first)
    if not os.path.exists(LIB):
        import __graft_entry__
        __graft_entry__.build()
    return C.CDLL(LIB)


def apply(md, op, d, a=None):
    import torch
    td = torch.from_numpy(d).cuda()
    ta = None if a is None else torch.from_numpy(a).cuda()
    out = torch.empty_like(td)
    torch.cuda.synchronize()
    rc = md.md_apply(op, C.c_void_p(0 if ta is None else ta.data_ptr()), C.c_void_p(td.data_ptr()),
                     C.c_void_p(out.data_ptr()), d.size)
    assert rc == 0
    return out.cpu().numpy()


def same(x, y):
    return np.array_equal(x.view(np.uint32), y.view(np.uint32))


SIGNIFICANDS = np.arange(1 << 23, dtype=np.uint32)


def with_exponent(e, negative=False):
    """Every float with exponent 2^e."""
    return (SIGNIFICANDS | np.uint32((127 + e) << 23) | np.uint32(negative << 31)).view(np.float32)


@pytest.mark.parametrize("e,negative", [(0, False), (0, True), (-1, False), (-60, False), (59, True), (-9, False)])
def test_reciprocal_every_significand(md, e, negative):
    d = with_exponent(e, negative)
    assert same(apply(md, RCP, d), np.float32(1) / d)


@pytest.mark.parametrize("e", [0, 1, -1, -60, 59, 16])
def test_root_every_significand(md, e):
    x = with_exponent(e)
    assert same(apply(md, SQRT, x), np.sqrt(x))


@pytest.mark.parametrize("seed", range(8))
def test_quotient(md, seed):
    """Exponents over the whole range of the operands and of the quotient."""
    rng = np.random.default_rng(seed)
    n = 1 << 22

    def draw(span):
        bits = rng.integers(0, 1 << 23, n).astype(np.uint32) | ((127 + rng.integers(-span, span, n)).astype(np.uint32) << 23)
        return (bits | (rng.integers(0, 2, n).astype(np.uint32) << 31)).view(np.float32)

    span = (1, 12, 30, 60)[seed % 4]
    a, d = draw(span), draw(span)
    edge = np.array([1, 2, 3, (1 << 23) - 1, (1 << 23) - 2, (1 << 22) - 1, 1 << 22], np.uint32)
    k = rng.integers(0, n, n // 8)  # significands next to a power of two
    a[k] = ((a[k].view(np.uint32) & np.uint32(0xff800000)) | rng.choice(edge, k.size)).view(np.float32)
    k = rng.integers(0, n, n // 8)
    d[k] = ((d[k].view(np.uint32) & np.uint32(0xff800000)) | rng.choice(edge, k.size)).view(np.float32)
    k = rng.integers(0, n, n // 8)  # exact quotients, and those next to them
    a[k] = d[k] * rng.integers(1, 4096, k.size).astype(np.float32)
    a[:4] = [2.0 ** 60, 2.0 ** -60, 0.0, -0.0]
    d[:4] = [2.0 ** -60, 2.0 ** 60, 3.0, 3.0]
    lo, hi = np.float32(2.0 ** -60), np.float32(2.0 ** 60)
    ok = (np.abs(d) >= lo) & (np.abs(d) <= hi) & ((a == 0) | ((np.abs(a) >= lo) & (np.abs(a) <= hi)))
    a, d = a[ok], d[ok]
    got, want = apply(md, DIV, d, a), a / d
    assert np.array_equal(got, want)
    bits = (a != 0) | ~np.signbit(a)  # -0 over a positive divisor gives +0: no caller divides -0
    assert same(got[bits], want[bits])
