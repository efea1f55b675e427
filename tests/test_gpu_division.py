"""The SOA sub-step's fast division (scalar.hpp, num::div_fast) against IEEE
a / b on the GPU, bit for bit (tests/cpp/div_check.hip): 2 x 2^24 operand
pairs spanning the ranges the sub-step feeds it, and 2 x 2^24 pairs whose
numerators lie in 2^-1074..2^-960, either side of the 2^-968 bound.  Inside
the range the division is exact on (numerator 0 or >= 2^-968, quotient
normal) no pair may differ; outside it some do, which is why the sub-step
checks that its operands stay inside (chain_device.hpp, soa_fast_exact).
Numerator zeros are +0: a -0 numerator gives +0 where IEEE gives -0, and the
sub-step's numerators are sums and products of non-negative values clipped
with max(x, 0), never -0."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(HERE, "_build", "libdivcheck.so")


@pytest.mark.parametrize("tiny", [0, 1], ids=["sub-step-range", "tiny-numerators"])
def test_division_is_correctly_rounded(tiny):
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    torch.cuda.init()
    if not os.path.exists(LIB):
        pytest.fail("%s not built: run __graft_entry__.build()" % LIB)
    lib = ctypes.CDLL(LIB)
    lib.div_check.restype = ctypes.c_longlong
    lib.div_check.argtypes = [ctypes.c_long, ctypes.c_ulonglong, ctypes.c_int,
                              ctypes.POINTER(ctypes.c_double),
                              ctypes.POINTER(ctypes.c_ulonglong)]
    first = (ctypes.c_double * 2)()
    outside = (ctypes.c_ulonglong * 2)()
    for seed in (1, 0x5eed):
        bad = lib.div_check(1 << 24, seed, tiny, first, outside)
        print("tiny %d seed %d: inside mismatches %d, outside %d of %d pairs"
              % (tiny, seed, bad, outside[0], outside[1]))
        assert bad == 0, (bad, first[0], first[1])
        if tiny:
            # the bound is where exactness ends: a few percent of the pairs
            # below it round differently
            assert outside[1] > (1 << 22) and outside[0] > 1000
        else:
            assert outside[1] == 0


def hard_pairs(divisors, rhos):
    """Numerators a with a / b beside the midpoint of two neighbouring doubles:
    for an odd 53-bit integer b, m = -rho / b mod 2^54 is odd, and with m of 54
    bits (a midpoint) a = (m b + rho) / 2^54 has a / b = 2^-54 (m + rho / b)."""
    a, b = [], []
    for d in divisors:
        inv = pow(d, -1, 1 << 54)
        for rho in rhos:
            m = -rho * inv % (1 << 54)
            if m >= 1 << 53:
                a.append((m * d + rho) >> 54)
                b.append(d)
    return np.array(a, dtype=np.float64), np.array(b, dtype=np.float64)


def quotients(a, b):
    """num::rcp(b), num::div_fast(a, b), 1 / b and a / b on the GPU"""
    import torch
    if not torch.cuda.is_available():
        pytest.fail("GPU test run without a GPU")
    if not os.path.exists(LIB):
        pytest.fail("%s not built: run __graft_entry__.build()" % LIB)
    lib = ctypes.CDLL(LIB)
    assert len(a) == len(b)
    da, db = torch.as_tensor(a).cuda(), torch.as_tensor(b).cuda()
    out = torch.empty((4, len(a)), dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
    assert lib.div_arrays(ctypes.c_long(len(a)), p(da), p(db), p(out)) == 0
    return out.cpu().numpy()


def differ(x, y):
    return np.flatnonzero(x.view(np.int64) != y.view(np.int64))


@pytest.mark.parametrize("scale", [-60, 0, 13])
def test_quotients_that_are_hard_to_round(scale):
    """Divisors just below a power of two, whose reciprocals lie closest to a
    midpoint, and any others, with numerators whose quotients do: the compiler's
    a / b bit for bit, for which the two sequences have to be the same.

    The reciprocals: 1 / (1 - j 2^-53) with odd j is j^2 2^-106 above a midpoint.
    The first Newton step leaves at most e = 2^-48.7 (the seed's 2^-24.37
    squared) and the second ends e^2 below, so only where j < 2^53 e < 32 may it
    fall on the wrong side."""
    rng = np.random.default_rng(7)
    near = [(1 << 53) - j for j in range(1, 1 << 17, 2)]
    some = [int(x) | 1 for x in rng.integers(1 << 52, 1 << 53, 20000)]
    for name, div, rhos in (("near", near, (1, -1, 3, -3)), ("any", some, range(-9, 10, 2))):
        a, b = hard_pairs(div, rhos)
        assert len(a) > 1 << 16
        j = (1 << 53) - b
        a, b = np.ldexp(a, scale - 52), np.ldexp(b, scale - 52)
        r, q, _, q0 = quotients(a, b)
        d = differ(q, q0)
        assert len(d) == 0, (name, [(x.hex(), y.hex()) for x, y in zip(a[d[:3]], b[d[:3]])])
        d = differ(r, 1.0 / b)
        assert (j[d] < 32).all(), (name, [x.hex() for x in b[d[:3]]])
        print("%s divisors: of %d pairs %d reciprocals and %d quotients differ from the CPU's"
              % (name, len(a), len(d), len(differ(q, a / b))))


@pytest.mark.parametrize("seed", [1, 2, 3, 4])
def test_reciprocals_are_correctly_rounded(seed):
    """2^24 random divisors; the reverse sweep takes the reciprocals uncorrected"""
    rng = np.random.default_rng(seed)
    b = np.ldexp(rng.uniform(1.0, 2.0, 1 << 24), rng.integers(-80, 80, 1 << 24))
    r, _, r0, _ = quotients(np.ones_like(b), b)
    for x in (r0, 1.0 / b):
        d = differ(r, x)
        assert len(d) == 0, [y.hex() for y in b[d[:3]]]
