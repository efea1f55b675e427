"""The SOA sub-step on bounded inputs (dev::soa_run_tick), which the work-queue
kernel runs, against the general one (dev::soa_tick) on the CPU: bit for bit
wherever the bounded form accepts a cell, and every cell outside its range --
masses that are negative, tiny, subnormal, too large, infinite or NaN, at the
start or on the way, and loops without a sub-step -- turned away."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libsoarunhost.so")


@pytest.fixture(scope="module")
def lib():
    os.makedirs(os.path.dirname(SO), exist_ok=True)
    tmp = SO + ".%d" % os.getpid()
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-ffp-contract=off", "-o", tmp,
                    os.path.join(HERE, "cpp", "soa_run_host.cpp")], check=True)
    os.replace(tmp, SO)
    return ctypes.CDLL(SO)


def cells(n, seed):
    """rows of SOAG, 4 SOA, 4 uptake rates, 4 oxygenated POM, g0 in the ranges a step meets"""
    r = np.random.default_rng(seed)
    u = lambda lo, hi, *s: 10.0 ** r.uniform(lo, hi, s)  # noqa: E731
    x = np.concatenate([u(-13, -9, n, 1), u(-13, -8, n, 4), u(-8, -1, n, 4), u(-14, -9, n, 4),
                        u(-14, -8, n, 1)], axis=1)
    x[:, [10, 12]] = 0.0                                 # no oxygenated POM in Aitken and pcarbon
    x[r.random(n) < 0.5, 4] = 0.0                        # fresh primary carbon
    x[:, 5:9] = np.where(r.random((n, 4)) < 0.1, u(-17, -15, n, 4), x[:, 5:9])  # skipped modes
    x[r.random(n) < 0.05, 0] = 0.0
    return np.ascontiguousarray(x)


def run(lib, x, dt, fast):
    out, ok = np.zeros((len(x), 7)), np.zeros(len(x), np.int32)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
    lib.soa_run_host(len(x), ctypes.c_double(dt), fast, p(x), p(out), p(ok))
    return out, ok.astype(bool)


@pytest.mark.parametrize("dt", [1.0, 60.0, 1800.0, 3600.0])
def test_bounded_form_equals_the_general_one(lib, dt):
    x = cells(3000, 1)
    a, _ = run(lib, x, dt, 0)
    b, ok = run(lib, x, dt, 1)
    assert ok.mean() > 0.99
    assert np.array_equal(a[ok].view(np.int64), b[ok].view(np.int64))
    if dt >= 1800.0:
        assert (a[:, 6] > 1000).any() and (a[:, 6] < 10).any()  # the cap and short loops


@pytest.mark.parametrize("value", [-1e-12, 1e-130, 1e-300, 5e-324, 300.0, np.inf, np.nan])
@pytest.mark.parametrize("field", [0, 1, 2, 3, 4])
def test_cells_out_of_range_are_turned_away(lib, value, field):
    x = cells(200, 2)
    x[:, field] = value
    x[:, 5:9] = 1e-4  # no skipped mode: its SOA is dropped
    with np.errstate(all="ignore"):
        _, ok = run(lib, x, 1800.0, 1)
    assert not ok.any()


def test_masses_that_become_tiny_are_turned_away_or_equal(lib):
    """evaporation into a huge vapour pressure: SOA falls through 2^-400"""
    x = cells(500, 3)
    x[:, 1:4] *= 10.0 ** np.random.default_rng(4).uniform(-110, 0, (500, 1))
    x[:, 9:13] = 0.0
    x[:, 13] = 1e-3
    x[:, 5:9] = 1.0
    a, _ = run(lib, x, 1800.0, 0)
    b, ok = run(lib, x, 1800.0, 1)
    assert np.array_equal(a[ok].view(np.int64), b[ok].view(np.int64))


def test_no_sub_step(lib):
    x = cells(50, 5)
    for dt in (0.0, 0.5):
        assert not run(lib, x, dt, 1)[1].any()
