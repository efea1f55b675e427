"""The SOA work queue's claims (csrc/queue_claims.hpp) on the CPU: every entry is
handed out once, over the accepted range of the claim sizes and up to the waves
of a full grid, where the 32-bit counters run furthest past the queue's end."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
SO = os.path.join(HERE, "_build", "libclaimshost.so")


@pytest.fixture(scope="module")
def lib():
    os.makedirs(os.path.dirname(SO), exist_ok=True)
    tmp = SO + ".%d" % os.getpid()
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-o", tmp,
                    os.path.join(HERE, "cpp", "claims_host.cpp")], check=True)
    os.replace(tmp, SO)
    return ctypes.CDLL(SO)


@pytest.mark.parametrize("nwave", [1, 4, 2048, 4096, 8192])
@pytest.mark.parametrize("chunk,short", [(0, 0), (1, 1), (7, 33), (1 << 18, 1 << 18),
                                         (64, 1 << 20), (1 << 20, 64), (1 << 20, 1 << 20)])
def test_every_entry_is_handed_out_once(lib, chunk, short, nwave):
    for nq in (0, 1, 31, 300001):
        for nsplit in sorted({0, nq // 3, nq}):
            seen = np.zeros(nq + 1, np.uint8)
            most = lib.claims_host(chunk, short, nwave, nq, nsplit,
                                   seen.ctypes.data_as(ctypes.c_void_p))
            assert 0 <= most <= 32
            assert (seen[:nq] == 1).all() and seen[nq] == 0, (nq, nsplit)
