"""The library's own rule for when many queries take the matrix-core kernel
(adaptq_amd/csrc/mquery_rule.hpp), so that a test of that kernel asserts that its
sizes reach it."""
import ctypes as C
import functools
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(None)
def _lib():
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "mquery_rule.so")
        subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC",
                        os.path.join(HERE, "cpp", "mquery_rule.cpp"), "-o", so], check=True)
        return C.CDLL(so)


def takes(heads, nq, n, padded):
    """Whether a dense decode of nq queries a head over n tokens takes it (2- to
    4-bit keys and values, padded 64 or 128)."""
    return padded in (64, 128) and bool(_lib().mq_takes(heads, nq, n, padded))


def heads_for(nq, n, padded):
    """The fewest heads at which it does."""
    return next(h for h in range(1, 100000) if takes(h, nq, n, padded))


def plan(heads, nq, n):
    out = (C.c_int * 5)()
    _lib().mq_plan_of(heads, nq, n, out)
    return dict(zip(("splits", "chunk", "qgroups", "qg", "qblocks"), out))
