"""Static queries with one wavefront per query (static_wave.h) against the
one-thread search they replace: every field, for the contact lists (all and
first, lists shorter than the contacts, no list), tolerance and contact space,
over meshes from a single triangle to hierarchies whose batches are ragged.
On the CPU with 64 lanes; on the GPU, lists just below and above the
wavefront's longest against each other."""
import ctypes as C
import os

import numpy as np
import pytest

import c2a_amd as G
from c2a_amd import workloads as W
from tests import test_static_queries as S

HERE = os.path.dirname(os.path.abspath(__file__))


def mesh(kind):
    if kind == "one":
        return np.array([[0.0, 0.0, 0.0, 0.9, 0.0, 0.1, 0.0, 0.8, -0.1]])
    if kind == "three":
        return W.icosphere(1, 0.1, 3)[0].reshape(-1, 9)[:3]
    if kind == "ball":
        return W.icosphere(2, 0.15, 51)[0].reshape(-1, 9)
    return W.torus_knot(n_seg=24, n_ring=5)[0].reshape(-1, 9)


def wave(t1, t2, kind, P, params=None, flag=1, cap=0):
    L = C.CDLL(os.environ.get("CCD_EMU64", os.path.join(HERE, "emu", "libccd_emu64.so")))
    dp, ip = C.POINTER(C.c_double), C.POINTER(C.c_int32)
    L.emu_static_wave.argtypes = [dp, C.c_int64, dp, C.c_int64, C.c_int, dp, dp, C.c_int,
                                  C.c_int64, C.c_int, ip, C.c_void_p]
    out = np.zeros(len(P), S.STATIC_OUT)
    pairs = np.full((len(P), max(cap, 1), 2), -1, np.int32)
    pr = None if params is None else np.ascontiguousarray(params, np.float64)
    rc = L.emu_static_wave(S._dp(t1), len(t1), S._dp(t2), len(t2), kind,
                           S._dp(np.ascontiguousarray(P)), None if pr is None else S._dp(pr),
                           flag, len(P), cap, S._ip(pairs), out.ctypes.data)
    assert rc == 0
    return out, pairs


def same(a, b):
    for f in S.STATIC_OUT.names:
        assert np.array_equal(a[0][f], b[0][f]), f
    assert np.array_equal(a[1], b[1])


PAIRS = [("one", "one"), ("one", "ball"), ("three", "knot"), ("ball", "ball"), ("knot", "knot")]


@pytest.mark.parametrize("m1,m2", PAIRS)
@pytest.mark.parametrize("flag,cap", [(1, 2048), (1, 3), (1, 1), (1, 0), (2, 4), (2, 0)])
def test_wave_collide(m1, m2, flag, cap):
    t1, t2 = mesh(m1), mesh(m2)
    P = S.cases(11, 6, seps=(0.0, 0.3, 0.7, 0.95, 1.05, 2.9))
    got = wave(t1, t2, S.SQ_COLLIDE, P, flag=flag, cap=cap)
    same(S.run_emu(t1, t2, S.SQ_COLLIDE, P, flag=flag, cap=cap), got)
    if m1 == "ball":
        assert (got[0]["found"] > 0).any() and (got[0]["found"] == 0).any()


@pytest.mark.parametrize("m1,m2", PAIRS)
@pytest.mark.parametrize("kind", [S.SQ_TOLERANCE, S.SQ_DISTANCE_CS])
def test_wave_first_found(m1, m2, kind):
    t1, t2 = mesh(m1), mesh(m2)
    P = S.cases(12, 5)
    base = S.run_emu(t1, t2, S.SQ_DISTANCE_QUEUE, P, qsize=64)[0]["distance"]
    for lim in (base * 0.99, base, base * 1.01 + 1e-3, base + 0.4, np.full(5, np.inf),
                np.zeros(5), np.full(5, -1.0)):
        same(S.run_emu(t1, t2, kind, P, params=lim), wave(t1, t2, kind, P, params=lim))


@pytest.mark.gpu
@pytest.mark.parametrize("cap", [1, 40, 2048])
def test_gpu_wave_lists_equal_thread_lists(cap):
    t1 = mesh("ball")
    meshes = [G.Mesh(t1), G.Mesh(mesh("knot"))]
    P = S.cases(13, 130, seps=(0.0, 0.4, 0.8, 1.0, 1.2))
    mp = np.tile([0, 1], (len(P), 1))
    print("collide pairs cap=%d" % cap, flush=True)
    r, pairs = G.collide_pairs(meshes, P, mp, flag=1, cap=cap)
    r2, pairs2 = G.collide_pairs(meshes, P, mp, flag=1, cap=2049)   # one thread per query
    for f in r.dtype.names:
        assert np.array_equal(r[f], r2[f]), f
    assert np.array_equal(pairs, pairs2[:, :cap])
    assert (r["found"] > 40).any()
