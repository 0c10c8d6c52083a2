"""The lane-parallel decision of a round's heap (heap_scan in ccd_core.h) with
64 lanes on the CPU, against the FP64 oracle field by field: every heap depth
(2 to 62 pairs; K = 7: 256 slots, up to eight heaps a round), hierarchies that are a single leaf on one or both sides,
heaps cut short by leaf pairs, and each traversal that uses it (CCD steps,
contact enumeration, distance and its overlap-only form)."""
import ctypes as C
import os

import numpy as np
import pytest

import c2a_amd as G
from c2a_amd import workloads as W
from oracle import oracle as O
from tests import test_distance as D
from tests.test_kernel_logic_cpu import run_emu, same

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emu64():
    L = C.CDLL(os.environ.get("CCD_EMU64", os.path.join(HERE, "emu", "libccd_emu64.so")))
    L.emu_set_arena_rounds.argtypes = [C.c_int]
    L.emu_set_arena_rounds(0)
    yield L
    L.emu_set_distance_k(5)
    L.emu_set_arena_rounds(1)


def mesh(kind):
    if kind == "one":   # a single triangle: the root is a leaf
        return np.array([[0.0, 0.0, 0.0, 0.4, 0.0, 0.1, 0.0, 0.3, -0.1]])
    if kind == "three":
        return W.icosphere(1, 0.1, 3)[0].reshape(-1, 9)[:3]
    return W.torus_knot(n_seg=24, n_ring=5)[0].reshape(-1, 9)


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 7])
@pytest.mark.parametrize("m1,m2", [("knot", "knot"), ("one", "knot"), ("three", "one")])
def test_heaps_ccd_bit_exact(emu64, m1, m2, K):
    t1, t2 = mesh(m1), mesh(m2)
    nq = 5
    P = W.knot_queries(nq, 40 + K, 0.8)
    ref = O.batch_toc(O.OModel(t1), O.OModel(t2), *P, 1e-3, 1e-4,
                      seeds=np.zeros((nq, 2), np.int32), with_contacts=True)
    got = run_emu(emu64, t1, t2, P,
                  G.default_params(tol_d=1e-3, tol_t=1e-4, spec_depth=min(K, 6),
                                   miss_depth=min(K, 3)), K)
    same(ref, got)


@pytest.mark.parametrize("K", [5, 7])
@pytest.mark.parametrize("rel,abs_,overlap", [(0.0, 0.0, 0), (0.5, 0.02, 0), (0.0, 0.0, 1)])
def test_heaps_distance_bit_exact(emu64, rel, abs_, overlap, K):
    t1, t2 = mesh("knot"), mesh("three")
    emu64.emu_set_distance_k(K)
    for a, b in ((t1, t1), (t1, t2)):
        rng = np.random.default_rng(int(rel * 10 + 7))
        cases = [D.random_case(rng, s) for s in rng.uniform(0.0, 1.6, 8)]
        seeds = np.stack([rng.integers(0, len(a), 8), rng.integers(0, len(b), 8)], 1)
        ref = D.oracle_batch(a, b, cases, rel, abs_, seeds, overlap_only=bool(overlap))
        D.check_same(ref, D.run_emu(emu64, a, b, cases, rel, abs_, seeds, overlap_only=overlap))


@pytest.mark.parametrize("ext,log", [(0, -1), (1, -1), (1, 64), (0, 0)])
def test_last_query_handed_over(emu64, ext, log):
    """The last unfinished query goes on in a second run, with the replay log
    of the first (or without one): same results."""
    t = mesh("knot")
    P = W.knot_queries(4, 3, 0.6)
    kw = dict(tol_d=1e-3, tol_t=1e-4, ext_levels=ext, miss_depth=3, replay_log=log)
    ref = run_emu(emu64, t, t, P, G.default_params(**kw), 5)
    emu64.emu_tail_count.restype = C.c_int64
    emu64.emu_set_tail_left(2)
    try:
        got = run_emu(emu64, t, t, P, G.default_params(**kw), 5)
    finally:
        emu64.emu_set_tail_left(0)
    assert emu64.emu_tail_count() == 1
    for f in ref.dtype.names:
        assert np.array_equal(ref[f], got[f]), f
