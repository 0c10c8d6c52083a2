"""Four wavefronts per query (K = 7, 256 lanes), the shape of small batches and
of a batch's last queries, on the CPU: ccd_core.h under its index checks with
wavefronts that run one after another between workgroup barriers, first to
last and last to first (tests/emu/simt.cpp), so that a missing barrier between
them gives a wrong result.  Field by field against the FP64 oracle, or, for
the learned order, against one wavefront."""
import ctypes as C
import os

import numpy as np
import pytest

import c2a_amd as G
from c2a_amd import workloads as W
from oracle import oracle as O
from tests import test_distance as D
from tests.test_kernel_heaps_cpu import mesh
from tests.test_kernel_logic_cpu import chain_queries, factorial_chain, run_emu, same

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(params=[0, 1], ids=["forward", "backward"])
def emu(request):
    L = C.CDLL(os.environ.get("CCD_EMU64", os.path.join(HERE, "emu", "libccd_emu64.so")))
    L.emu_set_scorer.argtypes = [C.c_void_p]
    L.emu_tail_count.restype = C.c_int64
    L.backward = request.param
    L.emu_set_arena_rounds(0)
    L.emu_set_ext_adaptive(1)
    L.emu_set_waves(4, request.param)
    yield L
    L.emu_set_waves(1, 0)
    L.emu_set_tail_shape(0, 0)
    L.emu_set_tail_left(0)
    L.emu_set_scorer(None)
    L.emu_set_distance_k(5)
    L.emu_set_ext_adaptive(0)
    L.emu_set_arena_rounds(1)


def queries(nq, seed, translation=False):
    P = W.knot_queries(nq, seed, 0.8)
    if translation:   # the first query does not rotate
        P[1][0, :9], P[3][0, :9] = P[0][0, :9], P[2][0, :9]
    return P


def oracle(t1, t2, P):
    return O.batch_toc(O.OModel(t1), O.OModel(t2), *P, 1e-3, 1e-4,
                       seeds=np.zeros((len(P[0]), 2), np.int32), with_contacts=True)


@pytest.mark.parametrize("m1,m2", [("knot", "knot"), ("one", "knot"), ("three", "one")])
@pytest.mark.parametrize("kw", [dict(miss_depth=4, ext_levels=1), dict(miss_depth=1),
                                dict(miss_depth=3, ext_levels=2, replay_log=64),
                                dict(replay_log=0)], ids=lambda k: "-".join(map(str, k.values())))
def test_waves_ccd(emu, m1, m2, kw):
    t1, t2 = mesh(m1), mesh(m2)
    P = queries(3, 70, translation=True)
    got = run_emu(emu, t1, t2, P, G.default_params(tol_d=1e-3, tol_t=1e-4, **kw), 7)
    same(oracle(t1, t2, P), got)


def test_waves_strict(emu):
    t = mesh("knot")
    P = queries(3, 71)
    with O.strict_mode():
        ref = oracle(t, t, P)
    same(ref, run_emu(emu, t, t, P, G.default_params(tol_d=1e-3, tol_t=1e-4, strict=1), 7))


def test_waves_96_entry_stack(emu):
    """Hierarchies too deep together for the 48-entry stack."""
    t1, t2 = factorial_chain(56, 1), factorial_chain(56, 2, mirror=True)
    need = G.Mesh(t1).max_depth + G.Mesh(t2).max_depth + 2
    assert 48 < need <= 96, need
    nq = 3
    P = chain_queries(nq, 808)
    seeds = np.full((nq, 2), 55, np.int32)
    ref = O.batch_toc(O.OModel(t1), O.OModel(t2), *P, 1e-6, 1e-6, seeds=seeds, with_contacts=True)
    same(ref, run_emu(emu, t1, t2, P, G.default_params(tol_d=1e-6, tol_t=1e-6, miss_depth=4), 7,
                      seeds=seeds))


def scorer_params():
    return (np.random.default_rng(3).normal(size=G.Scorer.NPARAM) * 0.1).astype(np.float32)


def one_wavefront(emu, f):
    emu.emu_set_waves(1, 0)
    try:
        return f()
    finally:
        emu.emu_set_waves(4, emu.backward)


def test_waves_learned_order(emu):
    t = mesh("knot")
    P = queries(3, 73)
    w = scorer_params()
    emu.emu_set_scorer(w.ctypes.data)
    kw = dict(tol_d=1e-3, tol_t=1e-4, miss_depth=3)
    ref = one_wavefront(emu, lambda: run_emu(emu, t, t, P, G.default_params(**kw), 5))
    got = run_emu(emu, t, t, P, G.default_params(**kw), 7)
    plain = oracle(t, t, P)
    assert not np.array_equal(ref["bv_tests"], plain["num_bv_tests"])   # it orders by score
    for f in ref.dtype.names:
        assert np.array_equal(ref[f], got[f]), f


@pytest.mark.parametrize("learned", [0, 1])
def test_last_query_goes_on_with_four_wavefronts(emu, learned):
    """The hand-over as the library makes it: one wavefront per query, then
    four on the last one, in the first run's arena."""
    t = mesh("knot")
    P = queries(4, 3)
    if learned:
        w = scorer_params()
        emu.emu_set_scorer(w.ctypes.data)
    kw = dict(tol_d=1e-3, tol_t=1e-4, ext_levels=0 if learned else 1, miss_depth=3)
    ref = one_wavefront(emu, lambda: run_emu(emu, t, t, P, G.default_params(**kw), 5))
    emu.emu_set_waves(1, 0)
    emu.emu_set_tail_shape(7, 4)
    emu.emu_set_tail_left(2)
    got = run_emu(emu, t, t, P, G.default_params(**kw), 5)
    assert emu.emu_tail_count() == 1
    for f in ref.dtype.names:
        assert np.array_equal(ref[f], got[f]), f


@pytest.mark.parametrize("rel,abs_,overlap", [(0.0, 0.0, 0), (0.5, 0.02, 0), (0.0, 0.0, 1)])
def test_waves_distance(emu, rel, abs_, overlap):
    emu.emu_set_distance_k(7)
    a, b = mesh("knot"), mesh("three")
    for t1, t2 in ((a, a), (a, b)):
        rng = np.random.default_rng(5)
        cases = [D.random_case(rng, s) for s in rng.uniform(0.0, 1.6, 4)]
        seeds = np.stack([rng.integers(0, len(t1), 4), rng.integers(0, len(t2), 4)], 1)
        ref = D.oracle_batch(t1, t2, cases, rel, abs_, seeds, overlap_only=bool(overlap))
        D.check_same(ref, D.run_emu(emu, t1, t2, cases, rel, abs_, seeds, overlap_only=overlap))
