"""Four wavefronts per query for small batches: the same results, every field,
as one wavefront per query, on both sides of the lines between the two (4
queries per compute unit for CCD, 2 for distance, contact and explicit-step
queries), for device-resident queries, strict mode, contacts, hierarchies of
one leaf, and hierarchies that take the deeper stacks."""
import numpy as np
import pytest
import torch

import c2a_amd as G
from c2a_amd import workloads as W
from tests import test_distance as D
from tests.test_kernel_logic_cpu import chain_queries, factorial_chain
from tests.test_zz_no_alloc import run_noalloc

pytestmark = pytest.mark.gpu


def cus():
    return torch.cuda.get_device_properties(0).multi_processor_count


def same(a, b):
    for f in a.dtype.names:
        assert np.array_equal(a[f], b[f]), f


@pytest.mark.parametrize("strict", [0, 1])
def test_wide_ccd(strict):
    t, idx = W.torus_knot(n_seg=64, n_ring=8)
    t9 = t.reshape(-1, 9)
    meshes = [G.Mesh(t9, vidx=idx), G.Mesh(t9, vidx=idx), G.Mesh(t9[:1])]
    n = 4 * cus()
    P = W.knot_queries(n + 1, 31, 0.4)
    mp = np.tile([0, 1], (n + 1, 1))
    mp[::7, 1] = 2
    kw = dict(tol_d=1e-3, tol_t=1e-4, with_contacts=1, strict=strict)
    ref = G.ccd_batch(meshes, G.make_queries(*P, mesh_pairs=mp), G.default_params(**kw))
    for k in (1, 3, n):
        print("wide strict=%d nq=%d" % (strict, k), flush=True)
        q = G.make_queries(*[p[:k] for p in P], mesh_pairs=mp[:k])
        same(ref[:k], G.ccd_batch(meshes, q, G.default_params(**kw)))
        one = G.ccd_batch(meshes, q, G.default_params(waves_per_query=1, **kw))
        same(ref[:k], one)
    assert (ref["num_contact"] > 0).any() and (ref["collisionfree"] == 1).any()


def test_wide_static():
    t9 = W.torus_knot(n_seg=64, n_ring=8)[0].reshape(-1, 9)
    meshes = [G.Mesh(t9), G.Mesh(t9)]
    n = 2 * cus()
    P = W.knot_queries(n + 1, 32, 0.4)
    poses = np.concatenate([P[0], P[2]], axis=1)
    mp = np.tile([0, 1], (n + 1, 1))
    ref = G.distance(meshes, poses, mp)
    thr = ref["distance"] + 0.02
    cnt, rec = G.contact_list(meshes, poses, mp, thr, 40)
    for k in (1, n):
        print("wide static nq=%d" % k, flush=True)
        same(ref[:k], G.distance(meshes, poses[:k], mp[:k]))
        c, r = G.contact_list(meshes, poses[:k], mp[:k], thr[:k], 40)
        assert np.array_equal(cnt[:k], c)
        for i in range(k):
            assert np.array_equal(rec[i, :min(c[i], 40)], r[i, :min(c[i], 40)])
    assert (cnt > 1).any()


@pytest.mark.parametrize("contacts", [0, 1])
def test_wide_device_resident(contacts):
    t9 = W.torus_knot(n_seg=64, n_ring=8)[0].reshape(-1, 9)
    meshes = [G.Mesh(t9), G.Mesh(t9)]
    n = 4 * cus()
    P = W.knot_queries(n + 1, 34, 0.4)
    kw = dict(tol_d=1e-3, tol_t=1e-4, with_contacts=contacts)
    ref = G.ccd_batch(meshes, G.make_queries(*P), G.default_params(waves_per_query=1, **kw))
    for k in (1, n, n + 1):
        print("wide noalloc contacts=%d nq=%d" % (contacts, k), flush=True)
        same(ref[:k], run_noalloc(meshes, [p[:k] for p in P], G.default_params(**kw)))


@pytest.mark.parametrize("n,cap", [(56, 96), (100, 192)])
def test_wide_stacks(n, cap):
    """Chains whose pairs take the 96-entry stack, and the 192-entry one, which
    only one wavefront has (the full kernel, also for static queries)."""
    t1, t2 = factorial_chain(n, 1), factorial_chain(n, 2, mirror=True)
    meshes = [G.Mesh(t1), G.Mesh(t2)]
    need = meshes[0].max_depth + meshes[1].max_depth + 2
    assert cap // 2 < need <= cap
    line = 2 * cus()
    P = chain_queries(line + 1, 909)
    poses, mp = np.concatenate([P[0], P[2]], axis=1), np.tile([0, 1], (line + 1, 1))
    ref = G.distance(meshes, poses, mp)
    pose = lambda a: (a[:9].reshape(3, 3), a[9:])   # noqa: E731
    cases = [pose(P[0][i]) + pose(P[2][i]) for i in range(4)]
    D.check_same(D.oracle_batch(t1, t2, cases, 0.0, 0.0, np.zeros((4, 2), int)), ref)
    over = G.distance(meshes, poses, mp, overlap_only=True)
    thr = ref["distance"] + 1e-3
    cnt, rec = G.contact_list(meshes, poses, mp, thr, 30)
    assert (cnt > 0).all()
    st = (G.StepQuery * (line + 1))()
    for i in range(line + 1):
        s = st[i]
        s.R1[:], s.T1[:], s.R2[:], s.T2[:] = P[0][i, :9], P[0][i, 9:], P[2][i, :9], P[2][i, 9:]
        for k in range(2):
            s.pose_s[k][:], s.pose_e[k][:] = P[2 * k][i], P[2 * k + 1][i]
        s.mesh[:] = [0, 1]
        s.numCA, s.mint_prev, s.UpboundTOC = i % 8, 0.02, 1.0
    names = [f for f, _ in G.StepResult._fields_ if f != "pad"]
    step = lambda r: [tuple(np.ravel(getattr(r, f))) for f in names]   # noqa: E731
    steps = [step(r) for r in G.ccd_step(meshes, st)]
    q = G.default_params(tol_d=1e-6, tol_t=1e-6, waves_per_query=1)
    ccd = G.ccd_batch(meshes, G.make_queries(*P), q)
    for k in (1, line):
        print("wide stack %d nq=%d" % (cap, k), flush=True)
        same(ref[:k], G.distance(meshes, poses[:k], mp[:k]))
        same(over[:k], G.distance(meshes, poses[:k], mp[:k], overlap_only=True))
        c, r = G.contact_list(meshes, poses[:k], mp[:k], thr[:k], 30)
        assert np.array_equal(cnt[:k], c)
        for i in range(k):
            assert np.array_equal(rec[i, :min(c[i], 30)], r[i, :min(c[i], 30)])
        sub = (G.StepQuery * k)(*st[:k])
        assert [step(r) for r in G.ccd_step(meshes, sub)] == steps[:k]
        same(ccd[:k], G.ccd_batch(meshes, G.make_queries(*[p[:k] for p in P]),
                                  G.default_params(tol_d=1e-6, tol_t=1e-6)))
