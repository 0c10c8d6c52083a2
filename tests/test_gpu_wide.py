"""Four wavefronts per query for small batches: the same results, every field,
as one wavefront per query, on both sides of the lines between the two (4
queries per compute unit for CCD, 2 for distance and contact queries), for
device-resident queries, strict mode, contacts and hierarchies of one leaf."""
import numpy as np
import pytest
import torch

import c2a_amd as G
from c2a_amd import workloads as W

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
