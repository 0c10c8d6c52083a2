"""Calls whose host arrays cannot be had return C2A_ERR_OOM: nothing is thrown
across the C entries."""
import ctypes as C

import numpy as np
import pytest

import c2a_amd as G
from c2a_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_counts_no_memory_holds_are_refused():
    t9 = W.torus_knot(n_seg=24, n_ring=5)[0].reshape(-1, 9)
    meshes = [G.Mesh(t9), G.Mesh(t9)]
    L, mt, nq = G.lib(), G._mesh_table(meshes), 1 << 58
    d, i, o = np.zeros(64), np.zeros(64, np.int32), np.zeros(4096, np.uint8)
    dp, ip, vp = G._dp(d), G._ip(i), C.c_void_p(o.ctypes.data)
    p, b = G.default_params(), C.c_void_p()
    calls = {
        "step": lambda n: L.c2a_ccd_step(mt, 2, (G.StepQuery * 1)(), n, (G.StepResult * 1)(), None),
        "contacts": lambda n: L.c2a_contact_count(mt, 2, dp, ip, dp, n, ip, None),
        "distance": lambda n: L.c2a_distance(mt, 2, dp, ip, None, 0.0, 0.0, n, vp, None),
        "queue": lambda n: L.c2a_distance_queue(mt, 2, dp, ip, None, 0.0, 0.0, 8, n, vp, None),
        "tolerance": lambda n: L.c2a_tolerance(mt, 2, dp, ip, dp, 2, n, vp, None),
        "collide": lambda n: L.c2a_collide_pairs(mt, 2, dp, ip, 1, n, 0, None, vp, None),
        "batch": lambda n: L.c2a_batch_create(mt, 2, (G.Query * 1)(), n, C.byref(p), C.byref(b)),
    }
    for name, call in calls.items():
        print("no host memory: %s" % name, flush=True)
        assert call(nq) == G.ERR_OOM, name
        assert b"host allocation failed" in L.c2a_last_error()
