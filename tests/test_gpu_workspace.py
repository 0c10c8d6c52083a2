"""The static queries' kept workspace: calls of different sizes one after
another and from several threads at once give what each gives alone, and the
workspace does not outlive the last mesh."""
import gc
import threading

import numpy as np
import pytest
import torch

import c2a_amd as G
from c2a_amd import workloads as W

pytestmark = pytest.mark.gpu


def test_workspace_is_shared_safely():
    t9 = W.torus_knot(n_seg=64, n_ring=8)[0].reshape(-1, 9)
    meshes = [G.Mesh(t9), G.Mesh(t9)]
    jobs = []
    for k, nq in enumerate((3, 700, 64, 257)):
        P = W.knot_queries(nq, 50 + k, 0.4)
        jobs.append((np.concatenate([P[0], P[2]], axis=1), np.tile([0, 1], (nq, 1))))

    def run(j):
        poses, mp = jobs[j]
        return (G.tolerance(meshes, poses, mp, 0.05), G.collide_pairs(meshes, poses, mp, cap=50),
                G.distance_queue(meshes, poses, mp, 8))

    def same(a, b):
        for f in a[0].dtype.names:
            assert np.array_equal(a[0][f], b[0][f]) and np.array_equal(a[1][0][f], b[1][0][f])
        assert np.array_equal(a[1][1], b[1][1])
        for f in a[2].dtype.names:
            assert np.array_equal(a[2][f], b[2][f])

    print("workspace: one after another", flush=True)
    ref = [run(j) for j in range(4)]
    for j in (1, 0, 3, 2):
        same(ref[j], run(j))
    print("workspace: four threads", flush=True)
    got = [None] * 4

    def work(j):
        got[j] = [run(j) for _ in range(3)]

    ths = [threading.Thread(target=work, args=(j,)) for j in range(4)]
    for t in ths:
        t.start()
    for t in ths:
        t.join()
    for j in range(4):
        for g in got[j]:
            same(ref[j], g)
    del meshes
    gc.collect()
    meshes = [G.Mesh(t9), G.Mesh(t9)]   # the workspace went with the last mesh
    same(ref[0], run(0))


def test_workspace_goes_with_the_last_mesh():
    t9 = W.torus_knot(n_seg=64, n_ring=8)[0].reshape(-1, 9)
    P = W.knot_queries(700, 51, 0.4)
    poses, mp = np.concatenate([P[0], P[2]], axis=1), np.tile([0, 1], (700, 1))
    gc.collect()
    if any(type(o) is G.Mesh for o in gc.get_objects()):
        pytest.skip("another test's mesh is alive: the workspace rightly stays")
    print("workspace: kept while a mesh lives, then freed", flush=True)
    for _ in range(2):
        meshes = [G.Mesh(t9), G.Mesh(t9)]
        G.tolerance(meshes, poses, mp, 0.05)
        held = torch.cuda.mem_get_info()[0]
        del meshes
        gc.collect()
        freed = torch.cuda.mem_get_info()[0]
    # 700 wavefronts' stacks of 32 pairs a level and more
    assert freed - held > 700 * 32 * 128
