"""The launches a default batch makes on either side of four queries per
compute unit: four wavefronts per query below, one wavefront and the hand-over
of the last queries above.  Every field equals the run with one wavefront per
query in one launch, in both orders, and tail_count says what was handed over."""
import numpy as np
import pytest
import torch

import c2a_amd as G
from c2a_amd import learn
from c2a_amd import workloads as W

pytestmark = pytest.mark.gpu


def same(a, b):
    for f in a.dtype.names:
        assert np.array_equal(a[f], b[f]), f


@pytest.mark.parametrize("learned", [0, 1])
def test_default_batch_equals_one_launch(learned):
    t, idx = W.torus_knot(n_seg=64, n_ring=8)
    meshes = [G.Mesh(t.reshape(-1, 9), vidx=idx), G.Mesh(t.reshape(-1, 9), vidx=idx)]
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    line = 4 * cus
    P = W.knot_queries(line + 300, 33, 0.4)
    sc = G.Scorer(path=learn.DEFAULT_SCORER) if learned else None
    kw = dict(tol_d=1e-3, tol_t=1e-4, with_contacts=1)
    if learned:
        kw.update(order=G.ORDER_LEARNED, scorer=sc)
    ref = G.ccd_batch(meshes, G.make_queries(*P), G.default_params(waves_per_query=1, **kw))
    if learned:
        plain = G.ccd_batch(meshes, G.make_queries(*P), G.default_params(tol_d=1e-3, tol_t=1e-4))
        assert not np.array_equal(plain["bv_tests"], ref["bv_tests"])
    for nq in (1, 3, line, line + 1, line + 300):
        print("hand-over learned=%d nq=%d" % (learned, nq), flush=True)
        b = G.Batch(meshes, G.make_queries(*[p[:nq] for p in P]), G.default_params(**kw),
                    scorer=sc)
        assert b.tail_count() == 0   # not run yet
        b.run()
        same(ref[:nq], b.fetch())
        assert (0 < b.tail_count() <= cus) if nq > line else b.tail_count() == 0
        if nq > line and not learned:
            for _ in range(3):
                b.run_graph()
                torch.cuda.synchronize()
                same(ref[:nq], b.fetch())
                assert 0 < b.tail_count() <= cus
                b.run()
                same(ref[:nq], b.fetch())
