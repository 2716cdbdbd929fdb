"""`linear` with one relation per edge at the edges of its kernels' tiles (64 sorted edges x 64 columns, 16 values of k):
both directions of the per-relation products against the oracle, dims that no vector load fits among them, and tiles that
hold one relation, several, or part of one.  Criterion and slack are those of the many-workers comparison (Adagrad turns a
gradient that is rounding noise into a full step)."""
import pytest

import tests.test_gpu_many_workers as many

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 2, 30, 33, 66, 128, 130])
@pytest.mark.parametrize("relations,num_pos,workers", [(1, 64, 1), (3, 65, 2), (40, 63, 3)])
def test_linear_dynamic_tile_edges(pbg, monkeypatch, dim, relations, num_pos, workers):
    monkeypatch.setitem(many.CASES, "tiles dim %d relations %d" % (dim, relations),
                        dict(operator="linear", comparator="dot", loss="logistic", dim=dim, num_pos=num_pos, dynamic=True,
                             num_batch_negs=16, num_uniform_negs=9, entities=400, relations=relations, scale=0.3, ks=(workers,)))
    many.test_many_workers_match_the_lockstep_oracle(pbg, "tiles dim %d relations %d" % (dim, relations), workers)
