"""Map compaction (64-node bit rows) against the oracle's serial scan, at the
edges of the rows' words and the smallest grids."""
import numpy as np
import pytest

from musichip import hip as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu


# grid nodes per axis: one word a row and less, exactly full words, one node
# into the next word, and the smallest grid the build accepts
@pytest.mark.parametrize("nodes", [(3, 3, 3), (3, 5, 4), (7, 4, 63), (5, 3, 64), (4, 6, 65), (9, 8, 127), (6, 5, 128),
                                   (3, 4, 129), (20, 21, 40)])
@pytest.mark.parametrize("cut_kJ", [0.5, 100.0])
def test_compaction_matches_the_serial_scan(nodes, cut_kJ):
    rng = np.random.default_rng(sum(nodes))
    h = 0.35
    L = np.array([(n - 1) * h + 1e-6 for n in nodes])
    # atoms dense enough that nodes of every kind (below, owned, rejected) occur
    n_at = max(2, int(L.prod() * 0.02))
    xyz = rng.uniform(0, 1, (n_at, 3)) * L
    ctx = H.Context(0)
    ctx.upload_framework(xyz, np.zeros(n_at, dtype=np.int32), np.zeros(n_at), L, L)
    ctx.set_lj([2.0e4], [150.0], [min(3.0, 0.49 * L.min()) ** 2], [1e-6])
    m = ctx.build_map(H.MH_MAP_LJ, H.MH_PREC_FP64, h, cut_kJ, keep_full=True)
    assert tuple(m.npnts) == nodes
    f32, _ = m.get_full()
    ptr_o, src, counts = O.compact(np.array(nodes), np.ascontiguousarray(f32[:, 0]), cut_kJ / 4.184)
    ptr, vals = m.get()
    assert list(m.counts) == list(counts)
    assert np.array_equal(ptr, ptr_o)
    assert np.array_equal(vals, f32[src].T)
