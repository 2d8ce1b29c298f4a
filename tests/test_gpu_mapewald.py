"""FP32 Ewald maps by near pairs and an interpolated far field against the
FP64 maps (direct sums), every column of the node values."""
import numpy as np
import pytest

from musichip import hip as H
from musichip import synth

pytestmark = pytest.mark.gpu


def _box(cells, edge, seed):
    rng = np.random.default_rng(seed)
    L = np.array(edge, dtype=np.float64)
    xyz = synth.lattice_faces(cells, 1.0, rng) / cells * L
    q = rng.uniform(-1.0, 1.0, len(xyz))
    return xyz, q - q.mean(), L


# edges, cells per axis, spacing, alpha, kmax: tiles of 40, 32, 24 and 16 nodes that
# do not divide the grid; a cutoff beyond half the edge (every tile has
# atoms whose image changes inside it); unequal edges; and the smallest grid
@pytest.mark.parametrize("edge,cells,spacing,alpha,kmax", [
    ((24.0, 24.0, 24.0), 3, 0.16, 0.42, 5),
    ((21.3, 21.3, 21.3), 3, 0.19, 0.25, 4),
    ((33.0, 29.5, 31.7), 4, 0.25, 0.33, 5),
    ((40.0, 40.0, 40.0), 5, 0.41, 0.30, 5),
    ((12.0, 12.0, 12.0), 2, 0.5, 0.40, 3),
])
def test_far_field_matches_the_direct_sum(edge, cells, spacing, alpha, kmax):
    xyz, q, L = _box(cells, edge, 11)
    ctx = H.Context(0)
    ctx.upload_framework(xyz, np.zeros(len(xyz), dtype=np.int32), q, L, L)
    ctx.set_ewald(alpha * L.min(), kmax, 1e-10)
    node = {}
    for prec in (H.MH_PREC_FP32, H.MH_PREC_FP64):
        m = ctx.build_map(H.MH_MAP_EWALD, prec, spacing, 100.0, keep_full=True)
        node[prec] = m.get_full()[1]
        m.close()
    a, b = node[H.MH_PREC_FP32], node[H.MH_PREC_FP64]
    far = np.abs(b[:, 0]) < 200.0  # nodes off the atoms' cores
    assert far.sum() > 0.5 * len(b)
    # interpolation 1e-9 of V and 1e-7 of the derivatives, the cut at erfc =
    # 1e-9 and the A&S fit's 1.5e-7 / r^2 in the derivatives: under 1e-6 of a
    # column's rms; the FP32 pair route of the smallest grid: 5e-5 kcal/mol
    for c in range(8):
        rms = np.sqrt((b[far, c] ** 2).mean())
        err = np.abs(a[far, c] - b[far, c]).max()
        print("column %d: max error %.2e of rms %.3e" % (c, err / rms, rms), flush=True)
        assert err < 5e-6 * rms + 5e-5
