"""FP32 Ewald maps by near pairs and an interpolated far field against the
FP64 maps (direct sums), every column of the node values, on each route the
build can choose (the timer names tell which one ran)."""
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


# edges, cells per axis, spacing, alpha, kmax, map boxes per axis, route (None:
# the FP32 pair kernel): every tile size and level on unequal edges with tiles
# that do not divide the grid; a cutoff beyond half the edge, so that atoms
# change their image inside a tile; coarse grids and the smallest one, which
# take the pairs; a map of an eighth of the cell
@pytest.mark.parametrize("edge,cells,spacing,alpha,kmax,reps,route", [
    ((30.0, 26.0, 33.0), 5, 0.16, 0.40, 5, 1, "ewald_far24"),
    ((30.0, 27.0, 28.5), 5, 0.14, 0.35, 5, 1, "ewald_far16_two"),
    ((36.0, 36.5, 37.0), 5, 0.14, 0.28, 5, 1, "ewald_far24_two"),
    ((22.0, 21.3, 21.0), 3, 0.115, 0.25, 4, 1, "ewald_far16_two"),
    ((33.0, 29.5, 31.7), 4, 0.25, 0.33, 5, 1, None),
    ((40.0, 40.0, 40.0), 5, 0.41, 0.30, 5, 1, None),
    ((12.0, 12.0, 12.0), 2, 0.5, 0.40, 3, 1, None),
    ((44.0, 40.0, 42.0), 6, 0.115, 0.36, 5, 2, "ewald_far24_two"),
])
def test_far_field_matches_the_direct_sum(edge, cells, spacing, alpha, kmax, reps, route):
    xyz, q, L = _box(cells, edge, 11)
    ctx = H.Context(0)
    ctx.upload_framework(xyz, np.zeros(len(xyz), dtype=np.int32), q, L / reps, L)
    ctx.set_ewald(alpha * L.min(), kmax, 1e-10)
    node, ran = {}, {}
    for prec in (H.MH_PREC_FP32, H.MH_PREC_FP64):
        ctx.set_timing(True)
        m = ctx.build_map(H.MH_MAP_EWALD, prec, spacing, 100.0, keep_full=True)
        ran[prec] = [k for k in ctx.timings() if k.startswith("ewald_far")]
        ctx.set_timing(False)
        node[prec] = m.get_full()[1]
        m.close()
    assert ran[H.MH_PREC_FP32] == ([route] if route else []) and ran[H.MH_PREC_FP64] == []
    a, b = node[H.MH_PREC_FP32], node[H.MH_PREC_FP64]
    # nodes off the atoms' cores
    far = np.abs(b[:, 0]) < 200.0
    assert far.sum() > 0.5 * len(b)
    # Largest errors over a column's rms: what rounding each FP32 pair term
    # leaves (measured on the pair kernel: V 1.2e-7, first derivatives 3.6e-7,
    # second 1.5e-7, third 1.1e-8, more where few atoms are in reach); bricks
    # at the cutoff hold such values on every route.  The far field must stay
    # within them, and its rms errors at the cut at erfc = 1e-9 and the slope
    # of the A&S fit (second derivatives 1e-6 / r^3, third 1e-6 / r^4 beyond
    # 3.5 A); the first derivatives have no such term.
    worst = [2e-7] + 3 * [5e-7] + 3 * [3e-7] + [3e-8]
    mean = [2e-9] + 3 * [4e-9] + 3 * [3e-8] + [3e-9]
    for c in range(8):
        rms = np.sqrt((b[far, c] ** 2).mean())
        err = np.abs(a[far, c] - b[far, c])
        e, s = err.max() / rms, np.sqrt((err ** 2).mean()) / rms
        print("column %d: max error %.2e, rms error %.2e of rms %.3e" % (c, e, s, rms), flush=True)
        assert e < worst[c]
        if route:
            assert s < mean[c]


# cells whose factors e^{-(kappa r)^2} reach down to 1e-33 and to 1e-8
@pytest.mark.parametrize("edge,spacing,alpha", [(24.0, 0.3, 0.42), (20.0, 0.3, 0.25)])
def test_direct_sums_against_long_double(edge, spacing, alpha):
    xyz, q, L = _box(3, (edge,) * 3, 1)
    ctx = H.Context(0)
    ctx.upload_framework(xyz, np.zeros(len(xyz), dtype=np.int32), q, L, L)
    assert ctx.set_ewald(alpha * edge, 3, 1e10) == 0  # no k vectors: the real-space sum alone
    m = ctx.build_map(H.MH_MAP_EWALD, H.MH_PREC_FP64, spacing, 100.0, keep_full=True)
    n, v = np.array(m.npnts), m.get_full()[1]
    m.close()
    LD = np.longdouble
    pick = np.random.default_rng(2).choice(len(v), 800, replace=False)
    pos = np.stack(np.unravel_index(pick, n, order="F"), 1) * (L / (n - 1))
    a1, a2, a3, a4, a5, p = (LD(np.float32(c)) for c in (0.254829592, -0.284496736, 1.421413741, -1.453152027,
                                                         1.061405429, 0.3275911))
    kappa = LD(alpha * edge / edge)
    d = pos[:, None].astype(LD) - xyz[None].astype(LD)
    d = np.where(d > 0.5 * edge, d - edge, np.where(d < -0.5 * edge, d + edge, d))
    r2 = (d * d).sum(-1)
    x = kappa * np.sqrt(r2)
    t, ek, w = 1 / (1 + p * x), np.exp(-x * x), 1 / r2
    u = q * t * (a1 + t * (a2 + t * (a3 + t * (a4 + t * a5)))) * ek / np.sqrt(r2)
    g = LD(2.0 * 0.5641896) * kappa * q * ek
    f1, f2 = -(u + g) * w, (3 * (u + g) + 2 * x * x * g) * w * w
    f3 = -(15 * (u + g) + (10 + 4 * x * x) * x * x * g) * w ** 3
    X, Y, Z = d[..., 0], d[..., 1], d[..., 2]
    ref = np.stack([s.sum(1) for s in (u, f1 * X, f1 * Y, f1 * Z, f2 * X * Y, f2 * X * Z, f2 * Y * Z,
                                       f3 * X * Y * Z)], 1) * LD(332.064)
    err = np.median((np.abs(v[pick] - ref) / np.abs(ref)).astype(float), 0)
    print("median relative error per column:", err, flush=True)
    # a pair sum with IEEE square root and division leaves 5e-16 (V) to 7.4e-16
    # (third derivative); 5e-15 per pair, one Newton step, leaves 1.1e-15 there
    assert (err < 8.5e-16).all()
