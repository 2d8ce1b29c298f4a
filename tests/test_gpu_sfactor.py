"""Which k vectors the Ewald set-up keeps, where the order of the structure
factor's sum over the atoms could decide it."""
import numpy as np
import pytest

from musichip import hip as H
from oracle import oracle as O

pytestmark = pytest.mark.gpu
L = np.array([11.0, 12.0, 13.0])


def _nk(xyz, q, kappa, kmax, locut):
    ctx = H.Context(0)
    ctx.upload_framework(xyz, np.zeros(len(xyz), dtype=np.int32), q, L, L)
    return ctx.set_ewald(kappa, kmax, locut), O.ewald_sfactor(xyz, q, L, kappa, kmax, locut)["nk"]


def test_extinct_vectors_by_the_reference_order():
    """Triples of charges q, q, -2 q at one place: added in order they cancel
    exactly for every vector, in any other order they leave rounding, which a
    cutoff of zero keeps."""
    rng = np.random.default_rng(3)
    xyz = np.repeat(rng.uniform(0, 1, (70, 3)) * L, 3, axis=0)
    q = (rng.uniform(0.2, 1.0, 70)[:, None] * np.array([1.0, 1.0, -2.0])).reshape(-1)
    assert _nk(xyz, q, 4.0, 4, 0.0) == (0, 0)


def test_kept_vectors_match_the_oracle():
    """Ordinary charges, with cutoffs that drop none, some and most vectors."""
    rng = np.random.default_rng(4)
    xyz = rng.uniform(0, 1, (300, 3)) * L
    q = rng.uniform(-1, 1, 300)
    seen = set()
    for locut in (0.0, 1e-10, 1e-6, 1e-5):
        nk, ref = _nk(xyz, q - q.mean(), 4.0, 5, locut)
        assert nk == ref
        seen.add(nk)
    assert len(seen) > 2
