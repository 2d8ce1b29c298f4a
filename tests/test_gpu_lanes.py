"""Lanes of a GCMC chain chosen at creation (the timer names tell them): FP32
chains of one species beyond one a CU run with 128 where two of them share a
CU, everything else with 256, and a caller's choice stands."""
import numpy as np
import pytest

from musichip import hip as H
from musichip import gcmc as G
from musichip import synth
from test_gpu_gcmc import _cell, _spec007

pytestmark = pytest.mark.gpu


def _co2(kmax):
    m = synth.co2_like()
    A, B = [], []
    for t in ("O", "C"):
        for u in ("O", "C"):
            (e1, s1), (e2, s2) = m["lj"][t], m["lj"][u]
            a, b = synth.lj_AB((s1 + s2) / 2, np.sqrt(e1 * e2))
            A.append(float(a))
            B.append(float(b))
    return dict(full_ell=[20.0] * 3, fund_ell=[20.0] * 3, ref=m["ref"], stype=[0, 1, 0], sq=m["q"], nst=2,
                lj=(A, B, [81.0] * 4, [0.25] * 4, [1] * 4), T=300.0, ewald=dict(kappa=0.3, kmax=kmax, rc=9.0),
                dtrans=0.4, drot=0.4,
                moves=[("RINSERT", 1.0), ("RDELETE", 1.0), ("RTRANSLATE", 1.0), ("RROTATE", 1.0)])


def _biased():
    return dict(_spec007(), moves=[("BINSERT", 1.0), ("BDELETE", 1.0), ("RTRANSLATE", 1.0)])


FP32, FP64 = H.MH_PREC_FP32, H.MH_PREC_FP64


@pytest.mark.parametrize("name,chains,maxn,prec,want", [
    ("methane", 257, 256, FP32, 128),
    ("methane", 256, 256, FP32, 256),
    ("methane", 300, 256, FP64, 256),
    # one chain's molecules take more than half of a CU's LDS
    ("methane", 300, 1100, FP32, 256),
    ("mixture", 300, 64, FP32, 256),
    ("cavity", 300, 256, FP32, 256),
    ("co2", 385, 256, FP32, 128),
    ("co2", 384, 256, FP32, 256),
    # 3429 k vectors fit the registers of 256 lanes, not of 128
    ("co2_k9", 400, 256, FP32, 256),
])
def test_lanes_chosen_at_creation(name, chains, maxn, prec, want):
    ctx = H.Context(0)
    _cell(ctx, [20.0] * 3)
    seeds = list(range(3, 3 + chains))
    if name == "mixture":
        b = G.GcmcMix(ctx, [_spec007()] * 2, [[3.0e4, 3.0e4]] * chains, seeds, maxN=maxn, precision=prec)
    else:
        spec = {"methane": _spec007, "cavity": _biased, "co2": lambda: _co2(6), "co2_k9": lambda: _co2(9)}[name]()
        b = G.GcmcBatch(ctx, spec, [3.0e4] * chains, seeds, maxN=maxn, precision=prec)
    if name == "cavity":
        b.set_cavity((10, 10, 10), [8], [0], tab=None, species_mask=1)

    def lanes():
        ctx.set_timing(True)
        b.run(20)
        t = ctx.timings()
        ctx.set_timing(False)
        return [k for k in t if k.startswith("gcmc_lanes")]

    assert lanes() == ["gcmc_lanes%d" % want]
    b.set_threads(512)
    assert lanes() == ["gcmc_lanes512"]
