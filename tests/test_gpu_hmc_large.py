"""Flexible molecules beyond one wave of sites: the force tasks of several
waves (bonded terms of 64 sites, map and pair terms of 16), neighbour lists
longer than the entries loaded ahead, and partial forces in global memory,
against the CPU oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from musichip import hip as H
from musichip import hmc as HM
from musichip import synth

pytestmark = pytest.mark.gpu
L40 = np.array([40.0, 40.0, 40.0])
HICUT = 12.8
NMOL = 70  # 280 sites: five bonded tasks and eighteen of map and pair terms


@pytest.fixture(scope="module")
def system():
    """40 A framework of 768 LJ atoms, device maps (and their host copies),
    70 butanes."""
    rng = np.random.default_rng(71)
    xyz = synth.lattice_faces(4, 10.0, rng)
    eps, sig, typ = synth.fw_types(rng, len(xyz))
    model = synth.butane_ua()
    ctx = H.Context(0)
    ctx.upload_framework(xyz, typ, np.zeros(len(xyz)), L40, L40)
    dev, host = {}, []
    for t, name in enumerate(model["types"]):
        e, s = model["lj"][name]
        ctx.set_lj(*synth.lb_table(eps, sig, e, s, HICUT))
        dev[t] = ctx.build_map(H.MH_MAP_LJ, H.MH_PREC_FP64, 0.4, 100.0)
        host.append((dev[t].npnts, dev[t].step) + dev[t].get())

    def ok(pos):
        good = np.ones(len(pos), dtype=bool)
        for npn, step, ptr, vals in host:
            g, v = O.pothermite(npn, step, ptr, vals, pos, fund_ell=L40)
            good &= g & (v < 0.0)
        return good

    rp = synth.place_chains(model, NMOL, L40, np.random.default_rng(72), ok, min_dist=3.4)
    # partners within the list radius of each site: from 32 on a lane of the
    # quad loads its next four entries while it works on four
    s = rp.reshape(-1, 3)
    d = s[:, None] - s[None]
    d -= L40 * np.rint(d / L40)
    near = ((d * d).sum(-1) < (HICUT + 1.0) ** 2) & (np.arange(len(s))[:, None] // 4 != np.arange(len(s)) // 4)
    assert (near.sum(1) >= 32).mean() > 0.9
    return ctx, model, dev, host, rp


def _spec(model, host, dt, nmd):
    sp = HM.hmc_spec(model, L40, L40, hicut=HICUT, dt=dt, nmd=nmd)
    sp["maps"] = host
    return sp


def test_large_fp64_matches_oracle(system):
    ctx, model, dev, host, rp = system
    sp = _spec(model, host, 0.001, 10)
    b = HM.HmcBatch(ctx, sp, dev, [101], maxN=NMOL, precision=H.MH_PREC_FP64)
    o = O.Hmc(sp, 101)
    b.set_config(0, rp)
    o.set_config(rp)
    eg, Fg, okg = b.energy_forces(0)
    eo, Fo, oko = o.energy_forces()
    assert okg and oko and abs(eg - eo) < 1e-10 * abs(eo)
    assert np.abs(Fg - Fo).max() < 1e-10 * np.abs(Fo).max()
    for mv in range(6):
        b.run(1)
        o.move()
        s = b.state()
        assert (s["att"][0], s["acc"][0], s["fail"][0]) == (o.st.att, o.st.acc, o.st.fail), mv
        assert abs(s["last_dH"][0] - o.st.last_dH) < 1e-8, mv
    assert s["acc"][0] > 1
    prp, pr = b.config(0)
    assert np.abs(prp - o.rp[:NMOL]).max() < 1e-8 and np.abs(pr - o.r[:NMOL]).max() < 1e-8
    b.close()


@pytest.mark.parametrize("prec", [H.MH_PREC_FP64, H.MH_PREC_FP32])
def test_large_md_trace_matches_oracle(system, prec):
    ctx, model, dev, host, rp = system
    sp = _spec(model, host, 0.001, 10)
    v = np.random.default_rng(73).normal(0.0, 3.0, rp.shape)
    b = HM.HmcBatch(ctx, sp, dev, [1], maxN=NMOL, precision=prec)
    b.set_config(0, rp)
    b.set_velocities(0, v)
    tr = b.md(60)
    o = O.Hmc(sp, 1)
    o.set_config(rp)
    done, ref, orp, orr, ov = o.md(v, 60)
    assert done == 60
    # the tolerances of the seven-molecule runs
    tol = np.full(10, 1e-9) if prec == H.MH_PREC_FP64 else np.array([1e-5] * 7 + [1e-4] * 3)
    err = (np.abs(tr[0] - ref) / np.maximum(np.abs(ref), 1.0)).max(axis=0)
    print("largest scaled errors of the trace:", err, flush=True)
    assert np.all(err < tol), err
    if prec == H.MH_PREC_FP64:
        assert np.abs(b.config(0)[0] - orp).max() < 1e-9 and np.abs(b.velocities(0) - ov).max() < 1e-9
    b.close()


def test_large_fp32_move_energies(system):
    """Energies that the FP32 moves carry, against FP64 at the same positions."""
    ctx, model, dev, host, rp = system
    sp = _spec(model, host, 0.001, 10)
    b = HM.HmcBatch(ctx, sp, dev, [5, 6, 7], maxN=NMOL, precision=H.MH_PREC_FP32)
    b64 = HM.HmcBatch(ctx, sp, dev, [5], maxN=NMOL, precision=H.MH_PREC_FP64)
    for r in range(3):
        b.set_config(r, rp)
    b.run(6)
    s = b.state()
    assert (s["acc"] > 0).all()
    for r in range(3):
        b64.set_config(0, b.config(r)[0])
        e, _, ok = b64.energy_forces(0)
        print("FP32 %.6f FP64 %.6f" % (s["energy"][r], e), flush=True)
        assert ok and abs(s["energy"][r] - e) < 1e-6 * abs(e)
    b.close()
    b64.close()


@pytest.mark.parametrize("prec", [H.MH_PREC_FP64, H.MH_PREC_FP32])
def test_partial_forces_in_global_memory(system, prec):
    """320 molecules of room (1280 sites of 128 B exceed a workgroup's LDS):
    the partial forces lie in global memory, with the same sums in the same
    order."""
    ctx, model, dev, host, rp = system
    sp = _spec(model, host, 0.001, 10)
    v = np.random.default_rng(74).normal(0.0, 3.0, rp.shape)
    out = []
    for maxn in (NMOL, 320):
        b = HM.HmcBatch(ctx, sp, dev, [31, 32], maxN=maxn, precision=prec, threads=512)
        for r in range(2):
            b.set_config(r, rp[:NMOL - 3 * r])
        b.run(4)
        s = b.state()
        got = [s[k] for k in ("N", "energy", "att", "acc", "fail", "last_dH", "ix", "iy")]
        for r in range(2):
            b.set_velocities(r, v[:NMOL - 3 * r])
        got.append(b.md(20))
        got += [b.config(r)[0] for r in range(2)] + [b.velocities(r) for r in range(2)]
        out.append(got)
        b.close()
    assert (out[0][3] > 0).all()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
