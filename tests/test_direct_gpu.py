"""GPU parity of the direct Stokes sums against the FP64 oracle.

Tolerances (max-norm relative error over the output):
  FP64 kernels           1e-12
  FP32 Device kernels    2e-5   (the reference's single-precision build)
  f32c (FP32 arithmetic, compensated accumulation, FP64 I/O)
                         5e-6 on vesicle surfaces, 2e-5 on random point clouds
                         (near-coincident random pairs make single terms large,
                         each carrying FP32 rounding)
"""
import numpy as np
import pytest
import torch

import oracle_lib as OL
from ves3d_amd import stokes as K
from ves3d_amd import workloads as W

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(11)


def _cuda(a, dtype=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


def _relerr(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


def _vesicle_case(nv, ss, ts, clustered=False):
    src = RNG.uniform(-1, 1, (nv, 3, ss))
    trg = RNG.uniform(-1, 1, (nv, 3, ts))
    if clustered:
        trg[:, :, : min(ss, ts)] = src[:, :, : min(ss, ts)]  # coincident pairs (r = 0)
    den = RNG.uniform(-1, 1, (nv, 3, ss))
    nrm = RNG.uniform(-1, 1, (nv, 3, ss))
    qw = RNG.uniform(0.1, 1, ss)
    return src, den, nrm, trg, qw


@pytest.mark.parametrize("nv,ss,ts,head,tail", [
    (2, 544, 544, 0, 544), (3, 37, 29, 3, 29), (1, 1, 1, 0, 1), (5, 312, 312, 100, 101),
    (4, 2114, 544, 0, 544)])
@pytest.mark.parametrize("use_qw", [True, False])
def test_direct_stokes_f64(hip, orc, nv, ss, ts, head, tail, use_qw):
    src, den, _, trg, qw = _vesicle_case(nv, ss, ts, clustered=True)
    q = qw if use_qw else None
    ref = np.zeros((nv, 3, ts))
    orc.orc_direct_stokes(OL.ci(ss), OL.ci(ts), OL.ci(nv), OL.ci(head), OL.ci(tail), OL.p(q), OL.p(trg),
                          OL.p(src), OL.p(den), OL.p(ref))
    pot = torch.zeros((nv, 3, ts), dtype=torch.float64, device="cuda")
    K.direct_stokes(_cuda(src), _cuda(den), _cuda(q) if use_qw else None, ss, ts, nv, _cuda(trg),
                    head, tail, pot)
    out = pot.cpu().numpy()
    assert _relerr(out, ref) < 1e-12
    assert np.all(out[:, :, :head] == 0) and np.all(out[:, :, tail:] == 0)


@pytest.mark.parametrize("use_qw", [True, False])
def test_direct_stokes_f32(hip, orc, use_qw):
    nv, ss, ts = 3, 544, 500
    src, den, _, trg, qw = _vesicle_case(nv, ss, ts)
    q = qw if use_qw else None
    ref = np.zeros((nv, 3, ts))
    orc.orc_direct_stokes(OL.ci(ss), OL.ci(ts), OL.ci(nv), OL.ci(0), OL.ci(ts), OL.p(q), OL.p(trg),
                          OL.p(src), OL.p(den), OL.p(ref))
    f = torch.float32
    pot = torch.zeros((nv, 3, ts), dtype=f, device="cuda")
    K.direct_stokes(_cuda(src, f), _cuda(den, f), _cuda(q, f) if use_qw else None, ss, ts, nv,
                    _cuda(trg, f), 0, ts, pot)
    assert _relerr(pot.double().cpu().numpy(), ref) < 2e-5


@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
@pytest.mark.parametrize("use_qw", [True, False])
def test_direct_stokes_dl(hip, orc, dtype, tol, use_qw):
    nv, ss, ts = 3, 544, 531
    src, den, nrm, trg, qw = _vesicle_case(nv, ss, ts)
    q = qw if use_qw else None
    ref = np.zeros((nv, 3, ts))
    orc.orc_direct_stokes_dl(OL.ci(ss), OL.ci(ts), OL.ci(nv), OL.ci(0), OL.ci(ts), OL.p(q), OL.p(trg),
                             OL.p(src), OL.p(nrm), OL.p(den), OL.p(ref))
    pot = torch.zeros((nv, 3, ts), dtype=dtype, device="cuda")
    K.direct_stokes_dl(_cuda(src, dtype), _cuda(nrm, dtype), _cuda(den, dtype),
                       _cuda(q, dtype) if use_qw else None, ss, ts, nv, _cuda(trg, dtype), 0, ts, pot)
    assert _relerr(pot.double().cpu().numpy(), ref) < tol


@pytest.mark.parametrize("dl", [False, True])
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
@pytest.mark.parametrize("nv,ss,ts", [(3, 1, 1), (3, 31, 65), (3, 33, 64), (3, 514, 129),
                                      (4100, 37, 3)])
def test_direct_stokes_edges(hip, orc, nv, ss, ts, dtype, tol, dl):
    """Sources split over 4 and 16 waves with parts of every length down to
    none, runs around 32, and vesicles with coincident points (0), a distance
    whose square is below the normal numbers (1) and one whose square
    overflows (2, both single layer only); tolerances as in the tests above."""
    src, den, nrm, trg, qw = (a.astype(np.float32).astype(np.float64)
                              for a in _vesicle_case(nv, ss, ts))
    n = min(ss, ts)
    trg[0, :, :n] = src[0, :, :n]
    tiny, huge = (1e-160, 1e200) if dtype == torch.float64 else (1e-20, 1e30)
    if not dl:
        src[1, :, ss - 1] = np.float64(np.float32(tiny)) if dtype == torch.float32 else tiny
        trg[1, :, 0] = 0
        trg[2, :, ts - 1] = np.float64(np.float32(huge)) if dtype == torch.float32 else huge
    ref = np.zeros((nv, 3, ts))
    geo = (OL.ci(ss), OL.ci(ts), OL.ci(nv), OL.ci(0), OL.ci(ts), OL.p(qw), OL.p(trg), OL.p(src))
    pot = torch.zeros((nv, 3, ts), dtype=dtype, device="cuda")
    c = lambda a: _cuda(a, dtype)
    if dl:
        orc.orc_direct_stokes_dl(*geo, OL.p(nrm), OL.p(den), OL.p(ref))
        K.direct_stokes_dl(c(src), c(nrm), c(den), c(qw), ss, ts, nv, c(trg), 0, ts, pot)
    else:
        orc.orc_direct_stokes(*geo, OL.p(den), OL.p(ref))
        K.direct_stokes(c(src), c(den), c(qw), ss, ts, nv, c(trg), 0, ts, pot)
    out = pot.double().cpu().numpy()
    assert np.all(np.isfinite(ref))
    # a pair whose r^2 overflows is at least sqrt(largest number) apart and gives
    # at most 2 w |f| / (8 pi r) < 1 / r per component, which the kernel drops
    lost = 0 if dl else ss / float(torch.finfo(dtype).max) ** 0.5
    for v in range(3):
        assert np.max(np.abs(out[v] - ref[v])) <= tol * np.max(np.abs(ref[v])) + lost, v
    assert _relerr(out[3:], ref[3:]) < tol if nv > 3 else True


@pytest.mark.parametrize("dl", [False, True])
@pytest.mark.parametrize("dtype,tol", [(torch.float64, 1e-12), (torch.float32, 2e-5)])
@pytest.mark.parametrize("nv,ss,ts", [(3, 16, 70), (3, 17, 70), (2, 40, 129), (2, 100, 64),
                                      (2, 300, 10), (1100, 65, 3), (2999, 128, 20),
                                      (3000, 128, 20), (3000, 127, 20)])
def test_direct_stokes_forms(hip, orc, nv, ss, ts, dtype, tol, dl):
    """Both sides of the lines between sources staged by one wave and split over
    1, 2, 4, 8 and 16; half of the targets on sources, head and tail inside.
    Tolerances as above; the vesicles at both ends are compared."""
    head, tail = min(2, ts - 1), ts
    src, den, nrm, trg, qw = _vesicle_case(nv, ss, ts)
    n = min(ss, ts) // 2
    trg[:, :, :n] = src[:, :, :n]
    c = lambda a: _cuda(a, dtype)
    pot = torch.full((nv, 3, ts), 7.0, dtype=dtype, device="cuda")
    if dl:
        K.direct_stokes_dl(c(src), c(nrm), c(den), c(qw), ss, ts, nv, c(trg), head, tail, pot)
    else:
        K.direct_stokes(c(src), c(den), c(qw), ss, ts, nv, c(trg), head, tail, pot)
    out = pot.double().cpu().numpy()
    assert np.all(out[:, :, :head] == 7.0) and np.all(np.isfinite(out))
    for v0 in sorted({0, max(0, nv - 40)}):
        m = min(40, nv - v0)
        cut = lambda a: np.ascontiguousarray(a[v0:v0 + m])
        s, d, t, ref = cut(src), cut(den), cut(trg), np.zeros((m, 3, ts))
        geo = (OL.ci(ss), OL.ci(ts), OL.ci(m), OL.ci(head), OL.ci(tail), OL.p(qw), OL.p(t), OL.p(s))
        if dl:
            nn = cut(nrm)
            orc.orc_direct_stokes_dl(*geo, OL.p(nn), OL.p(d), OL.p(ref))
        else:
            orc.orc_direct_stokes(*geo, OL.p(d), OL.p(ref))
        if dtype == torch.float64:
            assert _relerr(out[v0:v0 + m, :, head:], ref[:, :, head:]) < tol
        else:
            # random clouds: a pair at distance r carries the rounding of its two
            # positions, 2 sqrt(3) eps / r, in r^-1 (double layer: r^-2) terms; the
            # closest of the pairs dominates the error as it does the sum
            x = s.transpose(0, 2, 1)[:, None] - t.transpose(0, 2, 1)[:, :, None]
            r = np.linalg.norm(x, axis=3)
            r[r == 0] = np.inf
            terms = (3 / (4 * np.pi) / r ** 2 if dl else 1 / (8 * np.pi) / r)
            bound = 40 * 6e-8 * (terms * (3 + 3.5 / r)).sum(2)[:, None, head:]
            assert np.all(np.abs(out[v0:v0 + m, :, head:] - ref[:, :, head:]) <= bound)


def test_direct_stokes_bad_range(hip):
    src = torch.zeros(3 * 8, dtype=torch.float64, device="cuda")
    pot = torch.zeros(3 * 8, dtype=torch.float64, device="cuda")
    import ves3d_amd
    with pytest.raises(ves3d_amd.Ves3dError) as e:
        K.direct_stokes(src, src, None, 8, 8, 1, src, 5, 9, pot)
    assert e.value.code == 10


@pytest.mark.parametrize("n", [1, 2, 257, 3001])
def test_all2all(hip, orc, n):
    src = RNG.uniform(-3, 3, (n, 3))
    if n > 2:
        src[1] = src[0]  # duplicate point: its pair is skipped (r = 0)
    den = RNG.uniform(-1, 1, (n, 3))
    ref = np.zeros((n, 3))
    orc.orc_stokes_all2all(OL.p(src), OL.p(den), OL.cs(n), OL.p(ref))
    for mixed, tol in ((False, 1e-12), (True, 2e-5)):
        pot = torch.full((n, 3), np.nan, dtype=torch.float64, device="cuda")
        K.stokes_all2all(_cuda(src), _cuda(den), pot, mixed=mixed)
        out = pot.cpu().numpy()
        assert np.all(np.isfinite(out))
        assert _relerr(out, ref) < tol, (mixed, _relerr(out, ref))


def test_all2all_empty(hip):
    z = torch.zeros((0, 3), dtype=torch.float64, device="cuda")
    K.stokes_all2all(z, z, z)


@pytest.mark.parametrize("sl,dl", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("grouped", [False, True])
def test_direct_eval(hip, orc, sl, dl, grouped):
    nv, p = 6, 8
    pos, sld, dld, npv = W.stokes_direct_sum_case(nv=nv, p=p, volfrac=0.1, seed=5)
    ns = pos.shape[0]
    trg = pos.copy()  # targets are the surface points themselves
    spg = npv if grouped else 0
    a_sl = sld if sl else None
    a_dl = dld if dl else None
    ref = np.zeros((ns, 3))
    orc.orc_far_field(OL.p(pos), OL.p(a_sl), OL.p(a_dl), OL.cs(ns), OL.p(trg), OL.p(ref), OL.cs(ns),
                      OL.cs(spg), OL.cs(spg))
    for mixed, tol in ((False, 1e-12), (True, 5e-6)):
        out = torch.zeros((ns, 3), dtype=torch.float64, device="cuda")
        K.direct_eval(_cuda(pos), _cuda(a_sl) if sl else None, _cuda(a_dl) if dl else None, _cuda(trg), out,
                      spg, spg, mixed=mixed)
        e = _relerr(out.cpu().numpy(), ref)
        assert e < tol, (mixed, e)


def test_direct_eval_separate_targets(hip, orc):
    """Targets off the surfaces (n_trg != n_src) with the 128*eps mask."""
    pos, sld, dld, npv = W.stokes_direct_sum_case(nv=4, p=6, volfrac=0.1, seed=9)
    trg = RNG.uniform(pos.min(), pos.max(), (777, 3))
    trg[0] = pos[3]
    ref = np.zeros((777, 3))
    orc.orc_far_field(OL.p(pos), OL.p(sld), OL.p(dld), OL.cs(pos.shape[0]), OL.p(trg), OL.p(ref),
                      OL.cs(777), OL.cs(0), OL.cs(0))
    out = torch.zeros((777, 3), dtype=torch.float64, device="cuda")
    K.direct_eval(_cuda(pos), _cuda(sld), _cuda(dld), _cuda(trg), out)
    assert _relerr(out.cpu().numpy(), ref) < 1e-12


@pytest.mark.parametrize("sl,dl", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("ns,nt,spg", [
    (1, 1, 0), (31, 65, 0), (33, 64, 0), (256, 63, 0), (257, 1, 0), (3001, 700, 0),
    (64, 64, 32), (2 * 257, 2 * 65, 257), (7 * 84, 7 * 40, 84), (1300, 132000, 0)])
def test_direct_eval_split_edges(hip, orc, sl, dl, ns, nt, spg):
    """Around the slices' edges: parts of 32 sources, tiles of 256, waves of
    64 targets that span groups, shared and unshared target waves, a
    coincident point in the last run, and targets with no partner at all.
    FP64 sums of at most 3001 terms in another order: 1e-12 of the largest.
    The mixed form rounds each term to 24 bits: 2e-5 on random clouds."""
    rng = np.random.default_rng(ns + nt)
    pos = rng.uniform(-1, 1, (ns, 3))
    f, q = rng.uniform(-1, 1, (ns, 3)), rng.uniform(-1, 1, (ns, 6))
    trg = rng.uniform(-1, 1, (nt, 3))
    # keep random pairs apart (single terms would dominate the FP32 bound)
    trg += 3.0 * np.sign(trg)
    tpg = nt // (ns // spg) if spg else 0
    if not spg:
        trg[-1] = pos[-1]  # skipped: r = 0
    a_sl, a_dl = (f if sl else None), (q if dl else None)
    pick = np.unique(np.concatenate([np.arange(min(nt, 70)), [nt // 2, nt - 1]]))
    ref = np.zeros((nt, 3))
    if nt < 5000:
        orc.orc_far_field(OL.p(pos), OL.p(a_sl), OL.p(a_dl), OL.cs(ns), OL.p(trg), OL.p(ref),
                          OL.cs(nt), OL.cs(spg), OL.cs(tpg))
        pick = np.arange(nt)
    else:
        sub, rs = np.ascontiguousarray(trg[pick]), np.zeros((pick.size, 3))
        orc.orc_far_field(OL.p(pos), OL.p(a_sl), OL.p(a_dl), OL.cs(ns), OL.p(sub), OL.p(rs),
                          OL.cs(pick.size), OL.cs(0), OL.cs(0))
        ref[pick] = rs
    for mixed, tol in ((False, 1e-12), (True, 2e-5)):
        out = torch.full((nt, 3), np.nan, dtype=torch.float64, device="cuda")
        K.direct_eval(_cuda(pos), _cuda(f) if sl else None, _cuda(q) if dl else None, _cuda(trg),
                      out, spg, tpg, mixed=mixed)
        got = out.cpu().numpy()
        assert np.all(np.isfinite(got))
        assert _relerr(got[pick], ref[pick]) < tol, (mixed, _relerr(got[pick], ref[pick]))


@pytest.mark.parametrize("sl,dl", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("ns,nt,spg", [
    (128, 300, 0), (129, 300, 0), (512, 300, 0), (513, 300, 0), (513, 65535, 0), (513, 65536, 0),
    (700, 19999, 0), (700, 20000, 0), (20 * 64, 20 * 64, 64), (20 * 100, 20 * 77, 100),
    (20 * 101, 20 * 77, 101), (40 * 64, 40 * 60, 64), (26000, 700, 0)])
def test_direct_eval_forms(hip, orc, sl, dl, ns, nt, spg):
    """Both sides of the lines between the mixed form's records and LDS tiles,
    and slices in multiples of the XCDs, as test_direct_eval_split_edges."""
    test_direct_eval_split_edges(hip, orc, sl, dl, ns, nt, spg)


@pytest.mark.parametrize("mixed", [False, True])
@pytest.mark.parametrize("sl,dl", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), 1e300])
def test_direct_eval_own_group_not_read(hip, sl, dl, mixed, bad):
    """A target's own group is no part of its sum, whatever its densities and
    positions hold, in waves that one group fills and in waves that span
    groups: group k's targets get the same bits with any values in group k."""
    rng = np.random.default_rng(3)
    groups, spg, tpg = 5, 84, 90
    pos = _cuda(rng.uniform(-1, 1, (groups, spg, 3)) + 4.0 * np.arange(groups)[:, None, None])
    trg = _cuda(rng.uniform(-1, 1, (groups, tpg, 3)) + 4.0 * np.arange(groups)[:, None, None])
    f, q = _cuda(rng.uniform(-1, 1, (groups, spg, 3))), _cuda(rng.uniform(-1, 1, (groups, spg, 6)))

    def run(x, a, b):
        out = torch.full((groups, tpg, 3), 7.0, dtype=torch.float64, device="cuda")
        K.direct_eval(x, a if sl else None, b if dl else None, trg, out, spg, tpg, mixed=mixed)
        return out

    ref = run(pos, f, q)
    assert bool(torch.isfinite(ref).all())
    for k in range(groups):
        for what in range(3):
            args = [pos.clone(), f.clone(), q.clone()]
            args[what][k, spg // 2] = bad
            if what == 0 and mixed:
                args[0][k, spg // 2, 0] = float("nan")
            assert torch.equal(run(*args)[k], ref[k]), (k, what)


def test_full_size_far_field_properties(hip, orc):
    """512 vesicles at p=16 (278,528 points): f32c vs f64 on every target,
    and f64 vs the oracle on a sample of 96 targets."""
    pos, sld, dld, npv = W.stokes_direct_sum_case(nv=512, p=16)
    n = pos.shape[0]
    gp, gs, gd = _cuda(pos), _cuda(sld), _cuda(dld)
    v64 = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    v32 = torch.zeros((n, 3), dtype=torch.float64, device="cuda")
    K.direct_eval(gp, gs, gd, gp, v64, npv, npv)
    K.direct_eval(gp, gs, gd, gp, v32, npv, npv, mixed=True)
    a64 = v64.cpu().numpy()
    a32 = v32.cpu().numpy()
    rel = np.linalg.norm(a32 - a64) / np.linalg.norm(a64)
    assert rel < 1e-6, rel
    idx = np.sort(RNG.choice(n, 96, replace=False))
    # oracle restricted to the sampled targets: same groups (vesicle = idx // npv)
    ref = np.zeros((96, 3))
    for k, t in enumerate(idx):
        r1 = np.zeros((1, 3))
        orc.orc_far_field(OL.p(pos), OL.p(sld), OL.p(dld), OL.cs(n), OL.p(np.ascontiguousarray(pos[t:t + 1])),
                          OL.p(r1), OL.cs(1), OL.cs(n), OL.cs(0))
        own = slice((t // npv) * npv, (t // npv + 1) * npv)
        r_own = np.zeros((1, 3))
        orc.orc_far_field(OL.p(np.ascontiguousarray(pos[own])), OL.p(np.ascontiguousarray(sld[own])),
                          OL.p(np.ascontiguousarray(dld[own])), OL.cs(npv),
                          OL.p(np.ascontiguousarray(pos[t:t + 1])), OL.p(r_own), OL.cs(1), OL.cs(0), OL.cs(0))
        ref[k] = (r1 - r_own)[0]
    assert _relerr(a64[idx], ref) < 1e-10
