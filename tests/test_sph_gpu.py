"""GPU parity of the SphericalHarmonics transforms, rotations, singular
self-interaction build and self apply against the numpy FP64 oracle.

Tolerances (max-norm error relative to the max of the oracle output):
  FP64 transforms / rotations     1e-12
  FP64 singular operators         1e-9  (the host-built MatRotate differs from the
                                          oracle's by O(1e-8) in entries fed by the
                                          rotated-pole grid point, see test_oracle_sph)
  FP32 transforms                 1e-5
  FP32 singular operators         1e-5 (vs FP64 oracle)
"""
import numpy as np
import pytest
import torch

from oracle import sph as O
from oracle import ves
from ves3d_amd import sph as G
from ves3d_amd import workloads as W

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(21)


def cu(a, dt=torch.float64):
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dt)


def rel(a, b):
    return float(np.max(np.abs(a - b)) / max(np.max(np.abs(b)), 1e-300))


@pytest.mark.parametrize("p0,p1,N", [(6, 6, 5), (8, 16, 3), (12, 12, 7), (16, 32, 11), (16, 16, 1)])
@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_shc2grid(hip, p0, p1, N, dt, tol):
    S = RNG.standard_normal((N, O.ncoef(p0) if hasattr(O, "ncoef") else p0 * (p0 + 2)))
    X, Xt, Xp = O.shc2grid(S, p0, p1, True, True)
    g = lambda: torch.zeros((N, 2 * p1 * (p1 + 1)), dtype=dt, device="cuda")
    gx, gt, gp = g(), g(), g()
    G.shc2grid(cu(S, dt), N, p0, p1, gx, gt, gp)
    assert rel(gx.double().cpu().numpy(), X) < tol
    assert rel(gt.double().cpu().numpy(), Xt) < tol
    assert rel(gp.double().cpu().numpy(), Xp) < tol
    gx2 = g()
    G.shc2grid(cu(S, dt), N, p0, p1, gx2)  # no derivative outputs
    assert rel(gx2.double().cpu().numpy(), X) < tol


@pytest.mark.parametrize("p0,p1,N", [(6, 6, 5), (16, 8, 3), (12, 12, 7), (32, 16, 13), (24, 24, 2)])
@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_grid2shc_and_transpose(hip, p0, p1, N, dt, tol):
    X = RNG.standard_normal((N, 2 * p0 * (p0 + 1)))
    S = O.grid2shc(X, p0, p1)
    T = O.shc2grid_transpose(X, p0, p1)
    gs = torch.zeros((N, p1 * (p1 + 2)), dtype=dt, device="cuda")
    G.grid2shc(cu(X, dt), N, p0, p1, gs)
    assert rel(gs.double().cpu().numpy(), S) < tol
    G.shc2grid_transpose(cu(X, dt), N, p0, p1, gs)
    assert rel(gs.double().cpu().numpy(), T) < tol


@pytest.mark.parametrize("p0,p1,N", [(1, 1, 1), (2, 5, 3), (8, 8, 4), (9, 17, 1027), (16, 32, 683),
                                     (17, 3, 130), (24, 25, 1), (25, 24, 513), (32, 33, 2),
                                     (32, 32, 1365), (33, 12, 3), (12, 6, 16383),
                                     (12, 6, 16384), (6, 11, 6143), (6, 11, 6144), (6, 12, 12287),
                                     (6, 12, 12288)])
@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_one_kernel_transforms(hip, p0, p1, N, dt, tol):
    """The one-kernel transforms against the grouped GEMMs (which a forced tile
    selects) at the edges of their rules: padded and whole tiles of columns and
    rows, every functions-per-workgroup, partial last groups, and the orders
    and sizes on both sides of the line to the GEMMs."""
    from ves3d_amd import call
    S = torch.from_numpy(RNG.standard_normal((N, p0 * (p0 + 2)))).to("cuda", dt)
    X = torch.from_numpy(RNG.standard_normal((N, 2 * p0 * (p0 + 1)))).to("cuda", dt)
    grid = lambda: torch.zeros((N, 2 * p1 * (p1 + 1)), dtype=dt, device="cuda")
    out = {}
    try:
        for tile in (-1, 0):
            call("ves3d_hip_set_gemm_tile", tile)
            synth, a, t = [grid() for _ in range(4)], *(
                torch.zeros((N, p1 * (p1 + 2)), dtype=dt, device="cuda") for _ in range(2))
            G.shc2grid(S, N, p0, p1, *synth[:3])
            G.shc2grid(S, N, p0, p1, synth[3])
            G.grid2shc(X, N, p0, p1, a)
            G.shc2grid_transpose(X, N, p0, p1, t)
            torch.cuda.synchronize()
            out[tile] = [x.double() for x in synth + [a, t]]
    finally:
        call("ves3d_hip_set_gemm_tile", -1)
    # each output to its own size; but the longitude derivative of order 1 at 0 and
    # pi is zero up to the table's rounding of sin pi, and is held to a hundredth of
    # the values, whose sums it shares
    values = float(out[0][3].abs().max())
    for k, (x, y) in enumerate(zip(out[-1], out[0])):
        err = float((x - y).abs().max()) / max(float(y.abs().max()), 0.01 * values if k == 1 else 0)
        assert err < tol, (k, err)


@pytest.mark.parametrize("p0,p1,N", [(6, 6, 700), (8, 16, 300), (16, 32, 90), (24, 12, 200)])
@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_transforms_over_their_input(hip, p0, p1, N, dt, tol):
    """Outputs that lie over the input, at its start and beside it: a transform
    has read its input before it writes (every value; with derivatives only the
    last output, the latitude derivative, may lie over the coefficients)."""
    nc, ng = lambda p: p * (p + 2), lambda p: 2 * p * (p + 1)
    S = torch.from_numpy(RNG.standard_normal((N, nc(p0)))).to("cuda", dt)
    grid = lambda: torch.zeros((N, ng(p1)), dtype=dt, device="cuda")
    X, Xt, Xp = grid(), grid(), grid()
    G.shc2grid(S, N, p0, p1, X, Xt, Xp)
    A, T = (torch.zeros((N, nc(p0)), dtype=dt, device="cuda") for _ in range(2))
    G.grid2shc(Xt, N, p1, p0, A)
    G.shc2grid_transpose(Xt, N, p1, p0, T)
    err = lambda a, b: float((a - b).abs().max() / b.abs().max())
    for shift in (0, 7, N * nc(p0) // 2):
        def over(src, n_out):
            buf = torch.zeros(src.numel() + n_out + 2 * shift, dtype=dt, device="cuda")
            i = buf[shift:shift + src.numel()]
            i.copy_(src.reshape(-1))
            return i, buf[2 * shift:2 * shift + n_out]
        i, o = over(S, N * ng(p1))
        G.shc2grid(i, N, p0, p1, o)
        assert err(o.reshape(N, -1), X) < tol
        i, o = over(S, N * ng(p1))
        t, x = grid(), grid()
        G.shc2grid(i, N, p0, p1, x, t, o)
        assert err(o.reshape(N, -1), Xp) < tol and err(x, X) < tol and err(t, Xt) < tol
        for fn, ref in ((G.grid2shc, A), (G.shc2grid_transpose, T)):
            i, o = over(Xt, N * nc(p0))
            fn(i, N, p1, p0, o)
            assert err(o.reshape(N, -1), ref) < tol


@pytest.mark.parametrize("p0,p1,N", [
    (4, 4, 4095), (4, 4, 4096), (12, 12, 6143), (12, 12, 6144), (30, 20, 2047), (30, 20, 2048),
    (32, 32, 1279), (32, 32, 1280), (32, 32, 3071), (32, 32, 3072), (24, 12, 6143),
    (24, 12, 6144), (3, 3, 10239), (3, 3, 10240), (8, 8, 24575), (8, 8, 24576), (6, 3, 12287),
    (6, 3, 12288), (32, 32, 20480)])
@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-12), (torch.float32, 1e-5)])
def test_transform_lines_to_gemms(hip, p0, p1, N, dt, tol):
    """Both sides of the lines between the one-kernel transforms and the GEMMs,
    as test_one_kernel_transforms, and the value with its longitude derivative,
    which has a line of its own."""
    from ves3d_amd import call
    test_one_kernel_transforms(hip, p0, p1, N, dt, tol)
    S = torch.from_numpy(RNG.standard_normal((N, p0 * (p0 + 2)))).to("cuda", dt)
    out = {}
    try:
        for tile in (-1, 0):
            call("ves3d_hip_set_gemm_tile", tile)
            out[tile] = [torch.zeros((N, 2 * p1 * (p1 + 1)), dtype=dt, device="cuda")
                         for _ in range(2)]
            G.shc2grid(S, N, p0, p1, *out[tile])
            torch.cuda.synchronize()
    finally:
        call("ves3d_hip_set_gemm_tile", -1)
    for x, y in zip(out[-1], out[0]):
        assert float((x - y).abs().max() / y.abs().max()) < tol


@pytest.mark.parametrize("p,N", [(6, 4), (16, 9)])
def test_shc2pole(hip, p, N):
    S = RNG.standard_normal((N, p * (p + 2)))
    P = O.shc2pole(S, p)
    gp = torch.zeros((N, 2), dtype=torch.float64, device="cuda")
    G.shc2pole(cu(S), N, p, gp)
    assert rel(gp.cpu().numpy(), P) < 1e-13


@pytest.mark.parametrize("p,N,dof", [(6, 2, 3), (8, 1, 12), (16, 2, 3), (32, 1, 1)])
def test_rotations(hip, p, N, dof):
    """RotateAll / RotateTranspose against the oracle; p = 32 in FP64 takes
    the scatter kernel's unstaged path (four rows exceed its LDS staging)."""
    nc = p * (p + 2)
    S = RNG.standard_normal((N * dof, nc))
    R = O.rotate_all(S, p, dof)
    out = torch.zeros(R.size, dtype=torch.float64, device="cuda")
    G.rotate_all(cu(S), N, p, dof, out)
    # rotation matrices are rebuilt on the host; entries fed by the rotated-pole
    # grid point carry O(1e-8) rounding noise in both (see test_oracle_sph)
    assert rel(out.cpu().numpy().reshape(R.shape), R) < 1e-7
    Y = RNG.standard_normal(R.shape)
    T = O.rotate_transpose(Y, p, dof)
    out2 = torch.zeros(R.size, dtype=torch.float64, device="cuda")
    G.rotate_transpose(cu(Y), N, p, dof, out2)
    assert rel(out2.cpu().numpy().reshape(T.shape), T) < 1e-7


def _singular_case(nv, p0, seed):
    return W.perturbed_shapes(nv, p0, amp=0.1, seed=seed)


@pytest.mark.parametrize("nv,p0,p1", [(3, 6, 12), (2, 8, 16), (1, 12, 24)])
def test_singular_build_f64(hip, nv, p0, p1):
    X = _singular_case(nv, p0, seed=nv + p0)
    SL, DL = O.stokes_singular_integ(X, p0, p1)
    n = 3 * p0 * (p0 + 2)
    gsl = torch.zeros((nv, n, n), dtype=torch.float64, device="cuda")
    gdl = torch.zeros((nv, n, n), dtype=torch.float64, device="cuda")
    G.singular_build(cu(X), nv, p0, p1, gsl, gdl)
    e1 = rel(gsl.cpu().numpy(), SL)
    e2 = rel(gdl.cpu().numpy(), DL)
    assert e1 < 1e-9 and e2 < 1e-9, (e1, e2)
    # SL only
    g2 = torch.zeros_like(gsl)
    G.singular_build(cu(X), nv, p0, p1, g2, None)
    assert rel(g2.cpu().numpy(), SL) < 1e-9


def test_singular_build_f32(hip):
    nv, p0, p1 = 2, 8, 16
    X = _singular_case(nv, p0, seed=5)
    SL, DL = O.stokes_singular_integ(X, p0, p1)
    n = 3 * p0 * (p0 + 2)
    gsl = torch.zeros((nv, n, n), dtype=torch.float32, device="cuda")
    gdl = torch.zeros((nv, n, n), dtype=torch.float32, device="cuda")
    G.singular_build(cu(X), nv, p0, p1, gsl, gdl)
    assert rel(gsl.double().cpu().numpy(), SL) < 1e-5
    assert rel(gdl.double().cpu().numpy(), DL) < 1e-5


@pytest.mark.parametrize("p0", [12, 16, 24])
def test_singular_closed_forms_gpu(hip, p0):
    """Size-independent property at the workload's order: on unit spheres
    SL[c] = (2/3) c, DL[c] = -c/2 (the grid's outward normal, the
    reference orientation), SL[n] = 0 (p1 = 2 p0)."""
    nv = 2
    Xs, _ = W.sphere_grid(p0)
    X = np.stack([Xs, Xs * 1.0])
    n = 3 * p0 * (p0 + 2)
    nc = p0 * (p0 + 2)
    gsl = torch.zeros((nv, n, n), dtype=torch.float64, device="cuda")
    gdl = torch.zeros((nv, n, n), dtype=torch.float64, device="cuda")
    G.singular_build(cu(X), nv, p0, 2 * p0, gsl, gdl)
    c = np.array([0.3, -1.1, 0.7])
    f = np.repeat(c, Xs.shape[1]).reshape(3, -1)
    F = O.grid2shc(f, p0, p0).reshape(-1)
    Fn = O.grid2shc(Xs, p0, p0).reshape(-1)
    for v in range(nv):
        SLv = gsl[v].cpu().numpy()
        DLv = gdl[v].cpu().numpy()
        V = O.shc2grid((F @ SLv).reshape(3, nc), p0, p0)
        Vd = O.shc2grid((F @ DLv).reshape(3, nc), p0, p0)
        Vn = O.shc2grid((Fn @ SLv).reshape(3, nc), p0, p0)
        assert np.max(np.abs(V - 2.0 / 3.0 * f)) < 1e-9
        assert np.max(np.abs(Vd + 0.5 * f)) < 1e-9
        assert np.max(np.abs(Vn)) < 1e-9


@pytest.mark.parametrize("p0,p1,nv", [(6, 12, 5), (8, 16, 3), (12, 24, 2), (16, 32, 2), (24, 48, 1)])
def test_singular_build_f32_transforms(hip, p0, p1, nv):
    """The FP32 build's transforms are the grouped GEMMs (which a forced tile
    selects), whose sums do not depend on the tile: the same bits."""
    from ves3d_amd import call
    X = cu(_singular_case(nv, p0, seed=p0))
    n = 3 * p0 * (p0 + 2)
    out = {}
    try:
        for tile in (-1, 0):
            call("ves3d_hip_set_gemm_tile", tile)
            out[tile] = [torch.zeros((nv, n, n), device="cuda") for _ in range(2)]
            G.singular_build(X, nv, p0, p1, *out[tile])
            torch.cuda.synchronize()
    finally:
        call("ves3d_hip_set_gemm_tile", -1)
    for a, b in zip(out[-1], out[0]):
        assert torch.equal(a, b)


@pytest.mark.parametrize("p0,sl_tol", [(16, 5e-8), (24, 1e-8)])
def test_singular_identities_on_ellipsoids_gpu(hip, p0, sl_tol):
    """Shape-sensitive identities at the workloads' orders, on two rotated
    ellipsoids (semi-axes 1, 1, 0.6 +- 0.05), where a target rotated to the
    wrong pole would break them: DL[c] = -c/2 on the surface and SL[n] = 0
    (n truncated at p0, whose error decays with p0), p1 = 2 p0, for the
    FP64 build and, to the FP32 build's accuracy, the FP32 one."""
    nv = 2
    X = W.implicit_step_case(nv, p0, 0.2, seed=9)
    X = X - X.mean(axis=2, keepdims=True)
    n = 3 * p0 * (p0 + 2)
    nc = p0 * (p0 + 2)
    c = np.array([0.3, -1.1, 0.7])
    f = np.repeat(c, X.shape[2]).reshape(3, -1)
    F = O.grid2shc(f, p0, p0).reshape(-1)
    nrm = ves.Surface(X, p0).normal
    for dt, dl_tol, sl_bar in ((torch.float64, 1e-9, sl_tol), (torch.float32, 1e-4, 1e-4)):
        print("singular identities p0=%d %s" % (p0, dt), flush=True)
        gsl = torch.zeros((nv, n, n), dtype=dt, device="cuda")
        gdl = torch.zeros((nv, n, n), dtype=dt, device="cuda")
        G.singular_build(cu(X), nv, p0, 2 * p0, gsl, gdl)
        for v in range(nv):
            SLv = gsl[v].double().cpu().numpy()
            DLv = gdl[v].double().cpu().numpy()
            Vd = O.shc2grid((F @ DLv).reshape(3, nc), p0, p0)
            Fn = O.grid2shc(nrm[v], p0, p0).reshape(-1)
            Vn = O.shc2grid((Fn @ SLv).reshape(3, nc), p0, p0)
            assert np.max(np.abs(Vd + 0.5 * f)) < dl_tol, (dt, v)
            assert np.max(np.abs(Vn)) < sl_bar, (dt, v)
        del gsl, gdl


@pytest.mark.parametrize("dt,tol", [(torch.float64, 1e-13), (torch.float32, 1e-6)])
def test_self_apply(hip, dt, tol):
    nv, p = 5, 8
    n = 3 * p * (p + 2)
    SL = RNG.standard_normal((nv, n, n))
    DL = RNG.standard_normal((nv, n, n))
    F = RNG.standard_normal((nv, n))
    Gd = RNG.standard_normal((nv, n))
    ref = np.einsum("vr,vrc->vc", F, SL) + np.einsum("vr,vrc->vc", Gd, DL)
    V = torch.zeros((nv, n), dtype=torch.float64, device="cuda")
    G.self_apply(cu(SL, dt), cu(F), cu(DL, dt), cu(Gd), nv, p, V)
    assert rel(V.cpu().numpy(), ref) < tol
    ref1 = np.einsum("vr,vrc->vc", F, SL)
    G.self_apply(cu(SL, dt), cu(F), None, None, nv, p, V)
    assert rel(V.cpu().numpy(), ref1) < tol


@pytest.mark.parametrize("p0,p1,nv", [(6, 12, 1), (7, 14, 2), (9, 18, 5), (10, 20, 2), (12, 24, 9),
                                      (13, 26, 2), (15, 30, 4), (5, 12, 2), (3, 32, 2), (16, 32, 3)])
def test_pole_kernel_orders(hip, p0, p1, nv):
    """The fused pole kernel's instances against the separate kernels: orders
    whose longitudes and columns fill the matrix tiles in part, odd orders,
    upsampled orders above 2 p0, and fewer and more rotations (nv p0 (p0 + 1))
    than persistent workgroups.  Both sum the same products in FP64: 1e-12 as
    test_singular_build_fused_pole_stage."""
    from ves3d_amd import call
    X = cu(_singular_case(nv, p0, seed=p0 + p1))
    n = 3 * p0 * (p0 + 2)
    out = {}
    try:
        for fused in (1, 0):
            call("ves3d_hip_set_pole_kernel", fused)
            sl, dl = (torch.zeros((nv, n, n), dtype=torch.float64, device="cuda") for _ in range(2))
            G.singular_build(X, nv, p0, p1, sl, dl)
            torch.cuda.synchronize()
            out[fused] = sl.cpu().numpy(), dl.cpu().numpy()
    finally:
        call("ves3d_hip_set_pole_kernel", 1)
    assert rel(out[1][0], out[0][0]) < 1e-12 and rel(out[1][1], out[0][1]) < 1e-12


@pytest.mark.parametrize("p,nv", [(1, 1), (2, 3), (4, 70), (12, 2), (12, 330), (16, 5)])
@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_self_apply_rows_split(hip, p, nv, dt):
    """Rows split over 16 waves with parts down to none, partial and whole blocks
    of columns, one layer and both, and the sizes of the unsplit kernel (order
    12, 330 vesicles).  The matrices' entries are taken as they are and summed
    in FP64: n = 6 Ncoef products, n eps of the sum of their sizes."""
    n = 3 * p * (p + 2)
    g = torch.Generator(device="cuda").manual_seed(p + nv)
    M, D = (torch.randn((nv, n, n), dtype=dt, device="cuda", generator=g) for _ in range(2))
    F, H = (torch.randn((nv, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    for both in (False, True):
        V = torch.full((nv, n), 7.0, dtype=torch.float64, device="cuda")
        G.self_apply(M, F, D if both else None, H if both else None, nv, p, V)
        size = torch.zeros_like(V)
        ref = torch.zeros_like(V)
        for A, x in ((M, F),) + (((D, H),) if both else ()):
            for v in range(nv):
                ref[v] += x[v] @ A[v].double()
                size[v] += x[v].abs() @ A[v].double().abs()
        assert bool(((V - ref).abs() <= 2 * n * 2.3e-16 * size).all())


@pytest.mark.parametrize("dt,p,nv", [
    (torch.float64, 4, 767), (torch.float64, 4, 768), (torch.float64, 7, 511),
    (torch.float64, 7, 512), (torch.float64, 8, 683), (torch.float32, 4, 1023),
    (torch.float32, 4, 1024), (torch.float32, 9, 511), (torch.float32, 9, 512),
    (torch.float32, 13, 512)])
def test_self_apply_many_vesicles(hip, dt, p, nv):
    """Both sides of the line between a thread per column and split rows: 2 n eps
    of the sum of the products' sizes, as above."""
    n = 3 * p * (p + 2)
    g = torch.Generator(device="cuda").manual_seed(p + nv)
    M, D = (torch.randn((nv, n, n), dtype=dt, device="cuda", generator=g) for _ in range(2))
    F, H = (torch.randn((nv, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    V = torch.full((nv, n), 7.0, dtype=torch.float64, device="cuda")
    G.self_apply(M, F, D, H, nv, p, V)
    size, ref = torch.zeros_like(V), torch.zeros_like(V)
    for A, x in ((M, F), (D, H)):
        for v in range(nv):
            ref[v] += x[v] @ A[v].double()
            size[v] += x[v].abs() @ A[v].double().abs()
    assert bool(((V - ref).abs() <= 2 * n * 2.3e-16 * size).all())


@pytest.mark.parametrize("p,nv", [(3, 3), (4, 200), (5, 70), (7, 40), (8, 3), (8, 600)])
@pytest.mark.parametrize("dt", [torch.float64, torch.float32])
def test_self_apply_in_place(hip, p, nv, dt):
    """Up to order 8 a vesicle's coefficients are read before any of its results
    is written, so V may be F or G itself.  The sums of the call with a V of its
    own in any order: 2 n eps of the sum of their sizes, as above."""
    n = 3 * p * (p + 2)
    g = torch.Generator(device="cuda").manual_seed(p + nv)
    M, D = (torch.randn((nv, n, n), dtype=dt, device="cuda", generator=g) for _ in range(2))
    F, H = (torch.randn((nv, n), dtype=torch.float64, device="cuda", generator=g) for _ in range(2))
    for both, over in ((False, 0), (True, 0), (True, 1)):
        V = torch.zeros_like(F)
        G.self_apply(M, F, D if both else None, H if both else None, nv, p, V)
        size = torch.bmm(F.abs()[:, None], M.double().abs())[:, 0]
        if both:
            size += torch.bmm(H.abs()[:, None], D.double().abs())[:, 0]
        f, h = F.clone(), H.clone()
        G.self_apply(M, f, D if both else None, h if both else None, nv, p, h if over else f)
        assert bool((((h if over else f) - V).abs() <= 2 * n * 2.3e-16 * size).all())


@pytest.mark.parametrize("p0", [16, 8])
def test_singular_build_fused_pole_stage(hip, p0):
    """The FP64 build's fused pole kernel, transposed synthesis and rotation (the
    default where p1 is even, 12 to 32 and at least 2 p0) against the separate
    kernels, SL and DL.  Asserts that the fused stage applies on this device."""
    import ctypes
    from ves3d_amd import call
    nv, p1, dt, tol = 3, 2 * p0, torch.float64, 1e-12
    rows, threads, groups = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_int(0)
    call("ves3d_hip_pole_kernel_shape", p0, p1, ctypes.byref(rows), ctypes.byref(threads),
         ctypes.byref(groups))
    print("fused pole stage p0=%d: %d rows per pass, %d threads, %d workgroups"
          % (p0, rows.value, threads.value, groups.value), flush=True)
    # a latitude and its mirror per pass, two such pairs up to 16 longitudes
    assert rows.value == (4 if p1 <= 16 else 2) and threads.value == 256 and groups.value >= 1
    X = _singular_case(nv, p0, seed=41)
    n = 3 * p0 * (p0 + 2)
    out = {}
    try:
        for fused in (1, 0):
            call("ves3d_hip_set_pole_kernel", fused)
            sl = torch.zeros((nv, n, n), dtype=dt, device="cuda")
            dl = torch.zeros((nv, n, n), dtype=dt, device="cuda")
            G.singular_build(cu(X), nv, p0, p1, sl, dl)
            torch.cuda.synchronize()
            out[fused] = (sl.double().cpu().numpy(), dl.double().cpu().numpy())
    finally:
        call("ves3d_hip_set_pole_kernel", 1)
    e_sl, e_dl = rel(out[1][0], out[0][0]), rel(out[1][1], out[0][1])
    print("fused vs separate pole stage (p0=%d): SL %.2e, DL %.2e" % (p0, e_sl, e_dl), flush=True)
    assert e_sl < tol and e_dl < tol


@pytest.mark.parametrize("p0,fused,dt", [(16, 1, torch.float64), (16, 0, torch.float64),
                                         (12, 1, torch.float64), (16, 1, torch.float32)])
def test_singular_operator_block_symmetry(hip, p0, fused, dt):
    """The built SL and DL operators' 3 x 3 blocks of Ncoef x Ncoef satisfy
    B_ab = B_ba exactly (block (a, b) holds the rows of the symmetric tensor
    component c(a, b)), which the step's self apply relies on to read only
    the blocks a <= b.  Fused FP64 build (two instances), separate FP64 build,
    and the FP32 build."""
    from ves3d_amd import call
    nv = 2
    nc = p0 * (p0 + 2)
    X = _singular_case(nv, p0, seed=43)
    try:
        call("ves3d_hip_set_pole_kernel", fused)
        sl = torch.zeros((nv, 3 * nc, 3 * nc), dtype=dt, device="cuda")
        dl = torch.zeros((nv, 3 * nc, 3 * nc), dtype=dt, device="cuda")
        G.singular_build(cu(X), nv, p0, 2 * p0, sl, dl)
        torch.cuda.synchronize()
    finally:
        call("ves3d_hip_set_pole_kernel", 1)
    for M in (sl.cpu().numpy(), dl.cpu().numpy()):
        assert np.max(np.abs(M)) > 0
        for a in range(3):
            for b in range(a + 1, 3):
                B_ab = M[:, a * nc:(a + 1) * nc, b * nc:(b + 1) * nc]
                B_ba = M[:, b * nc:(b + 1) * nc, a * nc:(a + 1) * nc]
                assert np.array_equal(B_ab, B_ba), (a, b)
