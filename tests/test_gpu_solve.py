"""GPU nested-FGMRES solve against the oracle (SolveEquation +
GFGMRES restated in oracle/giem2g_oracle.c).

Bar: the FP64 GPU solve matches the oracle solution within 1e-6 relative
(observed ~1e-12) with the same outer iteration and matvec counts; the
mixed-precision solve (complex64 inner, FP64 outer) reaches an FP64 true
residual below the tolerance and matches the FP64 solution within 1e-6.
"""
import numpy as np
import pytest

from tests.conftest import rel

pytestmark = pytest.mark.gpu


def oracle_model(po, m):
    return po.Model(m.csigb(), m.thick, m.omega, m.Nx, m.Ny, m.Nz, m.dx, m.dy, m.z)


@pytest.fixture(scope="module")
def c0_case(oracle):
    from giem2g_amd import models
    m = models.c0()
    om = oracle_model(oracle, m)
    Gs = om.tensor_fft(om.tensor_realspace())
    out = {}
    for pol in (1, 0):  # EY first, then EX (giem2g.F90:346,435)
        E = om.plane_wave(pol)
        Es, info = om.solve(Gs, m.csiga(), E, m_out=30, m_in=30, maxit=100, tol=1e-8)
        out[pol] = (E, Es, info)
    return m, out


def test_fp64_solve_matches_oracle(c0_case):
    from giem2g_amd import operator as gop
    m, ref = c0_case
    op = gop.operator_for(m)
    for pol in (1, 0):
        E, Eo, info = ref[pol]
        assert rel(op.plane_wave(pol), E) < 1e-14
        Es, gi = op.solve(E, outer_m=30, inner_m=30, max_restart=100, tol=1e-8)
        print(pol, gi, info.iterations, info.matvecs, flush=True)
        assert gi["status"] == 1
        assert gi["outer_iterations"] == info.iterations
        assert gi["matvecs_fp64"] == info.matvecs
        assert gi["true_residual"] < 1e-8
        assert rel(Es, Eo) < 1e-6
    op.close()


def test_mixed_precision_solve(c0_case):
    from giem2g_amd import operator as gop
    m, ref = c0_case
    op = gop.operator_for(m)
    E, Eo, _ = ref[1]
    Es, gi = op.solve(E, outer_m=30, inner_m=30, max_restart=100, tol=1e-8, inner_precision=1)
    print(gi, flush=True)
    assert gi["status"] == 1 and gi["true_residual"] < 1e-8
    assert gi["matvecs_fp32"] > 0
    assert rel(Es, Eo) < 1e-6
    op.close()


def test_device_solve_warm_start_and_zero_rhs(c0_case):
    import torch
    from giem2g_amd import operator as gop
    m, ref = c0_case
    op = gop.operator_for(m)
    E, Eo, _ = ref[1]
    Et = torch.from_numpy(E).cuda()
    Es, gi = op.solve(Et, outer_m=30, inner_m=30, max_restart=100, tol=1e-8)
    torch.cuda.synchronize()
    assert rel(Es.cpu().numpy(), Eo) < 1e-6
    # warm start from the solution (ie_solver_module.F90:67-77): converged at once
    Es2, gi2 = op.solve(Et, E0=Es, outer_m=30, inner_m=30, max_restart=100, tol=1e-8)
    assert gi2["outer_iterations"] == 0 and gi2["matvecs_fp64"] == 1
    # zero right-hand side (gmres.F90:140-145)
    Z = torch.zeros_like(Et)
    Ez, gz = op.solve(Z, outer_m=5, inner_m=5, max_restart=3, tol=1e-8)
    assert gz["status"] == 1 and float(Ez.abs().max()) == 0.0
    op.close()


def test_nonconvergence_is_reported(c0_case):
    from giem2g_amd import operator as gop
    m, ref = c0_case
    op = gop.operator_for(m)
    E = ref[1][0]
    Es, gi = op.solve(E, outer_m=1, inner_m=1, max_restart=2, tol=1e-14)
    assert gi["status"] in (-1, 2)
    assert gi["outer_iterations"] == 2
    op.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_paired_polarizations_match_single_solves(prec):
    """giem2g_solve_pair_dev: the EY and EX solves of one frequency with
    paired two-vector operator products give the single solves' fields."""
    import torch
    from giem2g_amd import models, operator as gop
    print("paired precision", prec, flush=True)
    m = models.small(16, 16, 16, seed=31, freq=0.7, dz=20.0)
    op = gop.operator_for(m)
    Ey = torch.from_numpy(op.plane_wave(1)).cuda()
    Ex = torch.from_numpy(op.plane_wave(0)).cuda()
    kw = dict(outer_m=10, inner_m=10, max_restart=50, tol=1e-8, inner_precision=prec)
    sy, iy = op.solve(Ey, **kw)
    sx, ix = op.solve(Ex, **kw)
    py, px, jy, jx, cnt = op.solve_pair(Ey, Ex, **kw)
    print(iy, ix, jy, jx, cnt, flush=True)
    assert jy["status"] == 1 and jx["status"] == 1
    assert jy["true_residual"] < 1e-8 and jx["true_residual"] < 1e-8
    assert rel(py, sy) < 1e-10 and rel(px, sx) < 1e-10
    assert jy["outer_iterations"] == iy["outer_iterations"]
    assert jx["outer_iterations"] == ix["outer_iterations"]
    assert cnt[0] > 0
    op.close()


def test_blocking_waits_give_the_same_solves(monkeypatch):
    """GIEM2G_POLL_MS=0: the solver's host waits block in a stream or event
    synchronisation instead of polling the pinned-host mailbox.  Single and
    paired solves, FP64 and complex64-inner, then give the polled solves'
    iteration counts, the single solves' fields bit for bit (only the wait
    differs) and the paired ones within 1e-12."""
    import torch
    from giem2g_amd import models, operator as gop
    m = models.small(16, 16, 12, seed=41, freq=0.9, dz=25.0)
    op = gop.operator_for(m)
    Ey = torch.from_numpy(op.plane_wave(1)).cuda()
    Ex = torch.from_numpy(op.plane_wave(0)).cuda()
    out = {}
    for mode in ("poll", "block"):
        if mode == "block":
            monkeypatch.setenv("GIEM2G_POLL_MS", "0")
        else:
            monkeypatch.delenv("GIEM2G_POLL_MS", raising=False)
        for prec in (0, 1):
            print(mode, "precision", prec, flush=True)
            kw = dict(outer_m=10, inner_m=10, max_restart=50, tol=1e-8, inner_precision=prec)
            s, i = op.solve(Ey, **kw)
            py, px, jy, jx, cnt = op.solve_pair(Ey, Ex, **kw)
            host = [t.cpu().numpy() if hasattr(t, "cpu") else np.asarray(t) for t in (s, py, px)]
            out[mode, prec] = (host[0], i["outer_iterations"], i["matvecs_fp64"], i["matvecs_fp32"], host[1],
                               host[2], jy["outer_iterations"], jx["outer_iterations"])
    for prec in (0, 1):
        a, b = out["poll", prec], out["block", prec]
        assert a[1:4] == b[1:4] and a[6:] == b[6:], (a[1:4], b[1:4], a[6:], b[6:])
        assert np.array_equal(a[0], b[0])
        assert rel(a[4], b[4]) < 1e-12 and rel(a[5], b[5]) < 1e-12
    op.close()


@pytest.mark.parametrize("prec", [0, 1])
def test_inner_tolerance(prec):
    """inner_tol: the inner solves stop at their own relative residual.
    0 is the default (FP64 inner: the reference's shared tolerance;
    complex64 inner: the relaxed rule, factor 1).  A fixed 1e-2, the shared
    tolerance given explicitly and the relaxed rule with factor 10 all reach
    the FP64 1e-8 true residual and the default solve's field within 1e-6,
    with at most twice the default's matvecs plus one outer cycle; values from 1
    up are rejected."""
    import torch
    from giem2g_amd import lib as L, models, operator as gop
    print("inner tolerance, precision", prec, flush=True)
    m = models.small(16, 16, 12, seed=43, freq=0.5, dz=25.0)
    op = gop.operator_for(m)
    E = torch.from_numpy(op.plane_wave(1)).cuda()
    kw = dict(outer_m=10, inner_m=10, max_restart=50, tol=1e-8, inner_precision=prec)
    s0, i0 = op.solve(E, **kw)
    s1, i1 = op.solve(E, inner_tol=0.0, **kw)
    s0, s1 = s0.cpu().numpy(), s1.cpu().numpy()
    assert np.array_equal(s0, s1) and i0["outer_iterations"] == i1["outer_iterations"]
    mv = lambda i: i["matvecs_fp64"] + i["matvecs_fp32"]
    for itol in (1e-2, 1e-8, -10.0):
        s2, i2 = op.solve(E, inner_tol=itol, **kw)
        print(itol, i0, i2, flush=True)
        assert i2["status"] == 1 and i2["true_residual"] < 1e-8
        assert rel(s2.cpu().numpy(), s0) < 1e-6
        assert mv(i2) <= 2 * mv(i0) + 11
    with pytest.raises(L.G2GError, match="inner_tol"):
        op.solve(E, inner_tol=1.5, **kw)
    op.close()


@pytest.mark.parametrize("Nx,Ny,Nz,m", [(8, 8, 1, 4), (8, 10, 2, 8), (10, 8, 3, 9), (16, 14, 5, 17)])
def test_short_vectors_and_basis_sizes(oracle, Nx, Ny, Nz, m):
    """Gram-Schmidt passes whose vectors fill less than one block or end inside
    one, with bases at the edges of the groups of eight columns: the FP64
    solve against the oracle's (1e-6 and equal counts, as above) and the
    mixed solve's true residual."""
    from giem2g_amd import models, operator as gop
    print("short", Nx, Ny, Nz, m, flush=True)
    md = models.small(Nx, Ny, Nz, seed=Nx + Nz, freq=0.8, dz=20.0)
    om = oracle_model(oracle, md)
    E = om.plane_wave(1)
    Eo, info = om.solve(om.tensor_fft(om.tensor_realspace()), md.csiga(), E, m_out=m, m_in=m, maxit=100, tol=1e-8)
    op = gop.operator_for(md)
    Es, gi = op.solve(E, outer_m=m, inner_m=m, max_restart=100, tol=1e-8)
    assert gi["status"] == 1 and gi["true_residual"] < 1e-8
    assert (gi["outer_iterations"], gi["matvecs_fp64"]) == (info.iterations, info.matvecs)
    assert rel(Es, Eo) < 1e-6
    Em, gm = op.solve(E, outer_m=m, inner_m=m, max_restart=100, tol=1e-8, inner_precision=1)
    assert gm["status"] == 1 and gm["true_residual"] < 1e-8
    assert rel(Em, Eo) < 1e-6
    op.close()
