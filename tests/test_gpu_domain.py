"""Grids beyond powers of two and beyond 64 layers, as the reference accepts
them (any even Nx, Ny: CalcLocalKernelSize, Integral_Equation_Module.F90:
105-129; any Nz), against the oracle.

  - 2Nx- and 2Ny-point transforms that are not powers of two run factor-plan
    Stockham passes (radices 4, 2 and any odd prime: 20 = 4*5, 28 = 4*7,
    44 = 4*11, 52 = 4*13, 68 = 4*17, 48 = 4*4*3, 80 = 4*4*5);
  - more than 64 layers run the tiled vector-ALU contraction (72, 100, 256);
  - the operator apply (FP64 within 1e-12, complex64 within 2e-6) on the
    oracle's spectrum, the GPU tensor and its spectrum, and FP64 and
    mixed-precision solves;
  - the paper's COMMEMI3D-3 lateral grid, 176x224 (352- and 448-point
    transforms), with sampled real-space blocks and an apply on 4 layers;
  - the largest grid side accepted, 512 (1024-point transforms in x and in
    y): tensor, spectrum and apply at 512x16 and 16x512.
"""
import numpy as np
import pytest

from tests.conftest import rel, tensor_block_tol

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    assert torch.cuda.is_available()
    return torch


def oracle_model(po, m):
    return po.Model(m.csigb(), m.thick, m.omega, m.Nx, m.Ny, m.Nz, m.dx, m.dy, m.z)


def rand_vec(n, seed):
    rng = np.random.default_rng(seed)
    return rng.standard_normal(n) + 1j * rng.standard_normal(n)


@pytest.mark.parametrize("Nx,Ny,Nz", [(10, 14, 5), (24, 40, 8), (22, 12, 3), (12, 26, 6), (34, 16, 4),
                                      (8, 8, 72), (12, 10, 100), (16, 8, 256), (512, 16, 4), (16, 512, 4)])
def test_apply_on_oracle_spectrum(oracle, Nx, Ny, Nz):
    torch = _torch()
    from giem2g_amd import models, operator as gop
    print("apply", Nx, Ny, Nz, flush=True)
    m = models.small(Nx, Ny, Nz, seed=Nx + 3 * Ny + Nz, freq=0.8, dz=20.0)
    om = oracle_model(oracle, m)
    Gs = om.tensor_fft(om.tensor_realspace())
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.put_tensor(Gs, spectral=True)
    op.set_sigma(m.csiga())
    v = rand_vec(3 * m.ncell, Nz)
    ref = om.apply(Gs, m.csiga(), v)
    e64 = rel(op.apply_host(v), ref)
    vt = torch.from_numpy(v).cuda().to(torch.complex64)
    o32 = torch.empty_like(vt)
    op.apply_dev_f32(vt, o32)
    op.sync()
    e32 = rel(o32.cpu().numpy().astype(np.complex128), ref)
    print("  FP64 %.2e complex64 %.2e" % (e64, e32), flush=True)
    assert e64 < 1e-12 and e32 < 2e-6
    op.close()


@pytest.mark.parametrize("Nx,Ny,Nz", [(24, 40, 8), (10, 14, 72), (512, 16, 4), (16, 512, 4)])
def test_tensor_and_spectrum(oracle, Nx, Ny, Nz):
    """Layers of 20 m, so that the layer borders meet the background's 1 km
    interface.  A cell that straddles an interface (15 m layers: 990-1005 m)
    is outside what the layered kernel assumes (one background layer per
    cell, the layer of the cell's middle): there the reference's own Fortran
    blocks and the oracle's differ by 2e-2, and so would the GPU's."""
    from giem2g_amd import models, operator as gop
    print("tensor", Nx, Ny, Nz, flush=True)
    m = models.small(Nx, Ny, Nz, seed=5 * Nx + Nz, freq=2.0, dz=20.0)
    om = oracle_model(oracle, m)
    Gr = om.tensor_realspace()
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.tensor_stage(0)
    Gg = op.get_tensor()
    BS = op.block_size
    for lx, ly in [(0, 0), (1, 0), (0, 1), (Nx - 1, Ny - 1), (Nx // 2, 3)]:
        b = lx + Nx * ly
        assert np.linalg.norm(Gg[b * BS:(b + 1) * BS] - Gr[b * BS:(b + 1) * BS]) < tensor_block_tol(om, lx, ly)
    assert rel(Gg, Gr) < 1e-10
    op.tensor_stage(1)
    e = rel(op.get_tensor(), om.tensor_fft(Gg))
    print("  spectrum %.2e" % e, flush=True)
    assert e < 1e-12
    op.close()


@pytest.mark.parametrize("Nx,Ny,Nz", [(20, 12, 6), (12, 10, 72)])
def test_solves(oracle, Nx, Ny, Nz):
    torch = _torch()
    from giem2g_amd import models, operator as gop
    print("solve", Nx, Ny, Nz, flush=True)
    m = models.small(Nx, Ny, Nz, seed=Nx * Ny + Nz, freq=1.0, dz=20.0)
    om = oracle_model(oracle, m)
    Gs = om.tensor_fft(om.tensor_realspace())
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.put_tensor(Gs, spectral=True)
    op.set_sigma(m.csiga())
    Eb = op.plane_wave(1)
    kw = dict(outer_m=15, inner_m=15, max_restart=50, tol=1e-8)
    Eo, oi = om.solve(Gs, m.csiga(), Eb, m_out=15, m_in=15, maxit=50, tol=1e-8)
    E64, i64 = op.solve(Eb, **kw)
    Emx, imx = op.solve(torch.from_numpy(Eb).cuda(), inner_precision=1, **kw)
    e64, emx = rel(E64, Eo), rel(Emx.cpu().numpy(), Eo)
    print("  FP64 %.2e (outer %d / %d), mixed %.2e" % (e64, i64["outer_iterations"], oi.iterations, emx),
          flush=True)
    assert i64["status"] == 1 and imx["status"] == 1 and oi.stat == 1
    assert i64["outer_iterations"] == oi.iterations
    assert e64 < 1e-6 and emx < 1e-6
    op.close()


def test_commemi3d3_lateral_grid(oracle):
    """176 x 224 cells (the paper's scaling model, giem2g.pdf p.10) on 4
    layers: sampled real-space blocks against the oracle's elements, and one
    FP64 apply against the oracle's operator on the GPU's spectrum (the
    352- and 448-point passes)."""
    from giem2g_amd import models, operator as gop
    print("176x224x4", flush=True)
    m = models.small(176, 224, 4, seed=3, freq=1.0, dz=50.0)
    om = oracle_model(oracle, m)
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.tensor_stage(0)
    Gg = op.get_tensor()
    BS = op.block_size
    for lx, ly in [(0, 0), (1, 2), (175, 0), (0, 223), (100, 150), (175, 223)]:
        b = lx + 176 * ly
        blk = om.tensor_element(lx, ly)
        assert np.linalg.norm(Gg[b * BS:(b + 1) * BS] - blk) < tensor_block_tol(om, lx, ly), (lx, ly)
    del Gg
    op.tensor_stage(1)
    Gs = op.get_tensor()
    op.set_sigma(m.csiga())
    v = rand_vec(3 * m.ncell, 17)
    print("  oracle apply", flush=True)
    e = rel(op.apply_host(v), om.apply(Gs, m.csiga(), v))
    print("  apply %.2e" % e, flush=True)
    assert e < 1e-12
    op.close()


@pytest.mark.parametrize("N,Nz", [(8, 1), (8, 3), (12, 9), (22, 17), (34, 6), (64, 33)])
def test_half_tensor_spectrum(oracle, N, Nz):
    """On a square grid with dx = dy a build straight to the spectrum sums the
    offsets lx >= ly only and takes yy and yz from xx and xz with the axes
    exchanged; the two separate stages sum every block.  Tiles of 128 offsets
    and 32 entries with remainders in both.  Bar: the 1e-10 over the tensor
    that the GPU tensor is held to against the oracle's (here the oracle's
    spectrum for the small grids, the stages' for all)."""
    from giem2g_amd import models, operator as gop
    print("half", N, Nz, flush=True)
    m = models.small(N, N, Nz, seed=N + Nz, freq=1.0, dz=20.0)
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.build_tensor()
    Gb = op.get_tensor()
    op.tensor_stage(0)
    op.tensor_stage(1)
    Gs = op.get_tensor()
    e = rel(Gb, Gs)
    print("  build against stages %.2e" % e, flush=True)
    assert e < 1e-10
    if N <= 12:
        om = oracle_model(oracle, m)
        assert rel(Gb, om.tensor_fft(om.tensor_realspace())) < 1e-10
    # the mirror itself: xx(kx,ky) = yy(ky,kx), xz(kx,ky) = yz(ky,kx) to rounding
    P, B = Nz * (Nz + 1) // 2, Gb.reshape(N, N, -1)
    assert np.array_equal(B[:, :, :P], B[:, :, 2 * P:3 * P].transpose(1, 0, 2))
    assert np.array_equal(B[:, :, 4 * P:4 * P + Nz * Nz], B[:, :, 4 * P + Nz * Nz:].transpose(1, 0, 2))
    # no mirror where dx differs from dy
    op.set_geometry(m.dx, 1.5 * m.dy, m.z)
    op.build_tensor()
    Gb = op.get_tensor()
    op.tensor_stage(0)
    op.tensor_stage(1)
    assert np.array_equal(Gb, op.get_tensor())
    op.close()


def half_blocks(G, N, Nz):
    """The real-space blocks whose symmetrically extended, Nyquist-cancelled
    2-D transform is the spectrum G (both [ly][lx][entry]).  The map is
    invertible (condition 1.4 to 16 at N <= 64) once the offsets 0 of odd
    components, which are zero, are left out; on the oracle's spectra the blocks
    come back within 0.2 of tensor_block_tol."""
    def inverse(sg):
        E = np.zeros((N, 2 * N))
        for l in range(N):
            E[l, l] = 1
            if l:
                E[l, 2 * N - l] = sg
        F = np.fft.fft(E, axis=1)
        M = (F[:, :N] - F[:, N:N + 1] * (-1.0) ** np.arange(N)).T
        return np.linalg.inv(M) if sg > 0 else np.vstack([np.zeros(N), np.linalg.pinv(M[:, 1:])])
    inv = {sg: inverse(sg) for sg in (1, -1)}
    P, NN = Nz * (Nz + 1) // 2, Nz * Nz
    B = G.reshape(N, N, -1)
    out = np.empty_like(B)
    for a, b, sx, sy in ((0, P, 1, 1), (P, 2 * P, -1, -1), (2 * P, 4 * P, 1, 1), (4 * P, 4 * P + NN, -1, 1),
                         (4 * P + NN, 4 * P + 2 * NN, 1, -1)):
        out[:, :, a:b] = np.einsum("yk,kxe->yxe", inv[sy], np.einsum("xl,kle->kxe", inv[sx], B[:, :, a:b]))
    return out


@pytest.mark.parametrize("N,Nz", [(12, 9), (34, 6), (64, 2)])
def test_half_tensor_blocks(oracle, N, Nz):
    """The build straight to the spectrum, block by block: its spectrum's
    real-space blocks against the oracle's elements, each within its
    weight-error scale (a bar over the whole tensor does not see the far
    blocks, which are up to 1e7 times smaller than the near ones).  The block
    of an offset lx < ly is the oracle's at (ly,lx) with x and y exchanged: at
    a quarter of the offsets the 1e-12 mask of the weights, which is not
    symmetric in x and y, keeps other taps at (lx,ly) itself (most often one
    more or less), and the element there differs by up to 1.8 times the bar."""
    from giem2g_amd import models, operator as gop
    print("half blocks", N, Nz, flush=True)
    m = models.small(N, N, Nz, seed=N + Nz, freq=1.0, dz=20.0)
    om = oracle_model(oracle, m)
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    op.build_tensor()
    B = half_blocks(op.get_tensor(), N, Nz)
    P, NN = Nz * (Nz + 1) // 2, Nz * Nz
    far = (0, 1, 2, N // 2 - 1, N // 2, N - 2, N - 1)
    worst = 0.0
    for ly in range(N) if N <= 12 else far:
        for lx in range(N) if N <= 12 else far:
            e = om.tensor_element(max(lx, ly), min(lx, ly))
            if lx < ly:  # xx and yy, xz and yz change places
                e = np.concatenate([e[2 * P:3 * P], e[P:2 * P], e[:P], e[3 * P:4 * P], e[4 * P + NN:], e[4 * P:4 * P + NN]])
            d = np.linalg.norm(B[ly, lx] - e) / tensor_block_tol(om, max(lx, ly), min(lx, ly))
            assert d < 1, (lx, ly, d)
            worst = max(worst, d)
    print("  worst block %.2f of its bar" % worst, flush=True)
    op.close()


@pytest.mark.parametrize("Nx,Ny,Nz", [(8, 10, 65), (10, 8, 80), (8, 8, 113), (8, 12, 127), (8, 8, 128), (8, 10, 129),
                                      (8, 8, 136), (8, 8, 185), (10, 8, 255)])
def test_strip_contraction(oracle, Nx, Ny, Nz):
    """The contraction above 64 layers at the edges of its tiles of 16 layers
    and of its strips (16 columns up to 128 layers, 8 above): one apply on a
    random spectrum against the oracle's, FP64 within 1e-12 and complex64
    within 2e-6 (the bars of the applies above), and the same bits twice."""
    torch = _torch()
    from giem2g_amd import models, operator as gop
    print("strips", Nx, Ny, Nz, flush=True)
    m = models.small(Nx, Ny, Nz, seed=Nz, freq=0.8, dz=20.0)
    om = oracle_model(oracle, m)
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    Gs = rand_vec(Nx * Ny * op.block_size, Nz) * (20.0 / np.sqrt(3.0 * Nz))
    op.put_tensor(Gs, spectral=True)
    op.set_sigma(m.csiga())
    v = rand_vec(3 * m.ncell, Nz + 1)
    ref = om.apply(Gs, m.csiga(), v)
    r = op.apply_host(v)
    vt = torch.from_numpy(v).cuda().to(torch.complex64)
    o32 = torch.empty_like(vt)
    op.apply_dev_f32(vt, o32)
    op.sync()
    e64, e32 = rel(r, ref), rel(o32.cpu().numpy().astype(np.complex128), ref)
    print("  FP64 %.2e complex64 %.2e" % (e64, e32), flush=True)
    assert e64 < 1e-12 and e32 < 2e-6
    assert np.array_equal(op.apply_host(v), r)
    op.close()


@pytest.mark.parametrize("p", [3, 5, 7, 11, 13, 17, 31, 37, 47, 61, 83, 97, 127, 251])
def test_prime_lengths(oracle, p):
    """Transforms of 4p points (and 2p-point halves where complex64 takes
    them), alone and beside a length of other radices: registers up to 7, the
    matrix-core stage from 11 (tiles of 16 outputs by 8 butterflies with
    remainders at every prime here).  One apply on a random spectrum and the
    tensor's spectrum against the oracle's, with the bars of the tests above."""
    torch = _torch()
    from giem2g_amd import models, operator as gop
    N = 2 * p if p > 3 else 18
    Nx, Ny, Nz = (N, 12, 3) if p % 4 == 1 else (8, N, 3)
    if p == 31:
        Nx, Ny = 62, 66
    print("prime", p, Nx, Ny, flush=True)
    m = models.small(Nx, Ny, Nz, seed=p, freq=0.8, dz=20.0)
    om = oracle_model(oracle, m)
    op = gop.IEOperator.from_model(m)
    op.set_background(m.csigb(), m.thick, m.omega)
    Gs = rand_vec(Nx * Ny * op.block_size, p) * (20.0 / 3.0)
    op.put_tensor(Gs, spectral=True)
    op.set_sigma(m.csiga())
    v = rand_vec(3 * m.ncell, p + 1)
    ref = om.apply(Gs, m.csiga(), v)
    e64 = rel(op.apply_host(v), ref)
    vt = torch.from_numpy(v).cuda().to(torch.complex64)
    o32 = torch.empty_like(vt)
    op.apply_dev_f32(vt, o32)
    op.sync()
    e32 = rel(o32.cpu().numpy().astype(np.complex128), ref)
    op.put_tensor(Gs, spectral=False)
    op.tensor_stage(1)
    et = rel(op.get_tensor(), om.tensor_fft(Gs))
    print("  FP64 %.2e complex64 %.2e tensor %.2e" % (e64, e32, et), flush=True)
    assert e64 < 1e-12 and e32 < 2e-6 and et < 1e-12
    op.close()
