"""Workloads of the integral-equation solve that its speed is judged by.

A case is a dict of plain values; `prepare` makes its inputs and the handles a
program keeps, `run` makes one pass through the public entry points.  Kinds:

  apply      one operator product (nrhs = 1) or a batch of them, FP64 or
             complex64, on a tensor the library built or (loaded) on one that
             the program put back from a file
  frequency  what a multi-frequency driver does before each solve: new
             background, tensor build and spectrum, conductivity, first product
  solve      the nested FGMRES solve for a plane wave, FP64 or with complex64
             inner solves
  receivers  one frequency's continuation: receiver tensor, its spectrum, and
             the fields at the receivers
  forward    the learned preconditioner's network on one volume
  gradient   forward and parameter gradient of a training batch

Sizes are those of giem2g_amd.models and bench.py (32x32x8, 128x128x32,
256x256x32, batches of 8, networks at 256x256x32 and 8 x 64x64x16), the
reference deck (128x128x50) and the paper's scaling grid (176x224x118).
"""
import math
import os

import numpy as np
import torch

from giem2g_amd import learned, models
from giem2g_amd import operator as gop

EPS0 = 1.0 / (4e-7 * math.pi * 299792458.0 ** 2)
DEV = "cuda"


def listed():
    return [
        # the smallest solve grid's product: launches and latency
        dict(name="apply_fp64_32x32x8", kind="apply", Nx=32, Ny=32, Nz=8, bits=64, nrhs=1, loaded=False),
        # the operator benchmark
        dict(name="apply_fp64_128x128x32", kind="apply", Nx=128, Ny=128, Nz=32, bits=64, nrhs=1, loaded=False),
        # the inner solver's product on the large mixed-precision model
        dict(name="apply_c64_256x256x32", kind="apply", Nx=256, Ny=256, Nz=32, bits=32, nrhs=1, loaded=False),
        # the paper's scaling grid: no side a power of two, more than 64 layers
        dict(name="apply_fp64_176x224x118", kind="apply", Nx=176, Ny=224, Nz=118, bits=64, nrhs=1, loaded=False),
        # several sources at one frequency on a tensor kept in a file
        dict(name="batch8_c64_128x128x32", kind="apply", Nx=128, Ny=128, Nz=32, bits=32, nrhs=8, loaded=True),
        # a whole small FP64 solve: hundreds of short dependent launches
        dict(name="solve_fp64_32x32x8", kind="solve", Nx=32, Ny=32, Nz=8, bits=64, freq=1.0),
        # a whole large solve with complex64 inner solves
        dict(name="solve_mixed_256x256x32", kind="solve", Nx=256, Ny=256, Nz=32, bits=32, freq=0.1),
        # the next frequency on the operator benchmark's grid
        dict(name="frequency_128x128x32", kind="frequency", Nx=128, Ny=128, Nz=32),
        # the next frequency on the reference deck's grid: 50 layers
        dict(name="frequency_128x128x50", kind="frequency", Nx=128, Ny=128, Nz=50),
        # the next frequency's fields at the deck's two receivers
        dict(name="receivers_128x128x32", kind="receivers", Nx=128, Ny=128, Nz=32, Nr=2),
        # the network as the solver calls it on the large model
        dict(name="forward_256x256x32", kind="forward", B=1, Nx=256, Ny=256, Nz=32),
        # a training step's forward and backward
        dict(name="gradient_8x64x64x16", kind="gradient", B=8, Nx=64, Ny=64, Nz=16),
    ]


def _log_int(rng, lo, hi, step=1):
    return max(lo, min(hi, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "apply", "solve", "solve", "frequency", "frequency",
                       "receivers", "forward", "gradient"])
    if kind in ("forward", "gradient"):  # volumes of multiples of four
        B = rng.choice([1, 1, 2]) if kind == "forward" else rng.randint(1, 8)
        return dict(kind=kind, B=B, Nx=_log_int(rng, 16, 128, 4), Ny=_log_int(rng, 16, 128, 4),
                    Nz=_log_int(rng, 8, 32 if kind == "forward" else 16, 4))
    Nx = _log_int(rng, 16, 224, 2)  # any even side; half of the grids square
    Ny = Nx if rng.random() < 0.5 else _log_int(rng, 16, 224, 2)
    if kind == "apply":
        Nz = _log_int(rng, 3, 118)
        while Nx * Ny * Nz * Nz > 128 * 128 * 50 * 50:
            Nz -= Nz // 8 + 1
        bits = rng.choice([64, 32])
        nrhs = rng.choice([1, 1, 1, 2, 3, 8])
        loaded = rng.random() < 0.25 and Nx * Ny * Nz * Nz <= 64 * 64 * 40 * 40
        return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, bits=bits, nrhs=nrhs, loaded=loaded)
    Nz = _log_int(rng, 4, 50)
    if kind == "solve":
        Nx, Ny, Nz = min(Nx, 128), min(Ny, 128), min(Nz, 32)
        return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, bits=rng.choice([64, 32]),
                    freq=round(10.0 ** rng.uniform(-1.0, 1.0), 3))
    if kind == "receivers":
        Nx, Ny, Nz = min(Nx, 128), min(Ny, 128), min(Nz, 32)
        return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz, Nr=rng.randint(1, 4))
    while Nx * Ny * Nz * Nz > 128 * 128 * 50 * 50:
        Nz -= Nz // 8 + 1
    return dict(kind=kind, Nx=Nx, Ny=Ny, Nz=Nz)


# ----------------------------------------------------------------- inputs --
def _rng(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) % (1 << 40))
    return g


def _cvec(n, g, bits=64):
    """Currents: real and imaginary part N(0, 1)."""
    v = torch.randn(n, 2, generator=g, device=DEV, dtype=torch.float64)
    v = torch.view_as_complex(v)
    return v if bits == 64 else v.to(torch.complex64)


def _geometry(case, seed):
    """Background, cells and frequency: the benchmark models' three-layer
    earth (0.01, 0.1, 1 S/m) with cells of 100 x 100 m; layers that meet its
    interface at 1 km, and a frequency that varies with the seed."""
    Nz = case["Nz"]
    dz = next(d for d in (50.0, 25.0, 20.0, 10.0) if Nz * d <= 1000.0 or (d == 10.0))
    if "freq" in case:
        f = case["freq"]
    else:
        f = 10.0 * 10.0 ** float(np.random.default_rng(seed).uniform(-0.5, 0.5))
    return dict(z=np.arange(Nz + 1) * dz, dz=dz, freq=f, omega=2.0 * math.pi * f,
                sigma=[0.01, 0.1, 1.0], thick=[1000.0, 9000.0])


def _csigb(geo):
    return np.array([s - 1j * geo["omega"] * EPS0 for s in [1e-12] + geo["sigma"]])


def _sigma(case, geo, g):
    """Cells of 1e-3 to 1 S/m, log-uniform."""
    n = case["Nx"] * case["Ny"] * case["Nz"]
    s = 10.0 ** (torch.rand(n, generator=g, device=DEV, dtype=torch.float64) * 3.0 - 3.0)
    return torch.complex(s, torch.full_like(s, -geo["omega"] * EPS0))


def _block(Nz):
    return 2 * Nz * (Nz + 1) + 2 * Nz * Nz


def _loaded_tensor(case, geo, g):
    """A spectral tensor of the size the products meet: K of order one."""
    n = case["Nx"] * case["Ny"] * _block(case["Nz"])
    return _cvec(n, g) * (2.0 * geo["dz"] / math.sqrt(3.0 * case["Nz"]))


def _boxes(case, seed):
    """Twenty random boxes of 1e-3 to 10 S/m in a 0.01 S/m host."""
    rng = np.random.Generator(np.random.PCG64(seed))
    return models.random_boxes(rng, case["Nx"], case["Ny"], case["Nz"], 20, 0.01, 1e-3, 10.0,
                               size_lat=(2, max(4, case["Nx"] // 4)), size_z=(1, max(2, case["Nz"] // 2)))


def _volume(case, g):
    """Network input: a residual of unit RMS, log10 contrasts of boxes, log10 of the cell size."""
    B, X, Y, Z = case["B"], case["Nx"], case["Ny"], case["Nz"]
    x = torch.randn(B, Z, Y, X, 8, generator=g, device=DEV, dtype=torch.float32)
    c = torch.rand(B, Z // 4, Y // 4, X // 4, generator=g, device=DEV) * 4.0 - 1.0
    x[..., 6] = c.repeat_interleave(4, 1).repeat_interleave(4, 2).repeat_interleave(4, 3)
    k = torch.rand(B, 1, 1, 1, generator=g, device=DEV) * 2.0 - 2.5
    x[..., 7] = k.expand(B, Z, Y, X)
    return x


def _weights_file():
    return os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "giem2g_amd", "data",
                        "unet_c4.f32")


# ------------------------------------------------------------ prepare, run --
def prepare(case, seed):
    g = _rng(seed)
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        s = dict(kind=kind, net=learned.UNet(params=np.fromfile(_weights_file(), np.float32)),
                 x=_volume(case, g))
        if kind == "gradient":
            s["dy"] = torch.randn(s["x"].shape[:-1] + (6,), generator=g, device=DEV) / s["x"][..., 0].numel()
        return s
    geo = _geometry(case, seed)
    op = gop.IEOperator(case["Nx"], case["Ny"], case["Nz"], 100.0, 100.0, geo["z"])
    op.set_background(_csigb(geo), geo["thick"], geo["omega"])
    s = dict(kind=kind, op=op, geo=geo)
    if kind == "solve":
        sa = torch.from_numpy(_boxes(case, seed).reshape(-1)).to(DEV)
        op.build_tensor()
        op.set_sigma(torch.complex(sa, torch.full_like(sa, -geo["omega"] * EPS0)))
        s["E"] = torch.from_numpy(op.plane_wave(seed % 2)).to(DEV)
        # complex64 inner solves at a tolerance where the field no longer
        # depends on which of two inner iterations the solve stops at
        s["kw"] = dict(outer_m=30, inner_m=30, max_restart=100, tol=1e-8 if case["bits"] == 64 else 1e-10,
                       inner_precision=0 if case["bits"] == 64 else 1)
        return s
    s["sigma"] = _sigma(case, geo, g)
    if kind == "receivers":
        Nr = case["Nr"]
        s["E"] = _cvec(op.nvec, g)
        s["rc"] = gop.ReceiverOperator(op, [0.0] * Nr, [(-1) ** (r + 1) * 20000.0 + 30.0 * r for r in range(Nr)],
                                       [0.0] * Nr)
        s["Ea"] = torch.empty(s["rc"].nfield, dtype=torch.complex128, device=DEV)
        s["Ha"] = torch.empty_like(s["Ea"])
        return s
    if kind == "frequency":
        s["v"] = _cvec(op.nvec, g)
        s["out"] = torch.empty_like(s["v"])
        return s
    if case["loaded"]:
        op.put_tensor(_loaded_tensor(case, geo, g).cpu().numpy(), spectral=True)
    else:
        op.build_tensor()
    op.set_sigma(s["sigma"])
    s["v"] = _cvec(case["nrhs"] * op.nvec, g, case["bits"]).reshape(case["nrhs"], op.nvec)
    s["out"] = torch.empty_like(s["v"])
    torch.cuda.synchronize()
    return s


def run(s):
    kind = s["kind"]
    if kind == "apply":
        if s["v"].shape[0] > 1:
            s["op"].apply_batch_dev(s["v"], s["out"])
        elif s["v"].dtype == torch.complex128:
            s["op"].apply_dev(s["v"], s["out"])
        else:
            s["op"].apply_dev_f32(s["v"], s["out"])
        return s["out"]
    if kind == "solve":
        return s["op"].solve(s["E"], **s["kw"])[0]
    if kind == "frequency":
        geo = s["geo"]
        s["op"].set_background(_csigb(geo), geo["thick"], geo["omega"])
        s["op"].build_tensor()
        s["op"].set_sigma(s["sigma"])
        s["op"].apply_dev(s["v"], s["out"])
        return s["out"]
    if kind == "receivers":
        s["rc"].build()
        s["rc"].set_sigma(s["sigma"])
        s["rc"].recalculate_dev(s["E"], s["Ea"], s["Ha"])
        return {"Ea": s["Ea"], "Ha": s["Ha"]}
    if kind == "forward":
        return s["net"].forward(s["x"])
    y = s["net"].forward(s["x"], keep=True)
    return {"y": y, "grads": s["net"].backward(s["dy"])}


# ------------------------------------------------------------------- work --
def _apply_work(case, size, nrhs, square):
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    n, nc = Nx * Ny, Nx * Ny * Nz
    # a layered earth on square cells: the block of (ky, kx) is that of (kx, ky)
    blocks = n * (Nx + 1) // (2 * Nx) if square and Nx == Ny else n
    fft = 2 * 3 * Nz * (2 * Nx * Ny * 5 * math.log2(2 * Nx) * 0.5 + 4 * n * 5 * math.log2(2 * Ny))
    return dict(bytes=size * (blocks * _block(Nz) + 2 * nc + nrhs * 6 * nc),
                flops=nrhs * (n * 4 * 8 * 9 * Nz * Nz + fft))


def work(case):
    kind = case["kind"]
    if kind in ("forward", "gradient"):
        v = case["B"] * case["Nx"] * case["Ny"] * case["Nz"]
        f0 = 27 * (8 * 16 + 16 * 16 + 48 * 16 + 16 * 16) + 16 * 6
        f1 = 27 * (16 * 32 + 32 * 32 + 96 * 32 + 32 * 32)
        f2 = 27 * (32 * 64 + 64 * 64)
        fwd = 2 * v * (f0 + f1 / 8 + f2 / 64)
        if kind == "forward":
            return dict(bytes=4 * v * 14 + 4 * 356390, flops=fwd)
        # the first layer needs no data gradient
        return dict(bytes=4 * v * 20 + 8 * 356390, flops=3 * fwd - 2 * v * 27 * 8 * 16)
    Nx, Ny, Nz = case["Nx"], case["Ny"], case["Nz"]
    n, nc = Nx * Ny, Nx * Ny * Nz
    if kind == "apply":
        return _apply_work(case, case["bits"] // 4, case["nrhs"], not case["loaded"])
    if kind == "solve":
        # a few outer steps of up to 30 inner ones: 60 products with their share of the basis
        w = _apply_work(case, case["bits"] // 4, 1, True)
        return dict(bytes=60 * (w["bytes"] + case["bits"] // 4 * 30 * 3 * nc), flops=60 * w["flops"])
    if kind == "frequency":
        # 501 filter taps, a real weight times a complex kernel value each; the tensor written once
        w = _apply_work(case, 16, 1, True)
        return dict(bytes=16 * n * _block(Nz) + w["bytes"],
                    flops=501 * 4 * n * (3 * Nz * (Nz + 1) + 2 * Nz * Nz) + w["flops"])
    Nr = case["Nr"]
    return dict(bytes=16 * 4 * n * 15 * Nr * Nz * 2 + 8 * 501 * 6 * 4 * n * Nr + 16 * (4 * nc + 6 * n * Nr),
                flops=501 * 4 * 4 * n * Nr * Nz * 19)


# ------------------------------------------------------------------ exact --
def _exact_apply(case, seed):
    """The scaled operator on a given spectrum: out = sqrt(Re sb) (a v - F / (dz 4 Nx Ny)),
    F the cyclic convolution of (sa - sb) a v on the doubled grid."""
    g, geo = _rng(seed), _geometry(case, seed)
    Nx, Ny, Nz, nrhs = case["Nx"], case["Ny"], case["Nz"], case["nrhs"]
    sa = _sigma(case, geo, g).reshape(Nz, Ny, Nx)
    G = _loaded_tensor(case, geo, g).reshape(Ny, Nx, _block(Nz))
    v = _cvec(nrhs * 3 * Nz * Ny * Nx, g, case["bits"]).to(torch.complex128).reshape(nrhs, 3, Nz, Ny, Nx)
    top = np.concatenate([[0.0], np.cumsum(geo["thick"])])
    mid = (geo["z"][1:] + geo["z"][:-1]) / 2
    sb = np.array([geo["sigma"][int(np.searchsorted(top, m)) - 1] for m in mid])
    sb = torch.from_numpy(sb - 1j * geo["omega"] * EPS0).to(DEV).reshape(Nz, 1, 1)
    sq = torch.sqrt(sb.real)
    a = 2.0 * sq / (sa + sb.conj())
    S = torch.fft.fft2(v * ((sa - sb) * a), s=(2 * Ny, 2 * Nx))
    F = torch.zeros_like(S)
    iu = [(i, j) for j in range(Nz) for i in range(j + 1)]
    up = torch.tensor([[min(i, j) + max(i, j) * (max(i, j) + 1) // 2 for j in range(Nz)] for i in range(Nz)],
                      device=DEV)
    P = len(iu)
    for ky in range(Ny):
        B = G[ky]
        xx, xy, yy, zz = (B[:, c * P:(c + 1) * P][:, up] for c in range(4))
        xz = B[:, 4 * P:4 * P + Nz * Nz].reshape(Nx, Nz, Nz).transpose(1, 2)  # stored by columns
        yz = B[:, 4 * P + Nz * Nz:].reshape(Nx, Nz, Nz).transpose(1, 2)
        for s, m in ((1, 1), (-1, 1), (1, -1), (-1, -1)):
            if m < 0 and ky == 0:
                continue
            M = torch.cat([torch.cat([xx, s * m * xy, s * xz], 2), torch.cat([s * m * xy, yy, m * yz], 2),
                           torch.cat([-s * xz.transpose(1, 2), -m * yz.transpose(1, 2), zz], 2)], 1)
            kx = torch.arange(Nx, device=DEV) if s > 0 else torch.arange(1, Nx, device=DEV)
            px, py = (kx if s > 0 else 2 * Nx - kx), (ky if m > 0 else 2 * Ny - ky)
            V = S[:, :, :, py, px].reshape(nrhs, 3 * Nz, -1).permute(2, 1, 0).contiguous()
            F[:, :, :, py, px] = torch.matmul(M[kx].contiguous(), V).permute(2, 1, 0).reshape(nrhs, 3, Nz, -1)
    f = torch.fft.ifft2(F)[..., :Ny, :Nx] / geo["dz"]
    return (sq * (a * v - f)).reshape(nrhs, -1)


def _conv3(x, W, b):
    """3x3x3 or 1x1x1 convolution of (B, Z, Y, X, ci), zero outside, W (co, taps, ci)."""
    if W.shape[1] == 1:
        return x @ W[:, 0].T + b
    Z, Y, X = x.shape[1:4]
    p = torch.nn.functional.pad(x, (0, 0, 1, 1, 1, 1, 1, 1))
    out = b.expand(x.shape[:4] + b.shape)
    for t in range(27):
        dz, dy, dx = t // 9, (t // 3) % 3, t % 3
        out = out + p[:, dz:dz + Z, dy:dy + Y, dx:dx + X] @ W[:, t].T
    return out


def _exact_net(x, params):
    arch = [(8, 16, 27), (16, 16, 27), (16, 32, 27), (32, 32, 27), (32, 64, 27), (64, 64, 27), (96, 32, 27),
            (32, 32, 27), (48, 16, 27), (16, 16, 27), (16, 6, 1)]
    L, o = [], 0
    for ci, co, t in arch:
        L.append((params[o:o + co * t * ci].reshape(co, t, ci), params[o + co * t * ci:o + co * t * ci + co]))
        o += co * t * ci + co

    def conv(i, h):
        return torch.relu(_conv3(h, *L[i]))

    def pool(h):
        B, Z, Y, X, c = h.shape
        return h.reshape(B, Z // 2, 2, Y // 2, 2, X // 2, 2, c).mean((2, 4, 6))

    def up(h):
        return h.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    e1 = conv(1, conv(0, x))
    e2 = conv(3, conv(2, pool(e1)))
    m = conv(5, conv(4, pool(e2)))
    d2 = conv(7, conv(6, torch.cat([up(m), e2], -1)))
    d1 = conv(9, conv(8, torch.cat([up(d2), e1], -1)))
    return _conv3(d1, *L[10])


def exact(case, seed):
    if case["kind"] == "apply" and case["loaded"]:
        return _exact_apply(case, seed)
    if case["kind"] not in ("forward", "gradient"):
        return None  # the layered earth's Green tensor has no closed form to compare with
    g = _rng(seed)
    x = _volume(case, g).double()
    p = torch.from_numpy(np.fromfile(_weights_file(), np.float32)).to(DEV).double()
    if case["kind"] == "forward":
        with torch.no_grad():
            return _exact_net(x, p)
    dy = torch.randn(x.shape[:-1] + (6,), generator=g, device=DEV) / x[..., 0].numel()
    p.requires_grad_(True)
    y = _exact_net(x, p)
    (y * dy.double()).sum().backward()
    return {"y": y.detach(), "grads": p.grad.cpu().numpy()}
