"""GPU parity of the learned preconditioner's HIP kernels (U-Net forward,
backward and training on MFMA, feature packing) against the FP64 oracle
(oracle/unet_ref.py), and the solver's learned modes.

Bars: forward output within 2e-2 relative (2-norm) of the oracle with the
same bfloat16 roundings; per-layer parameter gradients within 5e-2
relative; features within 1e-6; learned solves reach the FP64 1e-8 true
residual and agree with the plain FP64 solve within 1e-6.
"""
import numpy as np
import pytest

from tests.conftest import rel

pytestmark = pytest.mark.gpu


def _torch():
    import torch
    assert torch.cuda.is_available(), "GPU test without a GPU"
    return torch


def _params(seed):
    from oracle import unet_ref as U
    rng = np.random.default_rng(seed)
    p = U.init_params(seed)
    # nonzero biases and a larger output layer so every path carries signal
    out = []
    for (W, b), (name, *_rest) in zip(U.split(p.astype(np.float64)), U.LAYERS):
        s = 10.0 if name == "out" else 1.0
        out.append((W * s).ravel())
        out.append(0.05 * rng.standard_normal(b.size))
    return np.concatenate(out).astype(np.float32)


@pytest.mark.parametrize("B,Z,Y,X", [(1, 4, 4, 4), (2, 8, 8, 12), (1, 8, 16, 8)])
def test_unet_forward_backward_match_oracle(B, Z, Y, X):
    torch = _torch()
    from giem2g_amd import learned
    from oracle import unet_ref as U
    print("case", B, Z, Y, X, flush=True)
    rng = np.random.default_rng(B * 100 + Z + Y + X)
    p = _params(7)
    net = learned.UNet(params=p)
    x = rng.standard_normal((B, Z, Y, X, 8)).astype(np.float32)
    x[..., 7] = 0
    y = net.forward(torch.from_numpy(x).cuda(), keep=True)
    torch.cuda.synchronize()
    y = y.cpu().numpy().astype(np.float64)
    dy = rng.standard_normal(y.shape).astype(np.float32)
    g = net.backward(torch.from_numpy(dy).cuda()).astype(np.float64)
    gref = np.zeros(p.size)
    for b in range(B):
        o, cache = U.forward(p.astype(np.float64), x[b].astype(np.float64), round_bf16=True)
        e = rel(y[b], o)
        assert e < 2e-2, ("forward", b, e)
        gref += U.backward(p, cache, dy[b].astype(np.float64), round_bf16=True)
    off = 0
    for li, (W, bb) in enumerate(U.split(gref)):
        n = W.size
        ew = rel(g[off:off + n], W.ravel())
        eb = rel(g[off + n:off + n + bb.size], bb)
        off += n + bb.size
        assert ew < 5e-2 and eb < 5e-2, ("grad layer", li, ew, eb)
    net.close()


def test_unet_training_reduces_loss():
    torch = _torch()
    from giem2g_amd import learned
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0)
    x = torch.randn((4, 8, 8, 8, 8), generator=gen, device="cuda")
    x[..., 7] = 0
    # a smooth, learnable target: a fixed linear map of the input channels
    M = torch.randn((8, 6), generator=gen, device="cuda") * 0.5
    t = (x @ M).contiguous()
    net = learned.UNet(seed=1)
    losses = [net.train_step(x, t, 2e-3) for _ in range(150)]
    print("loss", losses[0], losses[-1], flush=True)
    assert losses[-1] < 0.3 * losses[0]
    net.close()


def test_learned_features(oracle):
    torch = _torch()
    from giem2g_amd import learned, models, operator as gop
    m = models.small(8, 8, 4, seed=3, freq=3.0)
    op = gop.operator_for(m)
    net = learned.UNet(seed=0)
    op.set_learned(net)
    rng = np.random.default_rng(5)
    n = 3 * m.ncell
    r = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    e = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    x = torch.empty((m.Nz, m.Ny, m.Nx, 8), dtype=torch.float32, device="cuda")
    t = torch.empty((m.Nz, m.Ny, m.Nx, 6), dtype=torch.float32, device="cuda")
    op.learned_features(torch.from_numpy(r).cuda(), torch.from_numpy(e).cuda(), x, t)
    x, t = x.cpu().numpy(), t.cpu().numpy()
    rms = np.linalg.norm(r) / np.sqrt(n)
    rr = r.reshape(3, m.Nz, m.Ny, m.Nx)
    ee = e.reshape(3, m.Nz, m.Ny, m.Nx)
    om = oracle.Model(m.csigb(), m.thick, m.omega, m.Nx, m.Ny, m.Nz, m.dx, m.dy, m.z)
    ln = om.lnum()
    cb = m.csigb()
    sb = np.array([cb[ln[i + 1]] for i in range(m.Nz)])[:, None, None]
    sa = m.csiga().reshape(m.Nz, m.Ny, m.Nx)
    a = 2 * np.sqrt(sb.real) / (sa + np.conj(sb))
    for c in range(3):
        assert rel(x[..., 2 * c] + 1j * x[..., 2 * c + 1], rr[c] / rms) < 1e-6
        assert rel(t[..., 2 * c] + 1j * t[..., 2 * c + 1], a * ee[c] / rms) < 1e-6
    assert np.allclose(x[..., 6], np.log10(sa.real / sb.real), atol=1e-5)
    k = np.sqrt(m.omega * 4e-7 * np.pi * np.abs(sb))  # background wavenumber |k_b|
    assert np.allclose(x[..., 7], np.broadcast_to(np.log10(k * m.dx), x[..., 7].shape), atol=1e-5)
    op.set_learned(None)
    op.close()
    net.close()


@pytest.mark.parametrize("mode,prec", [(1, 0), (1, 1), (2, 0), (2, 1)])
def test_learned_modes_converge_with_untrained_net(mode, prec):
    """An untrained network must not break the solve: the fallback keeps the
    FP64 true residual below 1e-8 and the solution equal to plain FP64."""
    from giem2g_amd import learned, models, operator as gop
    print("mode", mode, "precision", prec, flush=True)
    m = models.small(16, 16, 8, seed=11, freq=1.0)
    op = gop.operator_for(m)
    E = op.plane_wave(1)
    E0, i0 = op.solve(E, outer_m=10, inner_m=10, max_restart=50, tol=1e-8)
    net = learned.UNet(seed=2)
    op.set_learned(net, accept=0.9)
    E1, i1 = op.solve(E, outer_m=10, inner_m=10, max_restart=50, tol=1e-8, inner_precision=prec,
                      precond=mode)
    print(i0, i1, flush=True)
    assert i1["status"] == 1 and i1["true_residual"] < 1e-8
    assert i1["precond_calls"] > 0
    assert rel(E1, E0) < 1e-6
    op.set_learned(None)
    op.close()
    net.close()


@pytest.mark.parametrize("B,Z,Y,X", [(1, 4, 4, 20), (2, 4, 12, 36), (1, 12, 20, 4), (1, 20, 36, 8)])
def test_unet_tiles_with_remainders(B, Z, Y, X):
    """Volumes that no tile shape (16x4x4, 8x8x4, 4x8x8 and their halves)
    divides, at every level: the output against the oracle with the same
    roundings (the 2e-2 bar above) and, bit for bit, the pass that reads the
    FP32 input itself against the one that keeps activations, and an input
    that is not 16-byte aligned against an aligned one."""
    torch = _torch()
    from giem2g_amd import learned
    from oracle import unet_ref as U
    print("case", B, Z, Y, X, flush=True)
    rng = np.random.default_rng(B * 100 + Z + Y + X)
    p = _params(11)
    x = rng.standard_normal((B, Z, Y, X, 8)).astype(np.float32)
    xt = torch.from_numpy(x).cuda()
    off = torch.empty(xt.numel() + 1, dtype=torch.float32, device="cuda")[1:].view(xt.shape)
    off.copy_(xt)
    assert off.data_ptr() % 16 and off.is_contiguous()
    net = learned.UNet(params=p)
    y = net.forward(xt)
    assert torch.equal(net.forward(off), y)
    assert torch.equal(net.forward(xt, keep=True), y)
    assert torch.equal(net.forward(off, keep=True), y)
    y = y.cpu().numpy().astype(np.float64)
    for b in range(B):
        o, _ = U.forward(p.astype(np.float64), x[b].astype(np.float64), round_bf16=True)
        assert rel(y[b], o) < 2e-2
    net.close()


@pytest.mark.parametrize("B,Z,Y,X", [(1, 4, 4, 4), (2, 12, 20, 36), (1, 8, 12, 64), (3, 4, 28, 16)])
def test_weight_gradient_sums(B, Z, Y, X):
    """Weight and bias gradients of the last two layers against FP64 sums of
    the same products, where they are known exactly: a network that hands
    channels 0-7 through (identity taps), so that both layers' input is
    relu(x) and the output gradient reaches them unmixed.  The products are
    exact and the sums FP32, over 32 voxels at a time: within
    (voxels / 32 + 64) 2^-24 of the sum of the terms' magnitudes."""
    torch = _torch()
    from giem2g_amd import learned
    print("case", B, Z, Y, X, flush=True)
    parts, offs, off = [], [], 0
    for li, (ci, co, t) in enumerate(learned.ARCH):
        W = np.zeros((co, t, ci), np.float32)
        for c in range(6 if li == 10 else 8):
            if li in (0, 1, 9, 10):
                W[c, t // 2, c] = 1
            elif li == 8:
                W[c, t // 2, 32 + c] = 1
        parts += [W.ravel(), np.zeros(co, np.float32)]
        offs.append(off)
        off += co * t * ci + co
    gen = torch.Generator(device="cuda")
    gen.manual_seed(X)
    x = torch.randn((B, Z, Y, X, 8), generator=gen, device="cuda").to(torch.bfloat16).float()
    dy = torch.randn((B, Z, Y, X, 6), generator=gen, device="cuda")
    net = learned.UNet(params=np.concatenate(parts))
    net.forward(x, keep=True)
    g = net.backward(dy)
    assert np.array_equal(net.backward(dy), g)  # fixed order of the sums
    g = g.astype(np.float64)
    a, d = torch.relu(x).double().cpu().numpy(), dy.double().cpu().numpy()
    n = B * Z * Y * X
    bar = (n / 32 + 64) * 2.0 ** -24
    A, D = a.reshape(n, 8), d.reshape(n, 6)
    w10 = g[offs[10]:offs[10] + 96].reshape(6, 16)[:, :8]
    assert np.all(np.abs(w10 - D.T @ A) <= bar * (np.abs(D).T @ A))
    assert np.all(np.abs(g[offs[10] + 96:] - D.sum(0)) <= bar * np.abs(D).sum(0))
    d9 = dy.to(torch.bfloat16).double().cpu().numpy() * (a[..., :6] > 0)
    D9 = d9.reshape(n, 6)
    p = np.pad(a, ((0, 0), (1, 1), (1, 1), (1, 1), (0, 0)))
    w9 = g[offs[9]:offs[9] + 16 * 27 * 16].reshape(16, 27, 16)
    for t in range(27):
        dz, ty, tx = t // 9, (t // 3) % 3, t % 3
        q = p[:, dz:dz + Z, ty:ty + Y, tx:tx + X].reshape(n, 8)
        assert np.all(np.abs(w9[:6, t, :8] - D9.T @ q) <= bar * (np.abs(D9).T @ q)), t
    b9 = g[offs[9] + 16 * 27 * 16:offs[10]]
    assert np.all(np.abs(b9[:6] - D9.sum(0)) <= bar * np.abs(D9).sum(0)) and not np.any(b9[6:])
    net.close()


@pytest.mark.parametrize("B,Z,Y,X", [(3, 12, 4, 8), (1, 8, 12, 20), (2, 4, 28, 4)])
def test_gradient_through_the_levels(B, Z, Y, X):
    """Layers whose output's gradient comes from a concatenation (the sum of
    the upsampled voxel's eight children) or from a concatenation and a pooling,
    on volumes of different sides: every layer's gradients against the oracle
    (the 5e-2 bar above) and the same bits twice."""
    torch = _torch()
    from giem2g_amd import learned
    from oracle import unet_ref as U
    print("case", B, Z, Y, X, flush=True)
    rng = np.random.default_rng(X)
    p = _params(5)
    x = rng.standard_normal((B, Z, Y, X, 8)).astype(np.float32)
    dy = rng.standard_normal((B, Z, Y, X, 6)).astype(np.float32)
    net = learned.UNet(params=p)
    net.forward(torch.from_numpy(x).cuda(), keep=True)
    g = net.backward(torch.from_numpy(dy).cuda())
    assert np.array_equal(net.backward(torch.from_numpy(dy).cuda()), g)
    gref = np.zeros(p.size)
    for b in range(B):
        _, cache = U.forward(p.astype(np.float64), x[b].astype(np.float64), round_bf16=True)
        gref += U.backward(p, cache, dy[b].astype(np.float64), round_bf16=True)
    off = 0
    for li, (W, bb) in enumerate(U.split(gref)):
        for ref in (W.ravel(), bb):
            assert rel(g[off:off + ref.size].astype(np.float64), ref) < 5e-2, ("layer", li)
            off += ref.size
    net.close()


@pytest.mark.parametrize("B,Z,Y,X,q", [(1, 4, 4, 20, (0, 0, 19)), (2, 12, 20, 12, (11, 19, 0)), (1, 8, 4, 36, (4, 2, 17)),
                                       (1, 4, 28, 16, (3, 27, 15))])
def test_infinite_activation_in_the_gradient(B, Z, Y, X, q):
    """One infinite input voxel through a network of positive weights: every
    layer's input is positive and infinite near that voxel, the output
    gradient is positive and finite.  A product of an infinite activation
    with a nonzero gradient is infinite, and voxels outside the volume (in
    tiles with remainders) have none: no entry of the gradient is NaN, the
    first layer's infinite entries are those whose tap reaches the voxel from
    inside the volume, and the rest are the sums of a run whose voxel is
    finite, to the bar of the sums above."""
    torch = _torch()
    from giem2g_amd import learned
    print("case", B, Z, Y, X, q, flush=True)
    rng = np.random.default_rng(X)
    parts = []
    for ci, co, t in learned.ARCH:
        parts += [rng.uniform(0.5, 1.5, co * t * ci) / (t * ci), np.full(co, 0.01)]
    net = learned.UNet(params=np.concatenate(parts).astype(np.float32))
    x = torch.from_numpy(rng.uniform(0.5, 1.0, (B, Z, Y, X, 8)).astype(np.float32)).cuda()
    dy = torch.from_numpy(rng.uniform(0.5, 1.0, (B, Z, Y, X, 6)).astype(np.float32)).cuda()
    ch, bat = 5, B - 1
    net.forward(x, keep=True)
    gf = net.backward(dy).astype(np.float64)
    x[(bat,) + q + (ch,)] = float("inf")
    y = net.forward(x, keep=True)
    assert not torch.isnan(y).any()
    g = net.backward(dy).astype(np.float64)
    assert not np.isnan(g).any() and np.all(g >= 0)
    n = B * Z * Y * X
    bar = 2 * (n / 32 + 64) * 2.0 ** -24
    off = 0
    for li, (ci, co, t) in enumerate(learned.ARCH):
        w, wf = g[off:off + co * t * ci].reshape(co, t, ci), gf[off:off + co * t * ci].reshape(co, t, ci)
        off += co * t * ci
        b, bf = g[off:off + co], gf[off:off + co]
        off += co
        assert np.all(np.abs(b - bf) <= bar * bf), ("bias", li)
        if li:
            assert np.isinf(w).any(), li
            continue
        for k in range(27):
            p = [q[0] - (k // 9 - 1), q[1] - ((k // 3) % 3 - 1), q[2] - (k % 3 - 1)]
            inside = all(0 <= a < s for a, s in zip(p, (Z, Y, X)))
            assert np.all(np.isinf(w[:, k, ch]) == inside), (k, inside)
        fin = np.isfinite(w)
        fin[:, :, ch] = False
        assert np.all(np.delete(fin, ch, 2))
        assert np.all(np.abs(w[fin] - wf[fin]) <= bar * wf[fin])
    # back on finite data, the same bits as before
    x[(bat,) + q + (ch,)] = 0.75
    net.forward(x, keep=True)
    g1 = net.backward(dy)
    net.forward(x, keep=True)
    assert np.array_equal(net.backward(dy), g1) and np.isfinite(g1).all()
    net.close()


def test_gradient_of_a_long_volume():
    """More layers than a launch grid's y axis takes (65535).  The output
    gradient is zero but for the last 8 layers.  It reaches fewer than 30 layers
    back and the activations there 30 further, so every layer's gradient is
    that of the last 96 layers alone.  Both are FP32 sums of the same products
    (at most 16 x 50 nonzero ones) in another order: 800 x 2^-24."""
    torch = _torch()
    from giem2g_amd import learned
    from oracle import unet_ref as U
    Z, K = 65540, 96
    rng = np.random.default_rng(4)
    net = learned.UNet(params=_params(2))
    x = torch.from_numpy(rng.standard_normal((1, Z, 4, 4, 8)).astype(np.float32)).cuda()
    dy = torch.zeros((1, Z, 4, 4, 6), device="cuda")
    dy[:, -8:] = torch.from_numpy(rng.standard_normal((1, 8, 4, 4, 6)).astype(np.float32)).cuda()
    net.forward(x, keep=True)
    g = net.backward(dy).astype(np.float64)
    net.forward(x[:, -K:].contiguous(), keep=True)
    ref = net.backward(dy[:, -K:].contiguous()).astype(np.float64)
    off = 0
    for li, (W, bb) in enumerate(U.split(ref)):
        for r in (W.ravel(), bb):
            e = rel(g[off:off + r.size], r)
            assert e < 800 * 2.0 ** -24, (li, e)
            off += r.size
    net.close()
