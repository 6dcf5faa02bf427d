"""Adjoint-state gradient on the GPU.

The gradient linearises an fp64 trajectory of the single-pass solve recorded
on the device (branch decisions and local partials in fp64, adjoint
recurrence in fp32, cross-shot sums in fp64); the misfit's residuals use the
picks of that trajectory.  Checked
* against the fp64 oracle's discrete adjoint of the same map (agreement to
  fp32 rounding of the recurrence, not bits);
* against FP64 central finite differences of the FP64 oracle forward, along
  smooth directions (<= 1e-3 relative), including the
  128-shot 301x1201 tomography workload on a 51x151 sub-block;
* linearity and run-to-run determinism of the vector-Jacobian product;
* the torch.autograd wrapper;
* the reference's ray-traced tomography gradient (correlation).
"""
import numpy as np
import pytest
from scipy.ndimage import gaussian_filter

from seisfat2d_amd import SCHED_PLAIN, SCHED_TILED, SCHED_TILED_DIAG, Eikonal, capi, models

pytestmark = pytest.mark.gpu


def smooth_slowness(rng, nz, nx, dh, sigma=3.0, amp=400.0):
    v = 2000 + amp * gaussian_filter(rng.standard_normal((nx, nz)), sigma) + 1.5 * np.arange(nz)[None, :] * dh
    return (1.0 / v).astype(np.float32)


def window_case(rng, nz=40, nx=160, dh=10.0):
    s = smooth_slowness(rng, nz, nx, dh)
    shots, rx, rz = [], [], []
    for sx, sz, x0, w in ((800.0, 0.0, 0, nx), (300.0, 50.0, 10, 60), (1200.0, 0.0, 70, 90), (1000.0, 120.0, 0, nx)):
        xs = np.arange(x0 + 1, x0 + w - 1, 3) * dh + 4.0
        shots.append((sx, sz, x0, w, len(rx), len(xs)))
        rx.extend(xs)
        rz.extend([15.0] * len(xs))
    return s, dh, shots, np.array(rx, np.float32), np.array(rz, np.float32)


def gpu_obs(e, s_true, b):
    e.set_slowness(s_true)
    b.run()
    return b.picks()


@pytest.mark.parametrize("sched", [SCHED_TILED, SCHED_TILED_DIAG, SCHED_PLAIN])
def test_gradient_matches_oracle_adjoint(oracle, rng, sched):
    check_gradient_against_oracle(oracle, rng, sched, nz=40)


def test_gradient_matches_oracle_adjoint_strips(oracle, rng):
    """Three 64-row strips per shot (156 padded rows): the FP64 walk and the
    reverse sweep pass each strip's last row to the next through tagged words."""
    check_gradient_against_oracle(oracle, rng, SCHED_TILED, nz=150)


def check_gradient_against_oracle(oracle, rng, sched, nz):
    s, dh, shots, rx, rz = window_case(rng, nz=nz)
    nx, nz = s.shape
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz, schedule=sched)
    obs = gpu_obs(e, (s * np.float32(1.03)).astype(np.float32), b)
    e.set_slowness(s)
    J, g, pk = b.misfit_gradient(obs)
    _, _, pko = oracle.batch_misfit(s, dh, dh, shots, rx, rz, obs, grad=False)
    assert np.array_equal(pk, pko)  # the production fp32 picks stay bit-exact
    Jo, go, _ = oracle.batch_misfit(s.astype(np.float64), dh, dh, shots, rx, rz, obs.astype(np.float64))
    assert np.isclose(J, Jo, rtol=1e-10)  # fp64 trajectory picks
    err = np.abs(g - go).max() / np.abs(go).max()
    print(f"sched {sched}: max|g| {np.abs(go).max():.3e}, max rel err vs oracle adjoint {err:.2e}")
    assert err < 1e-5
    b.close()
    e.close()


def test_vjp_linear_and_deterministic(rng):
    import torch
    s, dh, shots, rx, rz = window_case(rng, nz=70, nx=200)
    nx, nz = s.shape
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz)
    b.run_record()
    n = len(rx)
    w1 = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
    w2 = torch.from_numpy(rng.standard_normal(n).astype(np.float32)).cuda()
    out = []
    for w in (w1, w2, w1 + w2, w1):
        g = torch.empty((nx, nz), dtype=torch.float64, device="cuda")
        b.vjp_device(w.data_ptr(), g.data_ptr(), torch.cuda.current_stream().cuda_stream)
        out.append(g.cpu().numpy())
    g1, g2, g12, g1b = out
    assert np.array_equal(g1, g1b)
    assert np.abs(g12 - (g1 + g2)).max() <= 1e-5 * np.abs(g12).max()
    # a new model invalidates the recorded run
    e.set_slowness(s)
    g = torch.empty((nx, nz), dtype=torch.float64, device="cuda")
    with pytest.raises(capi.SeisfatError) as ex:
        b.vjp_device(w1.data_ptr(), g.data_ptr())
    assert ex.value.code == capi.ESTATE
    b.close()
    e.close()


def smooth_direction(rng, shape, box, sigma=4.0):
    v = np.zeros(shape)
    (x0, x1), (z0, z1) = box
    v[x0:x1, z0:z1] = gaussian_filter(rng.standard_normal((x1 - x0, z1 - z0)), sigma)
    return v / np.abs(v).max()


def blob(shape, cx, cz, sigma):
    x = np.arange(shape[0])[:, None]
    z = np.arange(shape[1])[None, :]
    return np.exp(-((x - cx) ** 2 + (z - cz) ** 2) / (2.0 * sigma ** 2))


def fd_check(oracle, s, dh, shots, rx, rz, obs, g, dirs, rel_h=1e-5, tol=1e-3):
    """Directional derivatives <g, v> against FP64 central differences of the
    FP64 forward.  Directions must not make the derivative cancel: the
    difference quotient carries an absolute noise of the kinks it straddles
    (branch switches within +-h), which no relative bar survives near zero."""
    s64 = s.astype(np.float64)
    worst = 0.0
    for v in dirs:
        h = rel_h * float(np.abs(s64).max())
        jp = oracle.batch_misfit(s64 + h * v, dh, dh, shots, rx, rz, obs.astype(np.float64), grad=False)[0]
        jm = oracle.batch_misfit(s64 - h * v, dh, dh, shots, rx, rz, obs.astype(np.float64), grad=False)[0]
        fd = (jp - jm) / (2 * h)
        an = float(np.sum(g * v))
        rel = abs(an - fd) / abs(fd)
        print(f"  directional derivative: adjoint {an:.6e}  FP64 FD {fd:.6e}  rel {rel:.2e}")
        worst = max(worst, rel)
    assert worst <= tol
    return worst


def test_gradient_vs_fp64_finite_differences(oracle, rng):
    s, dh, shots, rx, rz = window_case(rng, nz=60, nx=200)
    nx, nz = s.shape
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz)
    obs = gpu_obs(e, smooth_slowness(rng, nz, nx, dh, amp=300.0), b)
    e.set_slowness(s)
    _, g, _ = b.misfit_gradient(obs)
    dirs = [smooth_direction(rng, s.shape, ((20, 180), (5, 55))) for _ in range(3)]
    fd_check(oracle, s, dh, shots, rx, rz, obs, g, dirs)
    b.close()
    e.close()


def test_c5_tomography_gradient(oracle, rng):
    """128 shots x 401 receivers on 301x1201 (dh 10 m): observed picks from
    the true model (v(z) + 4 anomalies), gradient at the v(z) start model;
    FP64 finite differences on a 51x151 sub-block and the oracle adjoint."""
    w = models.c5()
    e = Eikonal(w.nz, w.nx, w.dz, w.dx)
    e.set_slowness(w.s)
    b = e.batch(w.shots, w.rx, w.rz)
    obs = gpu_obs(e, w.extra["s_true"], b)
    e.set_slowness(w.s)
    J, g, pk = b.misfit_gradient(obs)
    Jo, go, _ = oracle.batch_misfit(w.s.astype(np.float64), w.dx, w.dz, w.shots, w.rx, w.rz, obs.astype(np.float64))
    err = np.abs(g - go).max() / np.abs(go).max()
    print(f"C5: J {J:.6e} (oracle {Jo:.6e}); max rel err vs oracle adjoint {err:.2e}")
    assert np.isclose(J, Jo, rtol=1e-10)
    assert err < 1e-5
    # sub-block of 51 x 151 cells (z 100..150, x 525..675) around the middle:
    # one-signed bumps and smooth random fields supported on it
    box = ((525, 676), (100, 151))
    mask = np.zeros(w.s.shape)
    mask[525:676, 100:151] = 1.0
    dirs = [blob(w.s.shape, 600, 125, 8.0) * mask, blob(w.s.shape, 650, 110, 4.0) * mask,
            smooth_direction(rng, w.s.shape, box, sigma=6.0), smooth_direction(rng, w.s.shape, box, sigma=12.0)]
    worst = fd_check(oracle, w.s, w.dx, w.shots, w.rx, w.rz, obs, g, dirs)
    print(f"C5 sub-block FD: worst rel err {worst:.2e}")
    b.close()
    e.close()


def test_autograd_function(rng):
    import torch
    from seisfat2d_amd.autograd import eikonal_picks
    s, dh, shots, rx, rz = window_case(rng, nz=50, nx=180)
    nx, nz = s.shape
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz)
    obs = gpu_obs(e, (s * np.float32(0.97)).astype(np.float32), b)
    st = torch.from_numpy(s).cuda().requires_grad_(True)
    picks = eikonal_picks(st, b)
    loss = 0.5 * ((picks - torch.from_numpy(obs).cuda()) ** 2).sum()
    loss.backward()
    b.run()
    assert np.array_equal(picks.detach().cpu().numpy(), b.picks())
    # the backward is the vector-Jacobian product with w = dloss/dpicks
    w = (picks.detach() - torch.from_numpy(obs).cuda()).contiguous()
    b.run_record()
    g = torch.empty((nx, nz), dtype=torch.float64, device="cuda")
    b.vjp_device(w.data_ptr(), g.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(st.grad, g.float())
    # and it agrees with the misfit gradient (residuals of the fp64 trajectory)
    _, gm, _ = b.misfit_gradient(obs)
    assert np.abs(st.grad.cpu().numpy() - gm).max() <= 1e-3 * np.abs(gm).max()
    b.close()
    e.close()


def test_autograd_backward_refuses_a_stale_record(rng):
    """One batch holds one recorded trajectory.  After a second forward on the
    same batch (a line search, a second loss), the first graph's backward
    would linearise the second slowness: it raises instead; the second
    graph's backward is exact."""
    import torch
    from seisfat2d_amd.autograd import eikonal_picks
    s, dh, shots, rx, rz = window_case(rng, nz=40)
    nx, nz = s.shape
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz)
    s1 = torch.from_numpy(s).cuda().requires_grad_(True)
    s2 = torch.from_numpy((s * np.float32(1.02)).astype(np.float32)).cuda().requires_grad_(True)
    p1 = eikonal_picks(s1, b)
    p2 = eikonal_picks(s2, b)
    with pytest.raises(RuntimeError, match="another forward"):
        p1.sum().backward()
    p2.sum().backward()
    g = torch.empty((nx, nz), dtype=torch.float64, device="cuda")
    ones = torch.ones(len(rx), dtype=torch.float32, device="cuda")
    b.vjp_device(ones.data_ptr(), g.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(s2.grad, g.float())
    b.close()
    e.close()


def test_ray_gradient_correlation(oracle, rng):
    """The reference's tomography gradient G^T r (ray-traced, src/inversion/
    inversion.cpp:95-177) and the adjoint gradient of the same misfit agree in
    pattern: correlation after a light smoothing of both."""
    nz, nx, dh = 101, 401, 10.0
    v = 1500.0 + 1.0 * np.arange(nz)[None, :] * dh + np.zeros((nx, 1))
    xg, zg = np.meshgrid(np.arange(nx) * dh, np.arange(nz) * dh, indexing="ij")
    v_true = v * (1 + 0.05 * np.exp(-((xg - 2000) ** 2 + (zg - 500) ** 2) / (2 * 200.0 ** 2)))
    s = (1 / v).astype(np.float32)
    rx1 = np.arange(0, nx * dh - dh / 2, 20.0).astype(np.float32)
    shots = [((k + 0.5) * (nx - 1) * dh / 16, 0.0, 0, nx, k * len(rx1), len(rx1)) for k in range(16)]
    rx = np.tile(rx1, 16)
    rz = np.zeros_like(rx)
    e = Eikonal(nz, nx, dh, dh)
    e.set_slowness(s)
    b = e.batch(shots, rx, rz)
    obs = gpu_obs(e, (1 / v_true).astype(np.float32), b)
    e.set_slowness(s)
    _, g, pk = b.misfit_gradient(obs)
    res = pk.astype(np.float64) - obs
    g_ray = np.zeros(nx * nz)
    for k, sh in enumerate(shots):
        T = b.T(k)
        sl = slice(sh[4], sh[4] + sh[5])
        rec, cell, ln = oracle.ray_paths(T, nz, nx, dh, dh, sh[0], sh[1], rx[sl], rz[sl])
        np.add.at(g_ray, cell, ln * res[sl][rec])
    g_ray = g_ray.reshape(nx, nz)
    a = gaussian_filter(g, 3.0).ravel()
    r = gaussian_filter(g_ray, 3.0).ravel()
    corr = np.corrcoef(a, r)[0, 1]
    print(f"adjoint vs ray-traced gradient: correlation {corr:.3f}")
    assert corr > 0.9
    b.close()
    e.close()


# the FP64 walk at the edges of its strips (64 rows), blocks (8 steps) and ring,
# with skewed and clamped slowness columns (narrow windows, window edges) and
# both spacings: the misfit and its gradient against the FP64 oracle
@pytest.mark.parametrize("nz,nx,dz,dx,wins", [(8, 9, 10.0, 10.0, None), (57, 70, 10.0, 10.0, None),
                                              (58, 131, 10.0, 7.0, None), (59, 150, 6.0, 9.0, [(0, 90), (41, 109), (60, 30)]),
                                              (122, 200, 10.0, 10.0, [(0, 200), (3, 180), (100, 64), (150, 50)]),
                                              (190, 77, 12.0, 5.0, None)])
def test_walk_edges(oracle, nz, nx, dz, dx, wins):
    w = models.rough(nz, nx, dz, dx, seed=nz + nx, sigma=4.0, vlo=2000.0, vhi=3000.0)
    shots, rx, off = [], [], 0
    for k, (x0, wd) in enumerate(wins or [(0, nx)] * 2):
        r = np.linspace(x0 + 0.1, x0 + wd - 1.1, 7) * dx
        shots.append((float(np.float32((x0 + (0.3 + 0.2 * k % 0.6) * (wd - 1)) * dx)), 0.0, x0, wd, off, len(r)))
        rx.append(r)
        off += len(r)
    rx = np.concatenate(rx).astype(np.float32)
    rz = np.full(len(rx), 0.3 * dz, np.float32)
    obs = np.linspace(0.0, 0.3, len(rx)).astype(np.float32)
    e = Eikonal(nz, nx, dz, dx)
    e.set_slowness(w.s)
    b = e.batch(shots, rx, rz)
    J, g, _ = b.misfit_gradient(obs)
    Jo, go, _ = oracle.batch_misfit(w.s.astype(np.float64), dx, dz, shots, rx, rz, obs.astype(np.float64))
    assert np.isclose(J, Jo, rtol=1e-10)
    assert np.abs(g - go).max() <= 1e-5 * np.abs(go).max()
    b.close()
    e.close()
