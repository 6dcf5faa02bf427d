"""Kirchhoff depth migration on the GPU against the oracle.

Bars (the GPU forms each weight from per-table amplitudes and half-angle
cosines and sines, within a few ulp of the reference's order of roundings,
and its acosf / expf differ from the host's by an ulp or two; traveltime sums,
time indices, the convolutions and the trace order of the image-domain
adjoint are exact):
  - convolutions: bit-identical (the same double sums in the same order);
  - image-domain adjoint: |m_gpu - m_oracle| <= 1e-5 * max |m_oracle|;
  - forward (LDS accumulation order differs from the reference's atomics):
    per sample |d_gpu - d_oracle| <= 1e-5 * (L |m|) + 1e-30, L |m| the
    oracle's forward of |m|;
  - angle domain: the same bars on all but 0.1 % of the entries (an angle
    within an ulp of a bin edge may land in the neighbouring bin), and the
    gather summed over angles within the image-domain bar;
  - the migration loops: KDM as the adjoint; LSKDM residual norms within
    1e-4 relative (float64 sums here, float32 sums in trace order in the
    reference), the image within 1e-4 of its largest value, the angle
    gather within 1e-3 in norm after three iterations.
"""
import numpy as np
import pytest

from seisfat2d_amd import Eikonal, migration as mig, models

pytestmark = pytest.mark.gpu

NB = 3


@pytest.fixture(scope="module")
def torch():
    import torch
    return torch


def survey(nz=48, nx=84, dz=10.0, dx=10.0, nsrc=4, nrec=14, seed=1):
    m = models.rough(nz, nx, dz, dx, seed=seed, vlo=1800.0, vhi=3500.0, sigma=3.0)
    xs = np.linspace(40.0, (nx - 1) * dx - 40.0, nsrc).astype(np.float32)
    xr = np.linspace(0.0, (nx - 1) * dx, nrec).astype(np.float32)
    return m, xs, xr


def make(e, m, xs, xr, domain, nt=420, dt=2e-3, max_offset=500.0, aperture=30.0, da=3.0, max_angle=60.0,
         tables=None):
    return mig.Kirchhoff(e, xs, np.zeros_like(xs), xr, np.zeros_like(xr), nt, dt, aperture, max_offset, 30.0,
                         domain=domain, da=da, max_angle=max_angle, tables=tables)


@pytest.fixture(scope="module")
def setup():
    m, xs, xr = survey()
    e = Eikonal(m.s.shape[1], m.s.shape[0], m.dz, m.dx)
    e.set_slowness(m.s)
    ts = e.traveltime_tables(xs, np.zeros_like(xs))
    tr = e.traveltime_tables(xr, np.zeros_like(xr))
    yield dict(m=m, xs=xs, xr=xr, e=e, ts=ts, tr=tr)
    e.close()


def orc_args(oracle, K, st):
    S = oracle.expand_boundary(st["m"].s)
    return S, dict(dt=float(K.dt), dx=st["m"].dx, dz=st["m"].dz, aperture=30.0, da=float(K.da), nang=K.nang)


def test_tables_are_the_oracle_solves(oracle, setup):
    st = setup
    S = oracle.expand_boundary(st["m"].s)
    for k in (0, 3):
        T = oracle.solve_iso(S, st["m"].dx, st["m"].dz, float(st["xs"][k]), 0.0)
        assert np.array_equal(st["ts"][k], T)


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("nt,dt", [(1001, 1e-3), (64, 2e-3)])
def test_convolution_bit_exact(oracle, setup, torch, adjoint, nt, dt):
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], mig.IMAGE, nt=nt, dt=dt, tables=(st["ts"], st["tr"]))
    rng = np.random.default_rng(nt)
    x = rng.standard_normal((K.ntr, nt)).astype(np.float32)
    got = K.convolve(torch.from_numpy(x).cuda(), adjoint).cpu().numpy()
    assert np.array_equal(got, oracle.trace_convolve(x, K.wavelet, adjoint))
    K.close()


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("nt,dt,fmax", [(1001, 1e-3, 2.0),       # wavelet (3542) longer than the trace, in LDS
                                        (16000, 1e-3, 30.0),     # trace and wavelet just fit LDS
                                        (17000, 1e-3, 30.0)])    # neither: the global-memory kernel
def test_convolution_bit_exact_every_kernel(oracle, torch, adjoint, nt, dt, fmax):
    import ctypes as C
    from seisfat2d_amd import capi
    w = mig.ricker(dt, fmax)
    rng = np.random.default_rng(nt)
    x = rng.standard_normal((3, nt)).astype(np.float32)
    xi = torch.from_numpy(x).cuda()
    out = torch.empty_like(xi)
    capi.check(capi.lib().seisfat_trace_convolve(int(adjoint), 3, nt, capi._ptr(w), len(w), C.c_void_p(xi.data_ptr()),
                                                 C.c_void_p(out.data_ptr()), None))
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), oracle.trace_convolve(x, w, adjoint))


# (aperture, dt, nt): the sample case; a negative aperture (negative taper
# divisors: IEEE division for (x - cmp) / sigma); a time step above 1 s (the
# time index by IEEE division below 2^-100); the longest record
@pytest.mark.parametrize("aperture,dt,nt", [(30.0, 2e-3, 420), (-30.0, 2e-3, 420), (30.0, 1.25, 3),
                                              (30.0, 5e-5, 16384)])
def test_image_adjoint_matches_oracle(oracle, setup, torch, aperture, dt, nt):
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], mig.IMAGE, nt=nt, dt=dt, aperture=aperture,
             tables=(st["ts"], st["tr"]))
    assert K.ntr > 20
    S, op = orc_args(oracle, K, st)
    op["aperture"] = aperture
    rng = np.random.default_rng(5)
    d = rng.standard_normal((K.ntr, K.nt)).astype(np.float32)
    m0 = rng.standard_normal(K.model_shape).astype(np.float32) * 1e-3
    got = K.adjoint(torch.from_numpy(d).cuda(), torch.from_numpy(m0.copy()).cuda()).cpu().numpy()
    want = oracle.kdm(0, True, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, None, d, m0.copy(), **op)
    assert np.abs(want).max() > 1e-3
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
    K.close()


@pytest.mark.parametrize("nt", [420, 5000, 9000, 16384])   # 16384: the largest record (a 64 KB LDS histogram)
@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_forward_matches_oracle(oracle, setup, torch, domain, nt):
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], domain, nt=nt, tables=(st["ts"], st["tr"]))
    S, op = orc_args(oracle, K, st)
    rng = np.random.default_rng(7 + domain)
    m = rng.standard_normal(K.model_shape).astype(np.float32)
    d0 = rng.standard_normal((K.ntr, K.nt)).astype(np.float32) * 1e-4
    cid = K.cmp_id if domain == mig.ANGLE else None
    got = K.forward(torch.from_numpy(m).cuda(), torch.from_numpy(d0.copy()).cuda()).cpu().numpy()
    want = oracle.kdm(domain, False, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid, d0.copy(), m, **op)
    bound = oracle.kdm(domain, False, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid, np.abs(d0), np.abs(m), **op)
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert np.abs(want).max() > 0
    if domain == mig.IMAGE:
        assert not bad.any(), np.argwhere(bad)[:5]
    else:
        assert bad.mean() <= 1e-3, bad.sum()
    K.close()


def test_angle_adjoint_matches_oracle(oracle, setup, torch):
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], mig.ANGLE, tables=(st["ts"], st["tr"]))
    S, op = orc_args(oracle, K, st)
    assert K.model_shape == (K.ncmp, K.nang, 48) and K.nang == 21
    rng = np.random.default_rng(9)
    d = rng.standard_normal((K.ntr, K.nt)).astype(np.float32)
    got = K.adjoint(torch.from_numpy(d).cuda()).cpu().numpy()
    want = oracle.kdm(1, True, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, K.cmp_id, d,
                      np.zeros(K.model_shape, np.float32), **op)
    bound = oracle.kdm(1, True, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, K.cmp_id, np.abs(d),
                       np.zeros(K.model_shape, np.float32), **op)
    assert np.abs(want).max() > 0
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert bad.mean() <= 1e-3, bad.sum()
    g, w = got.sum(axis=1, dtype=np.float64), want.sum(axis=1, dtype=np.float64)
    assert np.abs(g - w).max() <= 1e-5 * bound.sum(axis=1).max()
    K.close()


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_dot_product(setup, torch, domain):
    """<L m, d> = <m, L^T d>: the reference's adjointness test of its
    operators (src/migration/migration.cu:282-396, without the convolutions).
    Both sides sum products of random signs, so they cancel: the float32
    rounding of L m and L^T d is bounded against <L|m|, |d|> (the sum of the
    terms' magnitudes), not against |a| + |b|."""
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], domain, tables=(st["ts"], st["tr"]))
    g = torch.Generator(device="cuda").manual_seed(3)
    m = torch.randn(K.model_shape, device="cuda", generator=g)
    d = torch.randn((K.ntr, K.nt), device="cuda", generator=g)
    Lm = K.forward(m)
    Ltd = K.adjoint(d)
    a = torch.sum(Lm.double() * d.double()).item()
    b = torch.sum(m.double() * Ltd.double()).item()
    scale = torch.sum(K.forward(m.abs()).double() * d.abs().double()).item()
    assert scale > 0 and abs(a - b) <= 1e-5 * scale, (a, b, scale)
    K.close()


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_migration_matches_oracle(oracle, setup, torch, domain):
    """KDM::kirchhoff_depth_migration: adjoint convolution of every trace,
    then the adjoint operator (IDKDM / ADKDM)."""
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], domain, tables=(st["ts"], st["tr"]))
    S, op = orc_args(oracle, K, st)
    rng = np.random.default_rng(13)
    seismic = rng.standard_normal((K.nsrc, K.nrec, K.nt)).astype(np.float32)
    got = K.migrate(seismic).cpu().numpy()
    d = np.ascontiguousarray(oracle.trace_convolve(seismic[K.src, K.rec], K.wavelet, True))
    cid = K.cmp_id if domain == mig.ANGLE else None
    want = oracle.kdm(domain, True, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid, d,
                      np.zeros(K.model_shape, np.float32), **op)
    bound = oracle.kdm(domain, True, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid, np.abs(d),
                       np.zeros(K.model_shape, np.float32), **op)
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert bad.mean() <= (0 if domain == mig.IMAGE else 1e-3), bad.sum()
    K.close()


@pytest.mark.parametrize("domain,smooth", [(mig.IMAGE, 0.0), (mig.ANGLE, 1e-3)])
def test_least_squares_migration_matches_oracle(oracle, setup, torch, domain, smooth):
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], domain, tables=(st["ts"], st["tr"]))
    S, op = orc_args(oracle, K, st)
    # consistent data: the forward model of a reflector
    cid = K.cmp_id if domain == mig.ANGLE else None
    m_true = np.zeros(K.model_shape, np.float32)
    m_true[..., 30] = 1.0
    d = oracle.kdm(domain, False, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid,
                   np.zeros((K.ntr, K.nt), np.float32), m_true, **op)
    dobs = oracle.trace_convolve(d, K.wavelet, False)
    seismic = np.zeros((K.nsrc, K.nrec, K.nt), np.float32)
    seismic[K.src, K.rec] = dobs
    got, res = K.lsm(seismic, max_it=3, smooth=smooth)
    want, wres = oracle.lskdm(domain, S, st["ts"], st["tr"], K.src, K.rec, K.cmp, cid, dobs, K.wavelet, 3, smooth,
                              op["dt"], op["dx"], op["dz"], op["aperture"], K.model_shape, op["da"], op["nang"])
    got = got.cpu().numpy()
    assert len(res) == len(wres) == 4
    assert np.allclose(res, wres, rtol=1e-4, atol=0), (res, wres)
    assert res[-1] < res[0]
    if domain == mig.IMAGE:
        assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max()
    else:   # a contribution moved to the neighbouring angle bin spreads over the later iterations
        assert np.linalg.norm(got - want) <= 1e-3 * np.linalg.norm(want)
    K.close()


def test_argument_errors(setup, torch):
    import ctypes as C
    from seisfat2d_amd import capi
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], mig.IMAGE, tables=(st["ts"], st["tr"]))
    with pytest.raises(ValueError):
        K.adjoint(torch.zeros((K.ntr, K.nt + 1), device="cuda"))
    with pytest.raises(ValueError):
        K.forward(torch.zeros((3, 3), device="cuda"))
    with pytest.raises(ValueError):
        make(st["e"], st["m"], st["xs"], st["xr"], mig.IMAGE, tables=(st["ts"][:2], st["tr"]))
    # trace indices out of range, a table index out of range, operators before any table
    bad = np.array([0, 99], np.int32)
    rc = capi.lib().seisfat_kdm_set_traces(K._k, 2, capi._ptr(bad), capi._ptr(np.zeros(2, np.int32)),
                                           capi._ptr(np.zeros(2, np.float32)), None)
    assert rc == capi.EINVAL and "out of range" in capi.lib().seisfat_last_error().decode()
    assert capi.lib().seisfat_kdm_set_table(K._k, 1, K.nrec, C.c_void_p(1), None) == capi.EINVAL
    K.close()
    e = st["e"]
    for params, msg in (((mig.IMAGE, 0, 1e-3, 30.0, 1.0, 1, 1), "nt"), ((7, 100, 1e-3, 30.0, 1.0, 1, 1), "domain"),
                        ((mig.ANGLE, 100, 1e-3, 30.0, 1.0, 0, 4), "angle domain"),
                        ((mig.IMAGE, 100, -1e-3, 30.0, 1.0, 1, 1), "dt")):
        h = C.c_void_p()
        p = capi.KdmParams(*params)
        assert capi.lib().seisfat_kdm_create(e._h, C.byref(p), 2, 3, C.byref(h)) == capi.EINVAL
        assert msg in capi.lib().seisfat_last_error().decode()
    h = C.c_void_p()
    p = capi.KdmParams(mig.IMAGE, 100, 1e-3, 30.0, 1.0, 1, 1)
    capi.check(capi.lib().seisfat_kdm_create(e._h, C.byref(p), 2, 3, C.byref(h)))
    d = torch.zeros((1, 100), device="cuda")
    m = torch.zeros((e.nx, e.nz), device="cuda")
    assert capi.lib().seisfat_kdm_adjoint(h, C.c_void_p(d.data_ptr()), C.c_void_p(m.data_ptr()), None) == capi.ESTATE
    capi.lib().seisfat_kdm_destroy(h)


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_adjoint_over_several_block_parts(oracle, setup, torch, domain):
    """13 sources: four source blocks, which the adjoint spreads over several
    waves per chunk (partial images added in order in the image domain)."""
    st = setup
    e = st["e"]
    xs = np.linspace(20.0, 810.0, 13).astype(np.float32)
    ts = e.traveltime_tables(xs, np.zeros_like(xs))
    K = make(e, st["m"], xs, st["xr"], domain, tables=(ts, st["tr"]))
    S, op = orc_args(oracle, K, st)
    cid = K.cmp_id if domain == mig.ANGLE else None
    rng = np.random.default_rng(41)
    d = rng.standard_normal((K.ntr, K.nt)).astype(np.float32)
    m0 = (rng.standard_normal(K.model_shape) * 1e-3).astype(np.float32) if domain == mig.IMAGE else \
        np.zeros(K.model_shape, np.float32)
    got = K.adjoint(torch.from_numpy(d).cuda(), torch.from_numpy(m0.copy()).cuda()).cpu().numpy()
    want = oracle.kdm(domain, True, S, ts, st["tr"], K.src, K.rec, K.cmp, cid, d, m0.copy(), **op)
    bound = oracle.kdm(domain, True, S, ts, st["tr"], K.src, K.rec, K.cmp, cid, np.abs(d), np.abs(m0), **op)
    assert np.abs(want).max() > 0
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert bad.mean() <= (0 if domain == mig.IMAGE else 1e-3), bad.sum()
    # the same adjoint twice: the image domain is deterministic
    again = K.adjoint(torch.from_numpy(d).cuda(), torch.from_numpy(m0.copy()).cuda()).cpu().numpy()
    if domain == mig.IMAGE:
        assert np.array_equal(again, got)
    K.close()


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_sums_outside_the_fast_division_range(oracle, setup, torch, domain):
    """Traveltime sums the known-divisor division does not serve: the first
    source table shifted down by 4 ms (negative sums near that source, nodes
    the reference's negative index leaves out) and a receiver on every source
    (zero-offset traces: sum 0 at the other sources' nodes, index 0).  The
    waves holding such a sum take the IEEE path; the results match the
    oracle."""
    st = setup
    xr = np.sort(np.concatenate([st["xr"], st["xs"]])).astype(np.float32)
    e = st["e"]
    ts = st["ts"].copy()
    ts[0] -= np.float32(4e-3)
    assert (ts[1:, 3:-3, 3:-3] == 0).sum() == len(ts) - 1      # sources on grid nodes
    tr = e.traveltime_tables(xr, np.zeros_like(xr))
    K = make(e, st["m"], st["xs"], xr, domain, tables=(ts, tr))
    assert (K.src.size > 0) and np.any(st["xs"][K.src] == xr[K.rec])
    S, op = orc_args(oracle, K, st)
    cid = K.cmp_id if domain == mig.ANGLE else None
    rng = np.random.default_rng(31)
    d = rng.standard_normal((K.ntr, K.nt)).astype(np.float32)
    zero = np.zeros(K.model_shape, np.float32)
    got = K.adjoint(torch.from_numpy(d).cuda()).cpu().numpy()
    want = oracle.kdm(domain, True, S, ts, tr, K.src, K.rec, K.cmp, cid, d, zero.copy(), **op)
    bound = oracle.kdm(domain, True, S, ts, tr, K.src, K.rec, K.cmp, cid, np.abs(d), zero.copy(), **op)
    assert np.abs(want).max() > 0
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert bad.mean() <= (0 if domain == mig.IMAGE else 1e-3), bad.sum()
    m = rng.standard_normal(K.model_shape).astype(np.float32)
    d0 = np.zeros((K.ntr, K.nt), np.float32)
    got = K.forward(torch.from_numpy(m).cuda()).cpu().numpy()
    want = oracle.kdm(domain, False, S, ts, tr, K.src, K.rec, K.cmp, cid, d0.copy(), m, **op)
    bound = oracle.kdm(domain, False, S, ts, tr, K.src, K.rec, K.cmp, cid, d0.copy(), np.abs(m), **op)
    bad = np.abs(got - want) > 1e-5 * bound + 1e-30
    assert bad.mean() <= (0 if domain == mig.IMAGE else 1e-3), bad.sum()
    K.close()


def test_tables_follow_the_slowness(oracle, setup, torch):
    """The table quantities hold the slowness they were evaluated with: after
    a slowness upload the operators refuse to run until every table is set
    again, and then weigh with the new slowness (the oracle on the new S)."""
    import ctypes as C
    from seisfat2d_amd import capi
    from seisfat2d_amd.capi import SeisfatError
    st = setup
    m = st["m"]
    e = Eikonal(m.s.shape[1], m.s.shape[0], m.dz, m.dx)
    try:
        e.set_slowness(m.s)
        K = make(e, m, st["xs"], st["xr"], mig.IMAGE, tables=(st["ts"], st["tr"]))
        d = torch.from_numpy(np.random.default_rng(21).standard_normal((K.ntr, K.nt)).astype(np.float32)).cuda()
        m1 = K.adjoint(d).cpu().numpy()
        s2 = (m.s * 1.25).astype(np.float32)
        e.set_slowness(s2)
        with pytest.raises(SeisfatError) as ex:
            K.adjoint(d)
        assert ex.value.code == capi.ESTATE and "slowness changed" in str(ex.value)
        ts = torch.from_numpy(np.ascontiguousarray(st["ts"], np.float32)).cuda()
        tr = torch.from_numpy(np.ascontiguousarray(st["tr"], np.float32)).cuda()
        # all but the last receiver table: still refused
        for which, tabs, n in ((0, ts, K.nsrc), (1, tr, K.nrec - 1)):
            for k in range(n):
                capi.check(capi.lib().seisfat_kdm_set_table(K._k, which, k, C.c_void_p(tabs[k].data_ptr()), None))
        with pytest.raises(SeisfatError) as ex:
            K.adjoint(d)
        assert ex.value.code == capi.ESTATE and "tables not set" in str(ex.value)
        capi.check(capi.lib().seisfat_kdm_set_table(K._k, 1, K.nrec - 1, C.c_void_p(tr[-1].data_ptr()), None))
        got = K.adjoint(d).cpu().numpy()
        _, op = orc_args(oracle, K, st)
        S2 = oracle.expand_boundary(s2)
        want = oracle.kdm(0, True, S2, st["ts"], st["tr"], K.src, K.rec, K.cmp, None, d.cpu().numpy(),
                          np.zeros(K.model_shape, np.float32), **op)
        assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()
        assert np.abs(got - m1).max() > 1e-3 * np.abs(m1).max()   # the slowness entered the weights
        # back to the first slowness, every table again (Kirchhoff.set_tables):
        # the first image, bit for bit
        e.set_slowness(m.s)
        K.set_tables(ts, tr)
        assert np.array_equal(K.adjoint(d).cpu().numpy(), m1)
        K.close()
    finally:
        e.close()


def test_no_traces_within_the_offset(setup, torch):
    """A maximum offset that keeps no pair: no traces, a zero image, a
    zero-trace forward."""
    st = setup
    K = make(st["e"], st["m"], st["xs"], st["xr"], mig.IMAGE, max_offset=1.0, tables=(st["ts"], st["tr"]))
    assert K.ntr == 0
    seismic = np.ones((K.nsrc, K.nrec, K.nt), np.float32)
    img = K.migrate(seismic)
    assert img.shape == K.model_shape and not img.any()
    assert tuple(K.forward(torch.ones(K.model_shape, device="cuda")).shape) == (0, K.nt)
    K.close()


# the table setup's usual path and its general one (traveltimes that are zero,
# tiny, huge or not finite, whole tables or single nodes), rows that wrap inside
# a chunk (nz below, at and above 64, no multiple of it), both domains
@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
@pytest.mark.parametrize("nz,nx,scale,spoil", [(5, 41, 1.0, None), (64, 33, 1.0, None), (65, 40, 1e-12, None),
                                               (131, 30, 1.0, 0.0), (70, 30, 1.0, np.inf), (70, 30, 1.0, np.nan),
                                               (70, 30, 1.0, 1e30)])
def test_table_setup_paths(oracle, torch, domain, nz, nx, scale, spoil):
    m, xs, xr = survey(nz=nz, nx=nx, nsrc=3, nrec=9, seed=nz)
    e = Eikonal(nz, nx, m.dz, m.dx)
    e.set_slowness(m.s)
    ts, tr = (scale * e.traveltime_tables(x, np.full_like(x, 11.0)) for x in (xs, xr))
    ts, tr = ts.astype(np.float32), tr.astype(np.float32)
    if spoil is not None:
        ts[1, 20, nz // 2], tr[4, 12:14, nz // 3] = spoil, spoil
    K = make(e, m, xs, xr, domain, nt=300, dt=1e-3, tables=(ts, tr), max_offset=400.0)
    S = oracle.expand_boundary(m.s)
    op = dict(dt=float(K.dt), dx=m.dx, dz=m.dz, aperture=30.0, da=float(K.da), nang=K.nang)
    d = np.random.default_rng(3).standard_normal((K.ntr, K.nt)).astype(np.float32)
    cid = K.cmp_id if domain == mig.ANGLE else None
    got = K.adjoint(torch.from_numpy(d).cuda()).cpu().numpy()
    want = oracle.kdm(domain, True, S, ts, tr, K.src, K.rec, K.cmp, cid, d, np.zeros(K.model_shape, np.float32), **op)
    fin = np.isfinite(want)
    assert np.array_equal(fin, np.isfinite(got))
    bad = np.abs(got - want)[fin] > 1e-5 * np.abs(want[fin]).max()
    assert bad.mean() <= (1e-3 if domain == mig.ANGLE else 0.0)
    K.close()
    e.close()


# the register-blocked convolution at the edges of its groups of 8, segments of
# 2048, traces per workgroup and taps per upload (896), and the direct kernel
# for a wavelet that is too long or not finite
@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("ntr,nt,nw", [(1, 1, 1), (70, 7, 9), (33, 8, 16), (3, 1023, 895), (5, 1024, 896), (3, 2047, 897),
                                       (2, 2048, 8), (2, 2049, 7), (2, 4100, 1793), (2, 300, 13000), (4, 50, -20)])
def test_convolution_block_edges(oracle, torch, adjoint, ntr, nt, nw):
    import ctypes as C
    from seisfat2d_amd import capi
    rng = np.random.default_rng(nt + abs(nw))
    w = rng.standard_normal(abs(nw)).astype(np.float32)
    if nw < 0:
        w[3] = np.inf
    x = rng.standard_normal((ntr, nt)).astype(np.float32)
    xi = torch.from_numpy(x).cuda()
    out = torch.empty_like(xi)
    capi.check(capi.lib().seisfat_trace_convolve(int(adjoint), ntr, nt, capi._ptr(w), len(w), C.c_void_p(xi.data_ptr()),
                                                 C.c_void_p(out.data_ptr()),
                                                 C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert np.array_equal(out.cpu().numpy(), oracle.trace_convolve(x, w, adjoint), equal_nan=True)


# the forward's tile kernel at the edges of its tiles (64 rows, 16 or 8
# columns), windows longer than its 1024 samples (several rounds), slices of a
# block's entries, NaN and negative traveltimes (indices 0 and skipped), and the
# trace kernel on the same survey under capture
@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
@pytest.mark.parametrize("nz,nx,nt,dt,shift", [(63, 33, 400, 2e-3, 0.0), (64, 32, 400, 2e-3, 0.0), (65, 31, 16384, 2e-5, 0.0),
                                               (130, 49, 3000, 2e-4, 0.0), (70, 40, 400, 1.5e-3, -0.05),
                                               (70, 40, 500, 1.5e-3, np.nan)])
def test_forward_tiles(oracle, torch, domain, nz, nx, nt, dt, shift):
    m, xs, xr = survey(nz=nz, nx=nx, nsrc=9, nrec=60, seed=nz)
    e = Eikonal(nz, nx, m.dz, m.dx)
    e.set_slowness(m.s)
    ts, tr = (e.traveltime_tables(x, np.full_like(x, 11.0)) for x in (xs, xr))
    if np.isnan(shift):
        ts[2, 20, 30], tr[5, 11, 40:43] = np.nan, np.nan
    else:
        tr += np.float32(shift)
    K = make(e, m, xs, xr, domain, nt=nt, dt=dt, tables=(ts, tr), max_offset=1e4)
    S = oracle.expand_boundary(m.s)
    op = dict(dt=float(K.dt), dx=m.dx, dz=m.dz, aperture=30.0, da=float(K.da), nang=K.nang)
    rng = np.random.default_rng(nz)
    x = rng.standard_normal(K.model_shape).astype(np.float32)
    d0 = (rng.standard_normal((K.ntr, nt)) * 1e-4).astype(np.float32)
    cid = K.cmp_id if domain == mig.ANGLE else None
    xd = torch.from_numpy(x).cuda()
    K.adjoint(torch.zeros((K.ntr, nt), device="cuda"))
    out = [torch.from_numpy(d0.copy()).cuda() for _ in range(2)]
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.forward(xd, out[1])
    K.forward(xd, out[0])
    g.replay()
    want = oracle.kdm(domain, False, S, ts, tr, K.src, K.rec, K.cmp, cid, d0.copy(), x, **op)
    bound = oracle.kdm(domain, False, S, ts, tr, K.src, K.rec, K.cmp, cid, np.abs(d0), np.abs(x), **op)
    fin = np.isfinite(want)
    for got in out:
        got = got.cpu().numpy()
        assert np.array_equal(np.isfinite(got), fin)
        bad = np.abs(got - want)[fin] > (1e-5 * bound + 1e-30)[fin]
        assert bad.mean() <= (1e-3 if domain == mig.ANGLE else 0.0)
    K.close()
    e.close()


@pytest.mark.parametrize("n,chunk", [(0, 3), (1, 3), (3, 3), (7, 3)])
def test_device_tables_are_the_host_tables(torch, n, chunk):
    """The constructor's tables, solved into device memory batch by batch,
    equal traveltime_tables bit for bit (batches partly filled, and none)."""
    from seisfat2d_amd import Eikonal, models
    w = models.rough(41, 77, 10.0, 10.0, seed=5, sigma=3.0, vlo=2000.0, vhi=3000.0)
    e = Eikonal(41, 77, 10.0, 10.0)
    e.set_slowness(w.s)
    x = np.linspace(0.0, 700.0, n)
    want = e.traveltime_tables(x, 0.0 * x, chunk=chunk)
    got = e._device_tables(x, 0.0 * x, chunk=chunk)
    assert got.is_cuda and got.dtype == torch.float32 and tuple(got.shape) == want.shape == (n, 83, 47)
    assert np.array_equal(got.cpu().numpy(), want)
    e.close()


# the forward's tile kernel, which a survey needs about 300 traces per tile and
# block to be given (200 sources, 240 receivers): rows and columns at and beside
# its tiles' edges, one slice of a block's entries and several, more entries than
# one list, and tables that hold negative, NaN and finite or infinite "not
# reached" values (1e30; 1e6 in a source and a receiver table), whose tiles'
# windows end with the record and take several rounds of its 1024 samples.
# Traces over the whole survey are compared, and those around the spoiled tables.
@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
@pytest.mark.parametrize("nz,nx,nt,dt,shift,spoil", [
    (63, 97, 400, 2e-3, 0.0, None), (64, 96, 400, 2e-3, 0.0, None), (65, 98, 900, 4e-4, 0.0, None),
    (65, 98, 400, 2e-3, -0.05, 1e30), (130, 49, 700, 1e-3, 0.0, np.nan), (65, 98, 2100, 3.5e-4, 0.0, 1e30),
    (65, 98, 2100, 3.5e-4, -0.05, 1e6), (65, 98, 900, 4e-4, 0.0, np.inf)])
def test_forward_by_tiles(oracle, torch, domain, nz, nx, nt, dt, shift, spoil):
    m, xs, xr = survey(nz=nz, nx=nx, nsrc=200, nrec=240, seed=nz)
    e = Eikonal(nz, nx, m.dz, m.dx)
    e.set_slowness(m.s)
    ts, tr = (e.traveltime_tables(x, np.full_like(x, 11.0)) for x in (xs, xr))
    tr += np.float32(shift)
    if spoil is not None:
        z = 25 if spoil == 1e6 else 35  # (where gradients are huge, no node beside both)
        ts[70, 20:60, 30], tr[100, 30:44, z:z + 15] = spoil, spoil
    K = make(e, m, xs, xr, domain, nt=nt, dt=dt, tables=(ts, tr), max_offset=1e4)
    S = oracle.expand_boundary(m.s)
    op = dict(dt=float(K.dt), dx=m.dx, dz=m.dz, aperture=30.0, da=float(K.da), nang=K.nang)
    rng = np.random.default_rng(nz)
    x = rng.standard_normal(K.model_shape).astype(np.float32)
    got = torch.zeros((K.ntr, nt), device="cuda")
    K.forward(torch.from_numpy(x).cuda(), got)
    sub = np.arange(K.ntr)
    near = (np.abs(K.src - 70) <= 1) & (np.abs(K.rec - 100) <= 6) | (sub % 997 == 0) | (sub >= K.ntr - 2)
    sub = sub[near]
    assert 60 <= len(sub) <= 120
    got = got.cpu().numpy()[sub]
    cid = None if domain == mig.IMAGE else K.cmp_id[sub]
    a = (domain, False, S, ts, tr, K.src[sub], K.rec[sub], K.cmp[sub], cid)
    want = oracle.kdm(*a, np.zeros((len(sub), nt), np.float32), x, **op)
    bound = oracle.kdm(*a, np.zeros((len(sub), nt), np.float32), np.abs(x), **op)
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin)
    bad = np.abs(got - want)[fin] > (1e-5 * bound + 1e-30)[fin]
    assert bad.mean() <= (1e-3 if domain == mig.ANGLE else 0.0)
    K.close()
    e.close()


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_captured_forward_follows_the_tables(torch, domain):
    """A forward captured after an eager one (which took the tile kernel)
    replays with the tables set since, and an eager one follows tables that a
    replay has set."""
    nz, nx, nt, dt = 65, 98, 400, 2e-3
    m, xs, xr = survey(nz=nz, nx=nx, nsrc=200, nrec=240, seed=nz)
    e = Eikonal(nz, nx, m.dz, m.dx)
    e.set_slowness(m.s)
    ts, tr = (torch.from_numpy(e.traveltime_tables(x, np.full_like(x, 11.0))).cuda() for x in (xs, xr))
    K = make(e, m, xs, xr, domain, nt=nt, dt=dt, tables=(ts, tr), max_offset=1e4)
    x = torch.rand(K.model_shape, device="cuda") + 0.5
    K.forward(x)
    out = torch.zeros((K.ntr, nt), device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.forward(x, out)
    for shift in (0.2, -0.05, 0.0):
        K.set_tables(ts, tr + shift)
        out.zero_()
        g.replay()
        want = K.forward(x)
        torch.cuda.synchronize()
        assert bool(want.abs().max() > 0)
        assert float((out - want).abs().max()) <= 1e-4 * float(want.abs().max()), shift
    rec = tr.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.set_tables(ts, rec)
    K.set_tables(ts, rec)
    K.forward(x)
    for shift in (0.2, 0.1):
        rec.copy_(tr + shift)
        g.replay()
        got = K.forward(x)
        K.set_tables(ts, tr + shift)
        want = K.forward(x)
        assert float((got - want).abs().max()) <= 1e-4 * float(want.abs().max()), shift
        rec.copy_(tr)
        K.set_tables(ts, rec)
        K.forward(x)
    K.close()
    e.close()


@pytest.mark.parametrize("domain", [mig.IMAGE, mig.ANGLE])
def test_adjoint_knows_negative_receiver_tables_on_any_stream(torch, domain):
    """Whether a source may be passed over on its own traveltimes depends on
    the receivers' being non-negative: as the tables stand, also for an
    adjoint on a second stream and for a captured one replayed."""
    nz, nx, nt, dt = 64, 90, 100, 1e-3
    m, xs, xr = survey(nz=nz, nx=nx, nsrc=3, nrec=50, seed=2)
    e = Eikonal(nz, nx, m.dz, m.dx)
    e.set_slowness(m.s)
    ts, tr = (torch.from_numpy(e.traveltime_tables(x, np.full_like(x, 11.0))).cuda() for x in (xs, xr))
    K = make(e, m, xs, xr, domain, nt=nt, dt=dt, tables=(ts, tr), max_offset=1e4)
    d = torch.rand((K.ntr, nt), device="cuda") + 0.5
    K.adjoint(d)
    captured = torch.zeros(K.model_shape, device="cuda")
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        K.adjoint(d, captured)
    K.set_tables(ts, tr - 0.15)  # sums within the record where the source's time alone is past it
    second, out = torch.cuda.Stream(), torch.zeros(K.model_shape, device="cuda")
    second.wait_stream(torch.cuda.current_stream())
    a = torch.randn(8192, 8192, device="cuda")
    for _ in range(4):  # the first stream's adjoint has yet to start when the second's runs
        torch.mm(a, a)
    late = K.adjoint(d)
    with torch.cuda.stream(second):
        K.adjoint(d, out)
    torch.cuda.synchronize()
    captured.zero_()
    g.replay()
    want = K.adjoint(d)
    torch.cuda.synchronize()
    one_by_one = K.adjoint(d)
    for got in (out, late, captured, one_by_one):
        assert float((got - want).abs().max()) <= 1e-4 * float(want.abs().max())
    # the sources' own times leave nothing of the model beyond the record
    K.set_tables(ts, tr)
    short = K.adjoint(d)
    assert bool((want != 0).sum() > 1.5 * (short != 0).sum())
    K.close()
    e.close()


# wavelets as long as the record and much longer: the register-blocked kernel
# passes over the taps that meet no sample, by wave, with several traces to a
# wave (9, 64), one (100, 512) and several segments (2100, 6000); one that leaves
# no output beyond its shift
@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("ntr,nt,nw", [(70, 9, 5000), (33, 64, 700), (3, 100, 13000), (5, 512, 513), (2, 2100, 9000),
                                       (2, 6000, 10384), (1, 40, 13640)])
def test_convolution_wavelet_longer_than_the_record(oracle, torch, adjoint, ntr, nt, nw):
    import ctypes as C
    from seisfat2d_amd import capi
    rng = np.random.default_rng(nt + nw)
    w = rng.standard_normal(nw).astype(np.float32)
    x = rng.standard_normal((ntr, nt)).astype(np.float32)
    xi = torch.from_numpy(x).cuda()
    out = torch.full_like(xi, 7.0)
    capi.check(capi.lib().seisfat_trace_convolve(int(adjoint), ntr, nt, capi._ptr(w), nw, C.c_void_p(xi.data_ptr()),
                                                 C.c_void_p(out.data_ptr()),
                                                 C.c_void_p(torch.cuda.current_stream().cuda_stream)))
    assert np.array_equal(out.cpu().numpy(), oracle.trace_convolve(x, w, adjoint))
