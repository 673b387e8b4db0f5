"""The fused sampler where a dimension, a tile or a launch shape ends: FP64
parity mode against the oracle (the bars of test_gpu_integrator.py)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def va():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import vegas_amd
    return vegas_amd


@pytest.mark.parametrize("dim,neval", [(14, 20000), (15, 20000), (16, 20000), (18, 2000), (24, 2000), (25, 2000),
                                       (40, 1000)])
def test_dims(va, orc, dim, neval):
    """Dimensions of their own up to 16, shared up to 24, and above."""
    c = [0.5 + 0.02 * ((d % 3) - 1) for d in range(dim)]
    f, fo = va.GaussianMixture([1.0], [8.0], [c]), orc.GaussMix([1.0], [8.0], [c])
    integ = va.Integrator([[0, 1]] * dim, neval=neval, seed=23, precision='f64', exact=True)
    r = integ(f, nitn=1)
    o = orc.OracleIntegrator([(0, 1)] * dim, neval=neval, seed=23)
    mean, var, nev = o.run(fo, 1)
    m = r.itn_results[0]
    assert integ.last_neval == nev[0]
    assert abs(m.mean - mean[0]) <= 1e-12 * abs(mean[0])
    assert abs(m.var - var[0]) <= 1e-10 * var[0]
    np.testing.assert_allclose(integ.sigf, o.sigf, rtol=1e-11)
    np.testing.assert_allclose(integ.map.grid, o.map.grid, rtol=1e-11, atol=1e-13)

    @va.lbatchintegrand
    def fl(x):
        return np.exp(-8.0 * ((x - np.array(c)) ** 2).sum(1))

    ra = va.Integrator([[0, 1]] * dim, neval=neval, seed=29, precision='f32')(f, nitn=1).itn_results[0]
    rb = va.Integrator([[0, 1]] * dim, neval=neval, seed=29, precision='f32')(fl, nitn=1).itn_results[0]
    assert abs(ra.mean - rb.mean) <= 2e-5 * abs(rb.mean)
    assert abs(ra.sdev - rb.sdev) <= 1e-3 * rb.sdev


@pytest.mark.parametrize("dim", [1, 4, 9])
@pytest.mark.parametrize("neval", [100, 2000, 4 * 256 * 256 - 1000, 4 * 256 * 256 + 50000, 8 * 256 * 256 + 50000])
@pytest.mark.parametrize("mode", ["parity", "f32", "unordered"])
def test_few_tiles(va, orc, dim, neval, mode):
    """From less than one tile, over one and two rounds of tiles per
    workgroup, to the launch shape of many: two iterations in parity mode;
    otherwise the oracle with the same 24-bit uniforms (FP32 bars)."""
    c = [0.5 + 0.02 * ((d % 3) - 1) for d in range(dim)]
    f, fo = va.GaussianMixture([1.0], [8.0], [c]), orc.GaussMix([1.0], [8.0], [c])
    kw = dict(precision='f64', exact=True) if mode == "parity" else dict(precision='f32',
                                                                         deterministic=mode == "f32")
    integ = va.Integrator([[0, 1]] * dim, neval=neval, seed=31, **kw)
    r = integ(f, nitn=2 if mode == "parity" else 1)
    o = orc.OracleIntegrator([(0, 1)] * dim, neval=neval, seed=31, rng_f32=mode != "parity")
    mean, var, nev = o.run(fo, len(r.itn_results))
    assert integ.last_neval == nev[-1]
    rm, rv, rg = (1e-12, 1e-10, 1e-11) if mode == "parity" else (2e-5, 2e-3, 1e-3)
    for m, mo, vo in zip(r.itn_results, mean, var):
        assert abs(m.mean - mo) <= rm * abs(mo)
        assert abs(m.var - vo) <= rv * vo
    np.testing.assert_allclose(integ.map.grid, o.map.grid, rtol=rg, atol=1e-13)


@pytest.mark.parametrize("nc,dim,neval,kind", [(256, 5, 4200000, "zeros"), (257, 12, 4200000, "plain"),
                                               (258, 8, 4200000, "negative"), (259, 7, 4200000, "wide"),
                                               (259, 6, 4200000, "huge"), (255, 8, 4200000, "plain"),
                                               (259, 4, 4200000, "plain"), (259, 13, 4200000, "plain")])
def test_long_mixture(va, nc, dim, neval, kind):
    """The long mixtures' loop and its neighbours, with every remainder of its
    steps, against FP64 terms at the same points (FP32 bars)."""
    import torch
    rng = np.random.default_rng(nc)
    sigma = 0.4 if kind == "wide" else 0.03 * np.sqrt(dim)
    f32 = lambda a: np.asarray(a, np.float32).astype(np.float64)
    A = f32(rng.uniform(0.5, 1.5, nc) * (1e30 if kind == "huge" else 1.0))
    if kind == "zeros":
        A[::3] = 0.0
        A[-1] = 0.0
    if kind == "negative":
        A[::5] *= -0.25
    B = f32(0.5 / (sigma * rng.uniform(0.7, 1.3, nc)) ** 2)
    c = f32(np.linspace(0.25, 0.75, nc)[:, None] + rng.uniform(-0.02, 0.02, (nc, dim)))
    f = va.GaussianMixture(A, B, c)
    dA, dB, dc = (torch.as_tensor(a, device="cuda") for a in (A, B, c))

    @va.gpu_lbatchintegrand
    def g(x):
        y = torch.zeros(x.shape[0], dtype=torch.float64, device=x.device)
        for k in range(nc):
            y += dA[k] * torch.exp(-dB[k] * ((x - dc[k]) ** 2).sum(1))
        return y

    ra = va.Integrator([[0, 1]] * dim, neval=neval, seed=29, precision='f32')(f, nitn=1).itn_results[0]
    rb = va.Integrator([[0, 1]] * dim, neval=neval, seed=29, precision='f32')(g, nitn=1).itn_results[0]
    assert abs(ra.mean - rb.mean) <= 2e-5 * abs(rb.mean)
    assert abs(ra.sdev - rb.sdev) <= 1e-3 * rb.sdev


@pytest.mark.parametrize("dim,neval,batch", [(1, 1000, 300), (2, 100, 1), (3, 257 * 12, 256), (4, 200000, 50001),
                                             (8, 300000, 10 ** 9), (16, 5000, 777), (17, 3000, 500), (30, 600, 10 ** 9)])
@pytest.mark.parametrize("precision", ["f64", "f32"])
def test_staged_points(va, dim, neval, batch, precision):
    """Points, weights and hcubes of the staged sampler, over batches that end
    inside and at a workgroup's 256 points, from their own y (1e-12: a few
    roundings of the map and the Jacobian)."""
    integ = va.Integrator([[-1, 2]] * dim, neval=neval, seed=5, min_neval_batch=batch, precision=precision)
    integ(va.GaussianMixture([1.0], [3.0], [[0.4] * dim]), nitn=2)
    parts = list(integ.random_batch(yield_hcube=True, yield_y=True))
    x, y, w, h = (np.concatenate([p[i] for p in parts]) for i in range(4))
    assert len(x) == integ.last_neval and np.all(np.diff(h) >= 0) and h[0] == 0 and h[-1] == integ.nhcube - 1
    ns = np.asarray(integ.nstrat, np.int64)
    own = np.zeros(len(y), np.int64)
    for d in range(dim)[::-1]:  # axis 0 varies fastest
        own = own * ns[d] + np.minimum((y[:, d] * ns[d]).astype(np.int64), ns[d] - 1)
    assert np.mean(own != h) <= 1e-3  # (a y next to a stratum's edge may round over it)
    xm, jac = (np.empty_like(y), np.empty(len(y)))
    integ.map.map(y, xm, jac)
    np.testing.assert_allclose(x, xm, rtol=1e-12, atol=1e-12)
    n_h = np.bincount(h, minlength=integ.nhcube)
    np.testing.assert_allclose(w, jac / integ.nhcube / n_h[h], rtol=1e-12)


@pytest.mark.parametrize("per", [2, 31, 32, 33, 64, 65, 2048, 2049, 5000])
def test_covariance_components(va, per):
    """Every number of components that has its own kernel (1-6) against the
    pairwise kernel (7) and the scalar path, with hcubes on both sides of each
    thread, wave and workgroup border.  The sums differ in their order only
    (per points: 1e-12 covers 5000 roundings of terms that do not cancel)."""
    import torch
    ns = [5, 3]

    def run(m):
        def f(x):
            g = torch.exp(-3.0 * ((x - 0.4) ** 2).sum(1))
            return torch.stack([g * (1 + x[:, 0] * k) * (1 + 0.5 * x[:, 1]) ** k for k in range(m)], 1) if m else g
        integ = va.Integrator([[0, 1], [0, 2]], neval=15 * per, nstrat=ns, beta=0.0, seed=3)
        r = integ(va.gpu_lbatchintegrand(f), nitn=1).itn_results[0]
        assert integ.last_neval == 15 * per
        return r

    full = run(7)
    cov, scale = np.asarray(full.cov), np.sqrt(np.diag(full.cov))
    for m in range(1, 7):
        r = run(m)
        np.testing.assert_allclose(np.asarray(r.mean), np.asarray(full.mean)[:m], rtol=1e-12)
        np.testing.assert_allclose(np.asarray(r.cov) / np.outer(scale[:m], scale[:m]),
                                   cov[:m, :m] / np.outer(scale[:m], scale[:m]), atol=1e-11)
    one = run(0)
    assert abs(one.mean - full.mean[0]) <= 1e-12 * one.mean
    assert abs(one.var - cov[0, 0]) <= 1e-10 * one.var


@pytest.mark.parametrize("dim,neval,batch", [(1, 50, 10 ** 9), (2, 1000, 1), (2, 1000, 2.5), (3, 30000, 7),
                                             (3, 30000, 8), (4, 200000, 49999), (4, 200000, 0), (5, 100000, float('inf')),
                                             (8, 900000, 100000)])
def test_batch_cuts(va, dim, neval, batch):
    """The device's batches (and those of the host beyond its limit) against
    the reference's cut of the same counts."""
    from vegas_amd import _geometry
    integ = va.Integrator([[0, 1]] * dim, neval=neval, seed=5)
    integ(va.GaussianMixture([1.0], [30.0], [[0.4] * dim]), nitn=2)
    integ.min_neval_batch = batch
    parts = [p[2] for p in integ.random_batch(yield_hcube=True)]
    h = np.concatenate(parts)
    cuts = _geometry.batches(np.bincount(h, minlength=integ.nhcube), batch)
    assert [len(p) for p in parts] == [p1 - p0 for _, _, p0, p1 in cuts]
    assert [int(p[0]) for p in parts] == [h0 for h0, _, _, _ in cuts]


@pytest.mark.parametrize("n", [1, 255, 1025, 4096 * 256 + 3])
@pytest.mark.parametrize("m", [1, 2, 3, 7, 300])
def test_batch_values(va, n, m):
    """Component 0 and the NaN flag of a batch, with a NaN in the last value."""
    import torch
    from vegas_amd import _lib
    n = min(n, 4 * 10 ** 6 // m)
    f = torch.rand((n, m), dtype=torch.float64, device='cuda')
    f[n // 2, m // 2] = float('inf')
    f0, flag = torch.empty(n, dtype=torch.float64, device='cuda'), torch.zeros(1, dtype=torch.int32, device='cuda')

    def run(out):
        _lib.check(_lib.lib().vgx_iter_values(_lib.ptr(f), n, m, out, _lib.ptr(flag), _lib.stream_ptr()))

    run(_lib.ptr(f0))
    assert torch.equal(f0, f[:, 0]) and int(flag.item()) == 0
    f[n - 1, m - 1] = float('nan')
    run(None)
    assert int(flag.item()) == 1


@pytest.mark.parametrize("nhcube", [992, 1024, 1056, 8190, 8281])
@pytest.mark.parametrize("beta", [0.75, 0.0])
def test_hcube_counts(va, orc, nhcube, beta):
    """Allocation by one workgroup (up to 8192 hcubes) and by many, on both
    sides of its 1024 threads, with adaptive and equal counts."""
    kw = dict(neval=(8 if beta else 2) * (nhcube + 1), seed=37, beta=beta)
    c = [[0.45, 0.55]]
    f, fo = va.GaussianMixture([1.0], [30.0], c), orc.GaussMix([1.0], [30.0], c)
    integ = va.Integrator([[0, 1]] * 2, precision='f64', exact=True, **kw)
    assert integ.nhcube == nhcube
    r = integ(f, nitn=3)
    o = orc.OracleIntegrator([(0, 1)] * 2, **kw)
    mean, var, nev = o.run(fo, 3)
    for k, m in enumerate(r.itn_results):
        assert abs(m.mean - mean[k]) <= 1e-12 * abs(mean[k])
        assert abs(m.var - var[k]) <= 1e-10 * var[k]
    assert integ.last_neval == nev[-1]
    # the counts of the next iteration, whole numbers, from the weights themselves
    h = np.concatenate([p[2] for p in integ.random_batch(yield_hcube=True)])
    want = np.full(nhcube, 2) if not beta else np.minimum(
        (integ.sigf * (integ.neval_frac * integ.neval / integ.sum_sigf)).astype(np.int64) + integ.min_neval_hcube,
        integ.max_neval_hcube)
    np.testing.assert_array_equal(np.bincount(h, minlength=nhcube), want)


@pytest.mark.parametrize("ns,per", [([1, 1], 33000), ([5, 1], 10000), ([5, 1], 128), ([5, 1], 129), ([40, 26], 32),
                                    ([40, 26], 33), ([40, 26], 130), ([64, 64], 40), ([300, 10], 2100),
                                    ([300, 220], 33)])
def test_covariance_plans(va, ns, per):
    """The launch plans of the covariance kernels (a workgroup per hcube, a few
    hcubes per workgroup, many; all pairs at once or pair by pair) against the
    points' own sums, hcube by hcube, in 64 bits: the sums differ in their
    order only (1e-12 for means; deviations are at least 0.01 of the values, so
    1e-10 for covariances, on the scale of the variances)."""
    import torch
    nh = ns[0] * ns[1]
    kw = dict(neval=nh * per, nstrat=ns, beta=0.0, seed=3, min_neval_batch=10 ** 9)
    region = [[0, 1], [0, 2]]

    def values(x, m):
        g = torch.exp(-3.0 * ((x - 0.4) ** 2).sum(1))
        return torch.stack([g * (1 + x[:, 0] * k) * (1 + 0.5 * x[:, 1]) ** k for k in range(m)], 1)

    for m in (1, 3, 4, 5, 6, 7):
        seen = []

        def f(x):
            seen.append(x.clone())
            return values(x, m)

        integ = va.Integrator(region, **kw)
        r = integ(va.gpu_lbatchintegrand(f), nitn=1).itn_results[0]
        x = seen[-1]
        assert x.shape[0] == nh * per
        # a uniform grid: every weight is the region's volume over the points
        wf = (values(x, m) * (2.0 / (nh * per))).reshape(nh, per, m)
        S = wf.sum(1)
        d = wf - (S / per)[:, None, :]
        mean = S.sum(0)
        cov = (torch.matmul(d.transpose(1, 2).contiguous(), d).sum(0) * (per / (per - 1.0))).cpu().numpy()
        sd = np.sqrt(np.diag(cov))
        np.testing.assert_allclose(np.asarray(r.mean), mean.cpu().numpy(), rtol=1e-12)
        np.testing.assert_allclose(np.asarray(r.cov) / np.outer(sd, sd), cov / np.outer(sd, sd), atol=1e-10)


@pytest.mark.parametrize("dim", [5, 6, 7, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("kind", ["narrow", "wide", "spread"])
def test_long_mixture_same_bits(va, dim, kind):
    """Components of weight 0 change nothing, so 255 of them (the plain loop)
    and the same with 1 to 4 more of weight 0 (the long mixtures' loop, its
    remainders) are one integrand: mean, variance, per-hcube sums, training
    histogram and grid are the same bits, with terms left out or not."""
    rng = np.random.default_rng(dim)
    nc, neval = 255, 4200000
    sigma = 0.4 if kind == "wide" else 0.02 * np.sqrt(dim)
    A = rng.uniform(0.5, 1.5, nc) * (np.exp(rng.uniform(-40, 40, nc)) if kind == "spread" else 1.0)
    B = 0.5 / (sigma * rng.uniform(0.7, 1.3, nc)) ** 2
    c = rng.permutation(np.linspace(0.25, 0.75, nc))[:, None] + rng.uniform(-0.02, 0.02, (nc, dim))

    def run(zeros):
        # the zeros first, in the middle and last
        at = np.sort(rng.integers(0, nc + 1, zeros)) if zeros else []
        f = va.GaussianMixture(np.insert(A, at, 0.0), np.insert(B, at, 50.0), np.insert(c, at, 0.5, axis=0))
        integ = va.Integrator([[0, 1]] * dim, neval=neval, seed=31, precision='f32')
        r = integ(f, nitn=1).itn_results[0]
        return r.mean, r.var, integ.sigf.copy(), integ.map.grid, integ._last_training()

    plain = run(0)
    for zeros in (1, 2, 3, 4):
        many = run(zeros)
        assert many[:2] == plain[:2]
        for a, b in zip(many[2:4] + many[4], plain[2:4] + plain[4]):
            assert np.array_equal(np.asarray(a), np.asarray(b))


def test_long_mixture_few_points(va):
    """A long mixture whose launch has few tiles after all (only 2 points in
    each of 256 hcubes) runs the sampler of few tiles."""
    rng = np.random.default_rng(3)
    c = rng.uniform(0.3, 0.7, (256, 8))

    def run(zeros):
        f = va.GaussianMixture([1.0] * 256 + [0.0] * zeros, [30.0] * (256 + zeros), np.concatenate([c, c[:zeros]]))
        integ = va.Integrator([[0, 1]] * 8, neval=4200000, nstrat=[2] * 8, seed=31, precision='f32', nitn=2)
        integ.neval_frac, integ.min_neval_hcube = 0.0, 2
        r = integ(f).itn_results[-1]
        assert integ.last_neval == 512
        return r.mean, r.var

    assert run(0) == run(3)


@pytest.mark.parametrize("dim", [9, 10, 11, 12, 13])
@pytest.mark.parametrize("nc", [1, 3, 4, 5, 15, 16, 17, 33])
@pytest.mark.parametrize("kind", ["mixture", "ridge"])
def test_component_steps_same_bits(va, dim, nc, kind):
    """Components of weight 0 in any place change no bit, whatever step of the
    components' loop (one, 4, 8 or 16 at a time) or its remainder they fall in."""
    rng = np.random.default_rng(nc)
    A, B = rng.uniform(0.5, 1.5, nc), rng.uniform(5.0, 20.0, nc)
    t = np.linspace(0.3, 0.7, nc)

    def run(at):
        a, b, c = (np.insert(v, at, z) for v, z in ((A, 0.0), (B, 9.0), (t, 0.5)))
        f = va.DiagonalRidge(a, b, c, dim) if kind == "ridge" else \
            va.GaussianMixture(a, b, c[:, None] * np.linspace(0.8, 1.2, dim)[None, :])
        integ = va.Integrator([[0, 1]] * dim, neval=20000, seed=31, precision='f32')
        r = integ(f, nitn=2)
        return [(g.mean, g.var) for g in r.itn_results], integ.map.grid

    plain = run([])
    for zeros in (1, 2, 3, 15):
        more = run(np.sort(rng.integers(0, nc + 1, zeros)))
        assert more[0] == plain[0] and np.array_equal(more[1], plain[1])
