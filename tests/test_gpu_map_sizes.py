"""AdaptiveMap kernels at the edges of their tiles, scans and LDS plans,
against the FP64 oracle (the bars of test_gpu_map.py: histograms bit for bit,
exact adapts 1e-13 relative)."""
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


@pytest.mark.parametrize("old,new", [(1, 5), (2, 3), (3, 64), (63, 65), (64, 64), (65, 63), (1000, 1),
                                     (1000, 1000), (129, 3072), (3072, 129), (3073, 70)])
@pytest.mark.parametrize("alpha", [0.0, 0.7])
def test_adapt_exact_sizes(va, orc, old, new, alpha):
    rng = np.random.default_rng(old + new)
    m, o = va.AdaptiveMap([[0, 1], [-2, 3]], ninc=old), orc.OracleMap([[0, 1], [-2, 3]], ninc=[old, old])
    y = rng.uniform(0, 1, (4000, 2))
    f = np.exp(rng.normal(0, 3, 4000)) * (y[:, 0] > 0.3)  # empty bins among them
    for q in (m, o):
        q.add_training_data(y, f)
        q.adapt(alpha=alpha, ninc=np.array([new, new]))
    np.testing.assert_allclose(m.grid[:, :new + 1], o.grid[:, :new + 1], rtol=1e-13, atol=1e-13)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1023, 1024, 1025, 17 * 1024 + 1])
@pytest.mark.parametrize("ninc", [[1, 2], [63, 64, 65], [1000] * 12, [1025, 2049]])
def test_train_hist_ordered_sizes(va, orc, n, ninc):
    """Wave, tile and scan-run remainders; bins beyond one scan block; more
    axes than one workgroup's counts; points crowded into few bins."""
    rng = np.random.default_rng(n)
    dim = len(ninc)
    m, o = va.AdaptiveMap([[0, 1]] * dim, ninc=ninc), orc.OracleMap([[0, 1]] * dim, ninc=ninc)
    y = rng.uniform(0, 1, (n, dim))
    y[:, -1] = y[:, -1] ** 8
    y[::7, 0] = 0.0
    f = rng.normal(size=n) * np.exp(rng.uniform(-20, 20, n))
    for _ in range(2):
        m.add_training_data(y, f)
        o.add_training_data(y, f)
    for d, k in enumerate(ninc):
        assert np.array_equal(m.sum_f[d, :k], o.sum_f[d, :k])
        assert np.array_equal(m.n_f[d, :k], o.n_f[d, :k])


@pytest.mark.parametrize("dim,ninc", [(1, 1), (1, 1000), (3, 7), (8, 1000), (17, 1000), (18, 1000), (64, 5)])
@pytest.mark.parametrize("n", [1, 63, 1025, 70001])
def test_map_invmap_sizes(va, orc, dim, ninc, n):
    """Tile remainders; grids staged in LDS (up to 17 axes of 1000) or not;
    invmap's search table (from 65536 points) on a grid with wide and narrow
    increments; x on the nodes, beside them and outside."""
    rng = np.random.default_rng(dim * n)
    grid = np.cumsum(np.exp(rng.normal(0, 2, (dim, ninc + 1))), axis=1)
    m, o = va.AdaptiveMap(grid.tolist()), orc.OracleMap(grid.tolist())
    y = rng.uniform(0, 1, (n, dim))
    y[::5] = rng.integers(0, ninc + 1, y[::5].shape) / ninc
    x, jac = m.map(y)
    xo, jo = o.map(y)
    assert np.array_equal(x.cpu().numpy(), xo)
    assert np.array_equal(jac.cpu().numpy(), jo)
    assert np.array_equal(m.jac1d(y[:1025]), o.jac1d(y[:1025]))
    lo, hi = grid[:, 0], grid[:, -1]
    xo[1::7] = lo - 1
    xo[2::7] = hi + rng.uniform(0, 1, xo[2::7].shape)
    xo[3::7] = np.nextafter(xo[3::7], -np.inf)
    yi, ji = m.invmap(xo)
    yr, jr = o.invmap(xo)
    assert np.array_equal(yi.cpu().numpy(), yr)
    assert np.array_equal(ji.cpu().numpy(), jr)


@pytest.mark.parametrize("dim", [1, 3, 16])
@pytest.mark.parametrize("ninc", [1, 2, 10, 400])
@pytest.mark.parametrize("kind", ["plain", "equal", "tiny", "huge"])
def test_invmap_table_and_search(va, dim, ninc, kind):
    """The search within a table's cell (from 65536 points) and over all nodes
    give the same bits for any x, NaN and infinities among them, on grids with
    equal nodes, denormal increments and lengths that overflow."""
    import torch
    rng = np.random.default_rng(ninc)
    inc = np.exp(rng.normal(0, 2, (dim, ninc)))
    if kind == "equal":
        inc[:, ::2] = 0.0
    grid = np.concatenate([np.zeros((dim, 1)), np.cumsum(inc, axis=1)], axis=1)
    if kind == "tiny":
        grid *= 5e-324 * 64 / inc.mean()
    if kind == "huge":
        grid = (grid / grid.max() * 2.0 - 1.0) * 1.7e308
    m = va.AdaptiveMap(grid.tolist())
    n = 1000
    x = grid[:, rng.integers(0, ninc + 1, n)].T.copy()
    with np.errstate(over='ignore'):
        x[::2] = x[::2] + rng.uniform(-0.1, 1.1, x[::2].shape) * (grid[:, 1] - grid[:, 0]).max()
    x[3::11] = np.nan
    x[4::11] = np.inf
    x[5::11] = -np.inf
    x[6::11] = np.nextafter(x[6::11], np.inf)
    x = torch.as_tensor(x, device='cuda')
    y, jac = m.invmap(x)
    yt, jt = m.invmap(x.repeat(70, 1))
    assert torch.equal(yt.view(torch.int64), y.view(torch.int64).repeat(70, 1))
    assert torch.equal(jt.view(torch.int64), jac.view(torch.int64).repeat(70))


@pytest.mark.parametrize("n", [2, 2047, 4095, 4096, 4097, 5 * 1024 + 64, 17 * 1024 - 1])
@pytest.mark.parametrize("ninc", [[1], [40, 3], [1000] * 3, [3000]])
def test_train_hist_few_tiles(va, orc, n, ninc):
    """The ordered histogram on both sides of its few tiles (up to 4 of 1024
    points), with whole and cut groups of 64 points in the last."""
    rng = np.random.default_rng(n)
    dim = len(ninc)
    m, o = va.AdaptiveMap([[0, 1]] * dim, ninc=ninc), orc.OracleMap([[0, 1]] * dim, ninc=ninc)
    y = rng.uniform(0, 1, (n, dim)) ** 3
    y[::5, 0] = 1.0
    f = rng.normal(size=n) * np.exp(rng.uniform(-20, 20, n))
    for _ in range(2):
        m.add_training_data(y, f)
        o.add_training_data(y, f)
    for d, k in enumerate(ninc):
        assert np.array_equal(m.sum_f[d, :k], o.sum_f[d, :k])
        assert np.array_equal(m.n_f[d, :k], o.n_f[d, :k])
