"""The work that a user of vegas_amd has it do, as timed cases.

Every case is one pass through the package's public entry points:

  integrate  ``Integrator(region)(device integrand, nitn=...)``
  staged     ``Integrator(region)(batch integrand in numpy or torch, nitn=...)``
  batch      ``BatchIntegrator(dims, nevals)(A, B, centers, nitn)``
  train      one learned-map training step: samples, gradient, Adam
  sample     ``CouplingFlow.sample``: the learned map's estimator
  apply      ``AdaptiveMap.map`` and ``AdaptiveMap.invmap``
  refine     ``AdaptiveMap.map`` / ``add_training_data`` / ``adapt``

``exact`` restates the same mathematics (Philox4x32-10 counters, stratified
sampling, the two-pass sums, the grid refinement, the coupling flow) in plain
torch and numpy in 64 bits.
"""
import math

import numpy as np
import torch

import vegas_amd
from vegas_amd.batch import BatchIntegrator, gaussian_params
from vegas_amd.flow import CouplingFlow

TINY = 10.0 ** (-307 + 50)
EPS = 2.220446049250313e-16 * 1e4
M32 = 0xFFFFFFFF


# ------------------------------------------------------------------- cases --
def listed():
    return [
        # the defaults on an easy integral: what an interactive user or a loop
        # over many small integrals calls; all latency
        dict(name="small_2d", kind="integrate", dim=2, neval=1000, nitn=10, fcn="mixture", ncomp=1, sigma=0.1,
             precision="f32", deterministic=True),
        # the textbook run: a 4-D Gaussian at 1e5 evaluations in FP64
        dict(name="gauss_4d_f64", kind="integrate", dim=4, neval=100000, nitn=10, fcn="mixture", ncomp=1,
             sigma=0.0707, precision="f64", deterministic=True),
        # two separated peaks in 8 dimensions at 1e7 evaluations: the
        # framework's headline workload
        dict(name="double_peak_8d", kind="integrate", dim=8, neval=10000000, nitn=3, fcn="mixture", ncomp=2,
             sigma=0.02, precision="f32", deterministic=True),
        # an expensive integrand (1000 Gaussians along a diagonal, given as a
        # plain mixture) at the largest evaluation count
        dict(name="ridge_8d", kind="integrate", dim=8, neval=20000000, nitn=1, fcn="mixture", ncomp=1000,
             sigma=0.005, precision="f32", deterministic=True),
        # more dimensions than the compiled-in ones, an odd count, FP64
        dict(name="gauss_13d_f64", kind="integrate", dim=13, neval=350001, nitn=5, fcn="mixture", ncomp=3,
             sigma=0.1, precision="f64", deterministic=True),
        # a numpy batch integrand: the reference's own way of use
        dict(name="numpy_4d", kind="staged", dim=4, neval=100000, nitn=4, m=1, host=True, sigma=0.1),
        # a torch integrand with four values (normalisation and moments): mean
        # vector and covariances
        dict(name="moments_8d", kind="staged", dim=8, neval=2500000, nitn=2, m=4, host=False, sigma=0.05),
        # a scan: a thousand independent Gaussian integrals of mixed
        # dimension and size in one launch
        dict(name="batch_1024", kind="batch", n=1024, dmin=2, dmax=10, nlo=10000, nhi=1000000, nitn=4),
        # one self-training step of the learned map on a 9-D ridge
        dict(name="flow_train_9d", kind="train", dim=9, nlayers=6, ncomp=500, batch=250000),
        # the learned map's estimator with the same integrand
        dict(name="flow_sample_9d", kind="sample", dim=9, nlayers=6, ncomp=500, n=4000000),
        # the map on its own, there and back, for points of another program
        # (reweighting samples, densities of a proposal)
        dict(name="map_invmap_8d", kind="apply", dim=8, ninc=1000, n=1000003, f32=False),
        # refining a map by hand with its default (reference-order) settings
        dict(name="map_refine_5d", kind="refine", dim=5, ninc=400, n=200000, alpha=0.5),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["integrate", "integrate", "integrate", "staged", "batch", "train", "sample", "apply", "refine"])
    if kind == "integrate":
        dim, nitn = rng.randint(1, 16), rng.randint(1, 10)
        precision = rng.choice(["f32", "f32", "f64"])
        fcn = rng.choice(["mixture", "mixture", "diag"])
        ncomp = _log(rng, 1, 1000 if precision == "f32" else 30)
        # at most the largest listed case's evaluations and integrand work
        top = min(2e7 / nitn, 1.8e10 * (1 if precision == "f32" else 0.03) / nitn / ncomp * 8 / max(dim, 8))
        return dict(kind=kind, dim=dim, neval=_log(rng, 1000, top), nitn=nitn, fcn=fcn, ncomp=ncomp,
                    sigma=round(math.exp(rng.uniform(math.log(0.02 * math.sqrt(dim)), math.log(0.2))), 4), precision=precision,
                    deterministic=rng.random() < 0.8)
    if kind == "staged":
        host = rng.random() < 0.3
        nitn = rng.randint(1, 4)
        dim = rng.randint(1, 12)
        return dict(kind=kind, dim=dim, neval=_log(rng, 2000, 200000 if host else 4e6 / nitn), nitn=nitn,
                    m=rng.choice([1, 1, 2, 3, 4, 6]), host=host,
                    sigma=round(rng.uniform(0.02 * math.sqrt(dim), 0.2), 4))
    if kind == "batch":
        dmin = rng.randint(1, 6)
        return dict(kind=kind, n=_log(rng, 16, 1500), dmin=dmin, dmax=rng.randint(dmin, 10), nlo=_log(rng, 2000, 20000),
                    nhi=_log(rng, 30000, 1000000), nitn=rng.randint(1, 4))
    if kind in ("train", "sample"):
        dim = rng.randint(2, 15)
        nlayers = rng.randint(int(math.ceil(math.log2(dim))) + 1, 8)  # every axis is moved by some layer
        size = dict(batch=_log(rng, 2000, 600000)) if kind == "train" else dict(n=_log(rng, 20000, 4000000))
        return dict(kind=kind, dim=dim, nlayers=nlayers, ncomp=_log(rng, 1, 600), **size)
    if kind == "apply":
        dim = rng.randint(1, 16)
        return dict(kind=kind, dim=dim, ninc=_log(rng, 10, 1000), n=_log(rng, 500, 1.6e7 / dim),
                    f32=rng.random() < 0.3)
    dim = rng.randint(1, 12)
    return dict(kind=kind, dim=dim, ninc=_log(rng, 20, 1000), n=_log(rng, 2000, 5e6 / dim),
                alpha=rng.choice([0.2, 0.5, 1.0]))


# ------------------------------------------------------------------ inputs --
def _mixture(case, seed):
    """A, B and the centres of the case's normalised Gaussians: a few peaks,
    or (10 and more) a ridge along a stretch of the main diagonal."""
    rng = np.random.default_rng([seed, 1])
    d, k, s = case["dim"], case["ncomp"], case["sigma"]
    A = np.full(k, (2 * math.pi * s * s) ** (-0.5 * d) / k)
    B = np.full(k, 0.5 / (s * s))
    if case["fcn"] == "diag" or k >= 10:
        t = np.linspace(0.25, 0.75, k) + rng.uniform(-0.05, 0.05)
        return A, B, t, np.repeat(t[:, None], d, axis=1)
    c = (0.33 + 0.34 * np.arange(k)[:, None] / max(k - 1, 1)) + rng.uniform(-0.05, 0.05, (k, d))
    return A, B, None, c


def _ridge(case, seed):
    """Parameters of the learned map's integrand: a ridge on the diagonal."""
    rng = np.random.default_rng([seed, 2])
    d, k, s = case["dim"], case["ncomp"], 0.015
    t = (np.linspace(0.25, 0.75, k) if k > 1 else np.array([0.5])) + rng.uniform(-0.02, 0.02)
    return np.full(k, (2 * math.pi * s * s) ** (-0.5 * d) / k), np.full(k, 0.5 / (s * s)), t


def _flow_params(case, seed):
    """Weights of a flow that has found the peak: its points lie around the
    ridge's middle, and every layer moves them."""
    from vegas_amd.flow import init_params, OFF_B2, OFF_W3, OFF_B3
    d, L = case["dim"], case["nlayers"]
    P = init_params(d, L, seed)
    rng = np.random.default_rng([seed, 3])
    P[:, OFF_B2:OFF_W3] = rng.normal(0, 0.05, P[:, OFF_B2:OFF_W3].shape)
    P[:, OFF_W3:OFF_B3] = rng.normal(0, 0.004, P[:, OFF_W3:OFF_B3].shape)
    P[:, OFF_B3:] = rng.normal(0, 0.01, P[:, OFF_B3:].shape)
    moved = 1.0 - np.array(_masks(d, L), float)  # [layer][axis]: the layer moves the axis
    P[:, OFF_B3:OFF_B3 + d] -= 2.5 * moved / moved.sum(0)
    return P


def _batch(case, seed):
    rng = np.random.default_rng([seed, 4])
    n = case["n"]
    dims = rng.integers(case["dmin"], case["dmax"] + 1, n)
    cs = [rng.uniform(0.2, 0.8, d) for d in dims]
    sig = np.exp(rng.uniform(math.log(0.03), math.log(0.15), n))
    nev = np.exp(rng.uniform(math.log(case["nlo"]), math.log(case["nhi"]), n)).round().astype(int)
    return dims, cs, sig, nev


def _grid(case, seed):
    """An adapted grid's nodes: increments over two decades."""
    rng = np.random.default_rng([seed, 5])
    inc = np.exp(rng.normal(0, 1.0, (case["dim"], case["ninc"])))
    g = np.concatenate([np.zeros((case["dim"], 1)), np.cumsum(inc, axis=1)], axis=1)
    return g / g[:, -1:]


def _gen(seed, dev="cuda"):
    return torch.Generator(device=dev).manual_seed(int(seed))


def _staged_fcn(case, seed, xp):
    """The batch integrand of a staged case (numpy or torch arrays alike): a
    Gaussian times 1, x0, x0 x1, ... for m values."""
    rng = np.random.default_rng([seed, 6])
    d, s, m = case["dim"], case["sigma"], case["m"]
    c = rng.uniform(0.4, 0.6, d)
    norm = (2 * math.pi * s * s) ** (-0.5 * d)
    cc = c if xp is np else torch.as_tensor(c, device="cuda")

    def f(x):
        p = norm * xp.exp(-(0.5 / (s * s)) * ((x - cc) ** 2).sum(-1))
        if m == 1:
            return p
        vals, q = [p], p
        for j in range(1, m):
            q = q * x[:, (j - 1) % d]
            vals.append(q)
        return xp.stack(vals, -1)
    return f


def prepare(case, seed):
    kind = case["kind"]
    if kind == "integrate":
        A, B, t, c = _mixture(case, seed)
        f = vegas_amd.DiagonalRidge(A, B, t, case["dim"]) if case["fcn"] == "diag" else vegas_amd.GaussianMixture(A, B, c)
        integ = vegas_amd.Integrator([[0, 1]] * case["dim"], neval=case["neval"], seed=seed, precision=case["precision"],
                                     deterministic=case["deterministic"])
        return dict(case=case, integ=integ, f=f)
    if kind == "staged":
        f = _staged_fcn(case, seed, np if case["host"] else torch)
        f = vegas_amd.lbatchintegrand(f) if case["host"] else vegas_amd.gpu_lbatchintegrand(f)
        integ = vegas_amd.Integrator([[0, 1]] * case["dim"], neval=case["neval"], seed=seed,
                                     min_neval_batch=100000 if case["host"] else 2000000)
        return dict(case=case, integ=integ, f=f)
    if kind == "batch":
        dims, cs, sig, nev = _batch(case, seed)
        A, B = gaussian_params(dims, sig)
        seeds = np.arange(1, case["n"] + 1, dtype=np.uint64) + np.uint64(seed * 100003)
        return dict(case=case, bi=BatchIntegrator(dims, nev, seeds=seeds, tiles_per_item=128), A=A, B=B, c=cs)
    if kind in ("train", "sample"):
        A, B, t = _ridge(case, seed)
        flow = CouplingFlow(case["dim"], case["nlayers"], params=_flow_params(case, seed))
        st = dict(case=case, flow=flow, f=vegas_amd.DiagonalRidge(A, B, t, case["dim"]), seed=seed, it=0)
        if kind == "train":
            st["status"] = torch.zeros(1, dtype=torch.int32, device="cuda")
            st["logw"] = torch.zeros(case["batch"], dtype=torch.float32, device="cuda")
        return st
    m = vegas_amd.AdaptiveMap(_grid(case, seed).tolist())
    y = torch.rand((case["n"], case["dim"]), dtype=torch.float32 if case.get("f32") else torch.float64, device="cuda",
                   generator=_gen(seed))
    st = dict(case=case, map=m, y=y)
    if kind == "refine":
        rng = np.random.default_rng([seed, 7])
        st["center"] = torch.as_tensor(rng.uniform(0.4, 0.6, case["dim"]), device="cuda")
    return st


def _ravg(r):
    """A scalar result's numbers: the average and every iteration."""
    return dict(mean=r.mean, sdev=r.sdev, chi2=r.chi2, neval=int(r.sum_neval),
                itn_mean=[g.mean for g in r.itn_results], itn_sdev=[g.sdev for g in r.itn_results])


def _peak(x, center):
    return torch.exp(-50.0 * ((x - center) ** 2).sum(-1))


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind in ("integrate", "staged"):
        integ = st["integ"]
        r = integ(st["f"], nitn=case["nitn"])
        out = dict(grid=integ.map._grid, sigf=integ._sigf, last_neval=integ.last_neval)
        if kind == "integrate" or case["m"] == 1:
            out.update(_ravg(r))
        else:
            out.update(mean=r.mean, cov=r.cov, first_mean=r.itn_results[0].mean, first_cov=r.itn_results[0].cov)
        return out
    if kind == "batch":
        bi = st["bi"]
        r = bi(st["A"], st["B"], st["c"], nitn=case["nitn"])
        return dict(mean=r.mean, sdev=r.sdev, chi2=r.chi2, itn_mean=r.itn_mean[1:], itn_sdev=r.itn_sdev[1:],
                    first_mean=r.itn_mean[0], first_sdev=r.itn_sdev[0], itn_neval=r.itn_neval, grid=bi.grid)
    if kind == "train":
        flow = st["flow"]
        st["it"] += 1
        _, _, x, fj = flow.sample(st["f"], case["batch"], seed=st["seed"], iteration=st["it"], keep_points=True,
                                  status=st["status"])
        flow.grad(x, fj, st["logw"], "squared")
        flow.adam(lr=1e-4)
        return dict(x=x[:, :case["dim"]], fj=fj, grad=flow.last_grad())
    if kind == "sample":
        st["it"] += 1
        s1, s2 = st["flow"].sample(st["f"], case["n"], seed=st["seed"], iteration=st["it"])
        return dict(s1=s1, s2=s2)
    m, y = st["map"], st["y"]
    x, jac = m.map(y)
    if kind == "apply":
        yb, jb = m.invmap(x)
        return dict(x=x, jac=jac, y=yb, jac_inv=jb)
    f = _peak(x, st["center"])
    m.add_training_data(y, (jac * f) ** 2)
    m.adapt(alpha=case["alpha"])
    return dict(x=x, jac=jac, grid=m._grid)


# -------------------------------------------------------------------- work --
def _strata(dim, neval, nf=0.75):
    """Strata and increments per axis of a default Integrator at neval."""
    q = (1 - nf) * neval / 2.0
    ns = max(int(q ** (1.0 / dim)), 1)
    up = int((np.log(q) - dim * np.log(ns)) / np.log(1 + 1.0 / ns))
    return [ns + 1] * up + [ns] * (dim - up)


def _incs(nstrat, neval, maxinc):
    """Increments per axis for these strata (strata beyond them merge)."""
    ni, out, st = min(int(neval / 10.0), maxinc), [], []
    for s in nstrat:
        if ni >= s:
            out.append(ni // s * s)
        elif s <= maxinc:
            out.append(s)
        else:
            s = s // ni * ni
            out.append(ni)
        st.append(s)
    return st, out


def work(case):
    """What a pass has to do: flops of the integrand, map, weight and sums per
    evaluation (a Gaussian 3 dim + 4, the rest 9 dim + 9, and 20 integer
    operations per random number); bytes of the state read and written and
    of the points that enter or leave."""
    kind, d = case["kind"], case.get("dim")
    if kind in ("integrate", "staged"):
        nh = float(np.prod(_strata(d, case["neval"])))
        evals = float(case["neval"]) * case["nitn"]
        comp = case.get("ncomp", 1) * (3 * d + 4 if case.get("fcn") != "diag" else 5) + (2 * case["m"] if "m" in case else 0)
        byts = case["nitn"] * (16.0 * nh + 16.0 * d * 1000)
        if kind == "staged":
            byts += evals * 8 * (2 * d + 2 * case["m"])
        return dict(bytes=byts, flops=evals * (comp + 29 * d + 9))
    if kind == "batch":
        mean = (case["nhi"] - case["nlo"]) / math.log(case["nhi"] / case["nlo"])
        evals = mean * case["n"] * case["nitn"]
        dm = 0.5 * (case["dmin"] + case["dmax"])
        return dict(bytes=case["nitn"] * case["n"] * (16.0 * dm * 501 + 2.0 * mean), flops=evals * (32 * dm + 13))
    if kind in ("train", "sample"):
        n = case["batch"] if kind == "train" else case["n"]
        fwd = 2.0 * (d * 128 + 128 * 128 + 128 * 2 * d) * case["nlayers"] * n
        f = fwd * (5 if kind == "train" else 1) + 5.0 * case["ncomp"] * n
        params = case["nlayers"] * 4.0 * 22688
        return dict(bytes=params * (8 if kind == "train" else 1) + (n * 4.0 * (d + 1) if kind == "train" else 0), flops=f)
    n, w = float(case["n"]), 4 if case.get("f32") else 8
    if kind == "apply":  # y in, x and jac out; x in, y and jac out (FP64)
        return dict(bytes=n * (w * (2 * d + 1) + w * d + 8 * (d + 1)), flops=n * d * 20)
    return dict(bytes=n * (8 * (2 * d + 1) + 8 * (d + 1)) + 64.0 * d * case["ninc"], flops=n * d * 15)


# ------------------------------------------------------------------- exact --
def _philox(p, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) of counters (p, c1, c2, c3), key
    (k0, k1): four int64 tensors of 32-bit words."""
    x, y = p & M32, torch.full_like(p, c1)
    z, w = torch.full_like(p, c2), torch.full_like(p, c3)

    def mul(a, b):
        lo = b * (a & 0xFFFF)
        hi = b * (a >> 16) + (lo >> 16)
        return hi >> 16, ((hi & 0xFFFF) << 16) | (lo & 0xFFFF)
    for _ in range(10):
        h0, l0 = mul(x, 0xD2511F53)
        h1, l1 = mul(z, 0xCD9E8D57)
        x, y, z, w = h1 ^ y ^ k0, l1, h0 ^ w ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & M32, (k1 + 0xBB67AE85) & M32
    return x, y, z, w


def _uniforms(p, dim, seed, it, bits53):
    k0, k1 = seed & M32, (seed >> 32) & M32
    out, per = [], 2 if bits53 else 4
    for b in range((dim + per - 1) // per):
        w = _philox(p, 0, it, b, k0, k1)
        if bits53:
            out += [((w[i] >> 5).double() * 67108864.0 + (w[i + 1] >> 6).double()) / 9007199254740992.0 for i in (0, 2)]
        else:
            out += [(v >> 8).double() / 16777216.0 for v in w]
    return out[:dim]


def _refine(g, ssum, cnt, alpha):
    """One grid refinement: average, smooth, compress, equal shares."""
    n = len(g) - 1
    if n < 2 or alpha <= 0:
        return g.copy()
    a = np.where(cnt > 0, ssum / np.maximum(cnt, TINY), 0.0)
    t = np.empty(n)
    t[0], t[-1] = abs(7 * a[0] + a[1]) / 8, abs(7 * a[-1] + a[-2]) / 8
    t[1:-1] = np.abs(6 * a[1:-1] + a[:-2] + a[2:]) / 8
    s = t.sum()
    v = t / s + TINY if s > 0 else np.full(n, TINY)
    ok = (v > 0) & (v <= 0.99999999)
    v[ok] = (-(1 - v[ok]) / np.log(v[ok])) ** alpha
    P = np.cumsum(v)
    target = np.arange(1, n) * (P[-1] / n)
    j = np.minimum(np.searchsorted(P, target, side="left"), n - 1)
    out = g.copy()
    out[1:-1] = g[j + 1] - (P[j] - target) / v[j] * (g[j + 1] - g[j])
    return out


def _first_iteration(dim, neval, seed, bits53, f, m=1, maxinc=1000, alpha=0.5, beta=0.75, frac=0.75):
    """The first iteration on the unit cube from a uniform grid: means and
    covariances of f's values, sigf and the refined grid."""
    nstrat, ninc = _incs(_strata(dim, neval, frac), neval, maxinc)
    nh = int(np.prod(nstrat))
    nmin = max(int((1 - frac) * neval / nh) if nh > 1 else int(neval), 2)
    n = min(int(frac * neval / nh) + nmin, max(50000, nmin)) if nh > 1 else int(neval / nh)
    grid = [np.linspace(0.0, 1.0, k + 1) for k in ninc]
    ssum, cnt = [np.zeros(k) for k in ninc], [np.zeros(k) for k in ninc]
    mean, cov, sig = torch.zeros(m, dtype=torch.float64, device="cuda"), torch.zeros(m, m, dtype=torch.float64, device="cuda"), []
    step = max(1, 2000000 // n)
    for h0 in range(0, nh, step):
        h = torch.arange(h0, min(h0 + step, nh), device="cuda")
        p = h0 * n + torch.arange(len(h) * n, device="cuda")
        hh = h.repeat_interleave(n)
        us = _uniforms(p, dim, seed, 0, bits53)
        x, J, bins, inside = [], torch.ones(len(p), dtype=torch.float64, device="cuda"), [], []
        for d in range(dim):
            c = (hh % nstrat[d]).double()
            hh = hh // nstrat[d]
            t = (c + us[d]) * (ninc[d] // nstrat[d]) if ninc[d] % nstrat[d] == 0 else (c + us[d]) / nstrat[d] * ninc[d]
            k = t.long().clamp_(max=ninc[d] - 1)
            g = torch.as_tensor(grid[d], device="cuda")
            inc = (g[1:] - g[:-1])[k]
            x.append(g[k] + inc * (t - k))
            J *= inc * ninc[d]
            bins.append(k)
            inside.append(t > 0)
        w = J / (nh * float(n))
        wf = w[:, None] * f(torch.stack(x, 1)).reshape(-1, m)
        c2 = (wf[:, 0] * n) ** 2
        for d in range(dim):
            keep = inside[d]
            ssum[d] += torch.zeros(ninc[d], dtype=torch.float64, device="cuda").index_add_(0, bins[d][keep], c2[keep]).cpu().numpy()
            cnt[d] += torch.bincount(bins[d][keep], minlength=ninc[d]).double().cpu().numpy()
        wf = wf.reshape(-1, n, m)
        S = wf.sum(1)
        mu = S / n
        dev = wf - mu[:, None, :]
        guard = EPS * mu.abs()[:, None, :]
        small = dev.abs() < guard
        dev = torch.where(small, torch.zeros_like(dev), dev)
        Q = dev.transpose(1, 2).contiguous() @ dev + torch.diag_embed((small * guard ** 2).sum(1))
        D = dev.sum(1)
        var = (n * Q - D[:, :, None] * D[:, None, :]) / (n - 1.0)
        mean += (S + D).sum(0)
        cov += var.sum(0)
        sig.append(var[:, 0, 0].abs() ** (beta / 2))
    ld = max(ninc) + 1
    out = np.empty((dim, ld))
    for d in range(dim):
        row = _refine(grid[d], ssum[d], cnt[d], alpha)
        out[d, :len(row)], out[d, len(row):] = row, row[-1]
    return mean.cpu().numpy(), cov.cpu().numpy(), torch.cat(sig) if nh > 1 else None, out


def _exact_mixture(A, B, t, c, x):
    d = x.shape[1]
    if t is not None:  # centres on the diagonal
        xb = x.mean(1)
        P = ((x - xb[:, None]) ** 2).sum(1)
        out = torch.zeros_like(P)
        for a, b, tk in zip(A.tolist(), B.tolist(), t.tolist()):
            out += a * torch.exp(-b * (P + d * (xb - tk) ** 2))
        return out
    return sum(a * torch.exp(-b * ((x - torch.as_tensor(ck, device=x.device)) ** 2).sum(1)) for a, b, ck in zip(A, B, c))


def _net(P, a):
    """A conditioner's scales and shifts for inputs a [n][16]."""
    W1, r = P[:2048].reshape(128, 16), P[2048:]
    W2, b2, W3, b3 = r[:16384].reshape(128, 128), r[16384:16512], r[16512:20608].reshape(32, 128), r[20608:]
    h = torch.relu(torch.relu(a @ W1.T) @ W2.T + b2)
    o = h @ W3.T + b3
    return 4.0 * torch.tanh(o[:, :16] / 4.0), o[:, 16:]


def _masks(dim, L):
    nb = max(1, int(math.ceil(math.log2(dim)))) if dim > 1 else 1
    return [[((d >> k) & 1) == 0 for d in range(dim)] if k < nb else [((d >> ((k - nb) % nb)) & 1) == 1 for d in range(dim)]
            for k in range(L)]


def _couple(P, u, mask, dim, inverse):
    on = torch.zeros(16, dtype=torch.float64, device=u.device)
    on[:dim] = torch.tensor([1.0 if v else 0.0 for v in mask], dtype=torch.float64, device=u.device)
    off = torch.zeros_like(on)
    off[:dim] = 1.0 - on[:dim]
    one = torch.zeros_like(on)
    one[15] = 1.0
    s, t = _net(P, u * on + one)
    s, t = s * off, t * off
    return ((u - t) * torch.exp(-s) if inverse else u * torch.exp(s) + t), s.sum(1)


def _logsig(u):
    return -u.abs() - 2.0 * torch.log1p(torch.exp(-u.abs()))


def _flow_sample(P, case, seed, it, i0, n):
    dim = case["dim"]
    k0, k1 = seed & M32, (seed >> 32) & M32
    i = torch.arange(i0, i0 + n, device="cuda")
    z = torch.stack([(v >> 8).double() / 16777216.0 + 1.0 / 33554432.0
                     for b in range(4) for v in _philox(i, 0, it, b, k0, k1)], 1)
    u = torch.log(z) - torch.log1p(-z)
    l = -_logsig(u[:, :dim]).sum(1)
    for k, m in enumerate(_masks(dim, case["nlayers"])):
        u, s = _couple(P[k], u, m, dim, False)
        l = l + s
    return torch.sigmoid(u[:, :dim]), l + _logsig(u[:, :dim]).sum(1)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("integrate", "staged"):
        dim = case["dim"]
        cost = float(case["neval"]) * (dim + case.get("ncomp", 1) / 8.0)
        if cost > 3e9:
            return None
        if kind == "integrate":
            A, B, t, c = _mixture(case, seed)
            bits53, m, f = case["precision"] == "f64", 1, lambda x: _exact_mixture(A, B, t, c, x)
        else:
            bits53, m, f = True, case["m"], _staged_fcn(case, seed, torch)
        mean, cov, sig, grid = _first_iteration(dim, case["neval"], seed, bits53, f, m)
        last = case["nitn"] == 1
        out = dict(grid=grid if last else None, sigf=sig if last else None)
        if m > 1:
            out.update(mean=mean if last else None, cov=cov if last else None, first_mean=mean, first_cov=cov)
        else:
            rest = [None] * (case["nitn"] - 1)
            sd = math.sqrt(cov[0, 0])
            out.update(mean=mean[0] if last else None, sdev=sd if last else None, itn_mean=[mean[0]] + rest,
                       itn_sdev=[sd] + rest)
        return out
    if kind == "batch":
        dims, cs, sig, nev = _batch(case, seed)
        if float(nev.sum()) > 6e8 or case["n"] > 1100:
            return None
        A, B = gaussian_params(dims, sig)
        res = [_first_iteration(int(d), int(ne), i + 1 + seed * 100003, False,
                                lambda x, i=i: _exact_mixture(A[i:i + 1], B[i:i + 1], None, [cs[i]], x), maxinc=500)[:2]
               for i, (d, ne) in enumerate(zip(dims, nev))]
        return dict(first_mean=np.array([r[0][0] for r in res]), first_sdev=np.sqrt([r[1][0, 0] for r in res]))
    if kind in ("train", "sample"):
        P = torch.as_tensor(_flow_params(case, seed).astype(np.float64), device="cuda").requires_grad_(kind == "train")
        A, B, t = _ridge(case, seed)
        n = case["batch"] if kind == "train" else case["n"]
        xs, fs, s1, s2 = [], [], 0.0, 0.0
        with torch.no_grad():
            for i0 in range(0, n, 500000):
                x, lj = _flow_sample(P, case, seed, 1, i0, min(500000, n - i0))
                fj = _exact_mixture(A, B, t, None, x) * torch.exp(lj)
                s1, s2 = s1 + float(fj.sum()), s2 + float((fj * fj).sum())
                if kind == "train":
                    xs.append(x)
                    fs.append(fj)
        if kind == "sample":
            return dict(s1=s1, s2=s2)
        x, fj = torch.cat(xs), torch.cat(fs)
        c = fj * fj / (fj * fj).sum()
        for i0 in range(0, n, 50000):
            xc = x[i0:i0 + 50000].clamp(1e-7, 1 - 1e-7)
            u = torch.zeros((len(xc), 16), dtype=torch.float64, device="cuda")
            u[:, :case["dim"]] = torch.log(xc) - torch.log1p(-xc)
            lq = -_logsig(u[:, :case["dim"]]).sum(1)
            for k, m in reversed(list(enumerate(_masks(case["dim"], case["nlayers"])))):
                u, s = _couple(P[k], u, m, case["dim"], True)
                lq = lq - s
            lq = lq + _logsig(u[:, :case["dim"]]).sum(1)
            (-(c[i0:i0 + 50000] * lq).sum()).backward()
        return dict(x=x, fj=fj, grad=P.grad.reshape(case["nlayers"], -1))
    # the map
    g = _grid(case, seed)
    dt = torch.float32 if case.get("f32") else torch.float64
    y = torch.rand((case["n"], case["dim"]), dtype=dt, device="cuda", generator=_gen(seed)).double()
    ni = case["ninc"]
    x, J, k_all = torch.empty_like(y), torch.ones(len(y), dtype=torch.float64, device="cuda"), []
    for d in range(case["dim"]):
        gd = torch.as_tensor(g[d], device="cuda")
        tt = y[:, d] * ni
        k = tt.long().clamp_(max=ni - 1)
        inc = (gd[1:] - gd[:-1])[k]
        x[:, d] = gd[k] + inc * (tt - k)
        J *= inc * ni
        k_all.append(k)
    if kind == "apply":
        xr = x.to(dt).double()
        yb, jb = torch.empty_like(y), torch.ones_like(J)
        for d in range(case["dim"]):
            gd = torch.as_tensor(g[d], device="cuda")
            k = (torch.searchsorted(gd, xr[:, d].contiguous(), right=True) - 1).clamp_(0, ni - 1)
            inc = (gd[1:] - gd[:-1])[k]
            yb[:, d] = (k + (xr[:, d] - gd[k]) / inc) / ni
            jb *= inc * ni
        return dict(x=x, jac=J, y=yb, jac_inv=jb)
    rng = np.random.default_rng([seed, 7])
    fv = (J * _peak(x, torch.as_tensor(rng.uniform(0.4, 0.6, case["dim"]), device="cuda"))) ** 2
    out = np.empty_like(g)
    for d in range(case["dim"]):
        keep = (y[:, d] > 0) & (y[:, d] < 1)
        s = torch.zeros(ni, dtype=torch.float64, device="cuda").index_add_(0, k_all[d][keep], fv[keep]).cpu().numpy()
        out[d] = _refine(g[d], s, torch.bincount(k_all[d][keep], minlength=ni).double().cpu().numpy(), case["alpha"])
    return dict(x=x, jac=J, grid=out)
