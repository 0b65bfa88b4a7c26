"""Workloads of the smartpca engine as its users call it, for timing and for comparing results.

listed() names them, draw() gives more of the same ranges, prepare() makes what a program
holds before the call, run() is one pass through the public entry points (eig_amd.Engine
and eig_amd.Server), work() the bytes and operations a pass cannot do without, and exact()
the same results in plain torch/numpy in 64 bits.

Genotypes are Balding-Nichols-like: ancestral frequency U(0.01, 0.5), per-population drift
Fst, a few per cent missing.  Twelve populations give ten eigenvectors above the noise
bulk, the reference's default number (numoutevec).
"""
from __future__ import annotations

import math

import numpy as np
import torch

import eig_amd

NPOP = 12
K = 10  # axes: the reference's default numoutevec
CHUNK = 1 << 25  # genotypes generated or unpacked at a time


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the whole of a small run (a pilot panel, the distributed example's scale): host
        # rows in, statistics, XTX, axes, loadings and projections out; latency and launches
        dict(name="pca_198", kind="pca", N=198, M=2000, form="fp64", rows="host", fst=0.05,
             miss=0.01),
        # an ordinary run of the default (FP64) form at 1,000 samples x 50,000 SNPs
        dict(name="pca_1k", kind="pca", N=1000, M=50000, form="fp64", rows="host", fst=0.05,
             miss=0.01),
        # a pass after outlier removal: ragged sizes, a subset of the loaded samples
        dict(name="pca_2503", kind="pca", N=2611, M=200003, form="fp64", rows="resident",
             drop=108, fst=0.03, miss=0.02),
        # one pass (statistics, XTX, all eigenvalues, ten axes) over a resident panel at the
        # benchmark's 5,000 x 600,000, in the fast and in the default form
        dict(name="pass_5k_bf16x4", kind="pass", N=5000, M=600000, form="bf16x4", fst=0.04,
             miss=0.02),
        dict(name="pass_5k_fp64", kind="pass", N=5000, M=600000, form="fp64", fst=0.04,
             miss=0.02),
        # fastmode (randomized PCA) at a size where the exact path is still an alternative,
        # and at the benchmark's 100,000 x 500,000 in the split form
        dict(name="fast_20k_fp64", kind="fast", N=20011, M=100003, form="fp64", L=20, I=10,
             fst=0.03, miss=0.01, gen="torch"),
        dict(name="fast_100k_bf16x4", kind="fast", N=100000, M=500000, form="bf16x4", L=20, I=10,
             fst=0.03, miss=0.01, gen="engine"),
        # SNP loadings of ten axes and lsqproject of every loaded individual
        dict(name="project_5k", kind="project", N=5000, M=600000, K=10, fst=0.04, miss=0.02),
        # serving: one sample alone (latency), and a burst of mixed requests (throughput)
        dict(name="serve_1", kind="serve", N=500, M=600000, K=10, nreq=1, most=1, fst=0.04,
             miss=0.02),
        dict(name="serve_burst", kind="serve", N=500, M=600000, K=10, nreq=24, most=512, fst=0.04,
             miss=0.02),
        # usepopsformissing with SNP weights: the explicit-column path
        dict(name="normal_1k", kind="normal", N=1003, M=30011, weight=True, ldregress=0, fst=0.05,
             miss=0.05),
        # every eigenvector of a caller's covariance matrix (the eigvecs contract)
        dict(name="eigh_all_1203", kind="eigh", n=1203, nvec=1203),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pca", "pca", "pass", "fast", "project", "serve", "normal", "eigh"])
    fst = round(rng.uniform(0.02, 0.08), 3)
    miss = round(rng.choice([0.0, 0.005, 0.02, 0.05]), 3)
    if kind in ("pca", "pass"):
        N = _log(rng, 150, 5000)
        M = _log(rng, 2000, min(600000, 1.4e13 / (N * N)))
        c = dict(kind=kind, N=N, M=M, form=rng.choice(["fp64", "fp64", "bf16x4"]), fst=fst,
                 miss=miss)
        if kind == "pca":
            c["rows"] = rng.choice(["host", "resident"])
            if rng.random() < 0.5:
                c["drop"] = max(1, N // 25)
        return c
    if kind == "fast":
        N = _log(rng, 1000, 40000)
        return dict(kind="fast", N=N, M=_log(rng, 5000, min(200000, 2.5e9 / N)),
                    form=rng.choice(["fp64", "bf16x4"]), L=20, I=rng.choice([5, 10]), fst=fst,
                    miss=miss, gen="torch")
    if kind == "project":
        return dict(kind="project", N=_log(rng, 300, 5000), M=_log(rng, 5000, 600000),
                    K=rng.choice([2, 4, 10]), fst=fst, miss=miss)
    if kind == "serve":
        return dict(kind="serve", N=300, M=_log(rng, 20000, 600000), K=rng.choice([2, 4, 10]),
                    nreq=rng.choice([1, 4, 16]), most=rng.choice([1, 16, 200, 512]), fst=fst,
                    miss=miss)
    if kind == "normal":
        return dict(kind="normal", N=_log(rng, 200, 1500), M=_log(rng, 2000, 40000),
                    weight=rng.choice([False, True]), ldregress=rng.choice([0, 0, 2]), fst=fst,
                    miss=0.05)
    n = _log(rng, 60, 1500)
    return dict(kind="eigh", n=n, nvec=rng.choice([n, 10]))


# ---------------------------------------------------------------- inputs
def _pop(N):
    return torch.arange(N, device="cuda") * NPOP // N


def _freqs(c, seed):
    """[NPOP, M] float64 population frequencies."""
    r = np.random.Generator(np.random.PCG64(seed))
    p = r.uniform(0.01, 0.5, c["M"])
    drift = r.standard_normal((NPOP, c["M"])) * np.sqrt(c["fst"] * p * (1 - p))
    return np.clip(p + drift, 0.0, 1.0)


def _codes(freq, pop, miss, seed):
    """Genotype codes [M, n] on the GPU (0/1/2, 3 = missing) of samples of populations
    pop [n]; miss: one missing rate, or one per sample."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    f = torch.from_numpy(freq).to("cuda", torch.float32)
    M, n = f.shape[1], len(pop)
    out = torch.empty((M, n), dtype=torch.uint8, device="cuda")
    step = max(1, CHUNK // n)
    miss = torch.as_tensor(miss, dtype=torch.float32, device="cuda")
    for m in range(0, M, step):
        fm = f[:, m:m + step].t()[:, pop]
        k = (torch.rand(fm.shape, generator=g, device="cuda") < fm).to(torch.uint8)
        k += torch.rand(fm.shape, generator=g, device="cuda") < fm
        k[torch.rand(fm.shape, generator=g, device="cuda") < miss] = 3
        out[m:m + step] = k
    return out


def _pack(codes, width):
    """2-bit rows of `width` bytes (the first code in the highest bits), on the host; the
    codes past the end of a row are 0."""
    R, n = codes.shape
    out = np.empty((R, width), np.uint8)
    step = max(1, CHUNK // (4 * width))
    for r in range(0, R, step):
        c = codes[r:r + step]
        p = torch.zeros((len(c), 4 * width), dtype=torch.uint8, device="cuda")
        p[:, :n] = c
        p = p.view(len(c), width, 4)
        out[r:r + step] = (p[..., 0] << 6 | p[..., 1] << 4 | p[..., 2] << 2 | p[..., 3]).cpu().numpy()
    return out


def _geno(c, seed):
    return _codes(_freqs(c, seed), _pop(c["N"]), c["miss"], seed)


def _rows(c, seed):
    return _pack(_geno(c, seed), max(48, (c["N"] + 3) // 4))


def _kept(c, seed):
    """The samples of the pass: all, or all but `drop` of them."""
    gone = np.random.Generator(np.random.PCG64(seed + 1)).choice(c["N"], c.get("drop", 0),
                                                                 replace=False)
    return np.setdiff1d(np.arange(c["N"], dtype=np.int32), gone).astype(np.int32)


def _axes(c, seed):
    """K orthonormal axes with population structure, as eigenvectors have."""
    r = np.random.Generator(np.random.PCG64(seed + 2))
    pop = np.arange(c["N"]) * NPOP // c["N"]
    a = r.standard_normal((c["K"], NPOP))[:, pop] + 0.1 * r.standard_normal((c["K"], c["N"]))
    q = np.linalg.qr((a - a.mean(axis=1, keepdims=True)).T)[0].T
    return np.ascontiguousarray(q)


def _requests(c):
    """Request sizes, the same for every seed: log-uniform up to `most`."""
    r = np.random.Generator(np.random.PCG64([c["nreq"], c["most"]]))
    n = np.floor(np.exp(r.uniform(0, math.log(c["most"] + 1), c["nreq"]))).astype(int)
    return [int(x) for x in np.clip(n, 1, c["most"])]


def _queries(c, seed):
    """Query codes [nq, M]: samples of the panel's populations, missing rates U(0, 0.9)."""
    r = np.random.Generator(np.random.PCG64(seed + 4))
    nq = sum(_requests(c))
    pop = torch.from_numpy(r.integers(0, NPOP, nq)).cuda()
    return _codes(_freqs(c, seed), pop, r.uniform(0.0, 0.9, nq), seed + 4).t()


def _eigscale(c):
    return 1.0 + 0.05 * np.arange(c["K"])


def _weight(c, seed):
    return np.random.Generator(np.random.PCG64(seed + 5)).uniform(0.5, 1.5, c["M"])


def _covariance(c, seed):
    r = np.random.Generator(np.random.PCG64(seed + 6))
    x = r.standard_normal((c["n"], 2 * c["n"] + 5))
    x[:, :40] += 3.0 * r.standard_normal((c["n"], 1)) * r.standard_normal(40)
    return np.ascontiguousarray(x @ x.T / x.shape[1])


FORMS = {"fp64": eig_amd.FORM_FP64, "bf16x4": eig_amd.FORM_BF16X4}


class Session:
    """An engine (and perhaps a server) with a case's inputs; released with the object."""

    def __init__(self, case):
        self.case = case
        self.eng = eig_amd.Engine(0)
        self.srv = None
        self.pool = None

    def __del__(self):
        if self.srv is not None:
            self.srv.stop()
        if self.pool is not None:
            self.eng.dev_free(self.pool)
        self.eng.close()


def prepare(case, seed):
    c = case
    s = Session(c)
    eng, kind = s.eng, c["kind"]
    if kind == "eigh":
        s.a = _covariance(c, seed)
        return s
    if kind == "fast":
        s.omega = np.random.Generator(np.random.PCG64(seed + 7)).standard_normal((c["N"], c["L"]))
    if c.get("gen") == "engine":
        f = _freqs(c, seed)
        thr = np.minimum(np.floor(f * 4294967296.0), 4294967295.0).astype(np.uint32)
        pop = (np.arange(c["N"]) * NPOP // c["N"]).astype(np.int32)
        eng.synth(c["M"], c["N"], thr, np.repeat(pop[:, None], 3, axis=1),
                  np.full((c["N"], 2), 0xFFFFFFFF, np.uint32), int(c["miss"] * 4294967296.0), seed)
    else:
        s.rows = _rows(c, seed)
        if not (kind == "pca" and c["rows"] == "host"):
            eng.load_packed(s.rows, c["N"])
            s.rows = None
    s.xindex = _kept(c, seed)
    s.use = np.ones(c["N"], np.int32)
    if kind in ("fast", "project", "serve", "normal"):
        eng.select(s.xindex)
        eng.snpstats(fetch=False)
    if kind in ("project", "serve"):
        s.vec = _axes(c, seed)
    if kind == "normal":
        s.xtypes = (np.arange(c["N"]) * NPOP // c["N"]).astype(np.int32)
        s.weight = _weight(c, seed) if c["weight"] else None
        s.chrom = (1 + np.arange(c["M"]) * 22 // c["M"]).astype(np.int32)
        s.ppos = 1000.0 * np.arange(c["M"])
        s.gpos = 1e-5 * np.arange(c["M"])
    if kind == "serve":
        eng.loadings(s.vec, want_ffvecs=False)
        s.srv = eig_amd.Server(eng, eigscale=_eigscale(c))
        s.stride = s.srv.rowpad
        s.sizes = _requests(c)
        q = _pack(_queries(c, seed), s.stride)
        s.pool = eng.dev_alloc(q.size)
        eng.memcpy(s.pool, q, q.size)
    return s


# ---------------------------------------------------------------- one pass
def run(s):
    c, eng = s.case, s.eng
    kind = c["kind"]
    if kind == "pca":
        # the analysis of a smartpca run, with the outputs its files hold
        if c["rows"] == "host":
            eng.load_packed(s.rows, c["N"])
        eng.select(s.xindex)
        st = eng.snpstats()
        scale, _ = eng.xtx(FORMS[c["form"]], 256, want_matrix=False)
        ev, vec = eng.eigh_xtx(K)
        ff, fx = eng.loadings(vec)
        a, b, ps = eng.lsqproject(s.use, K)
        return dict(c0=st["c0"], c1=st["c1"], nmiss=st["nmiss"], status=st["status"],
                    mean=st["mean"], fancy=st["fancy"], scale=scale, evals=ev, evecs=vec,
                    ffvecs=ff, fxscal=fx, a=a, b=b, pstatus=ps)
    if kind == "pass":
        eng.select(s.xindex)
        eng.snpstats(fetch=False)
        scale, _ = eng.xtx(FORMS[c["form"]], 256, want_matrix=False)
        ev, vec = eng.eigh_xtx(K)
        return dict(scale=scale, evals=ev, evecs=vec)
    if kind == "fast":
        ev, vec = eng.fpca(K, c["L"], c["I"], omega=s.omega, form=FORMS[c["form"]])
        return dict(evals=ev, evecs=vec)
    if kind == "project":
        ff, fx = eng.loadings(s.vec)
        a, b, ps = eng.lsqproject(s.use, c["K"])
        return dict(ffvecs=ff, fxscal=fx, a=a, b=b, pstatus=ps)
    if kind == "serve":
        tickets, at = [], 0
        for n in s.sizes:
            tickets.append(s.srv.submit(device_ptr=s.pool + at * s.stride, nq=n, stride=s.stride))
            at += n
        got = [s.srv.poll(t) for t in tickets]
        return dict(coords=np.concatenate([g[0] for g in got]),
                    status=np.concatenate([g[1] for g in got]))
    if kind == "normal":
        scale, ynum, st, _ = eng.xtx_normal(xtypes=s.xtypes, npop=NPOP, weight=s.weight,
                                            ldregress=c["ldregress"], chrom=s.chrom, ppos=s.ppos,
                                            gpos=s.gpos, want_matrix=False)
        ev, vec = eng.eigh_xtx(K)
        return dict(c0=st["c0"], c1=st["c1"], nmiss=st["nmiss"], status=st["status"], scale=scale,
                    ynumsnps=ynum, evals=ev, evecs=vec)
    ev, vec = eng.eigh(s.a, c["nvec"])
    return dict(evals=ev, evecs=vec)


def work(case):
    c, kind = case, case["kind"]
    if kind == "eigh":
        n, v = c["n"], c["nvec"]
        return dict(bytes=8.0 * (n * n + n + v * n), flops=4.0 / 3 * n ** 3 + 2.0 * n * n * v)
    N, M = c["N"], c["M"]
    rows = M * ((N + 3) // 4)
    gram = lambda k: M * (k * (k + 1.0) + 2 * k)  # one sample's normal equations
    if kind in ("pca", "pass", "normal"):
        n = N - c.get("drop", 0)
        flops = 1.0 * n * (n + 1) * M + 4.0 / 3 * n ** 3 + 2.0 * n * n * K
        b = rows + 8.0 * (n + K * n)
        if kind == "pca":
            flops += 4.0 * n * M * K + N * gram(K)
            b += 32.0 * M + 8.0 * K * M + 16.0 * K * N
        if kind == "normal":
            b += 16.0 * M + 8.0 * M * c["weight"]
        return dict(bytes=b, flops=flops)
    if kind == "fast":
        q = (c["I"] + 1) * c["L"]
        return dict(bytes=rows * 1.0 + 8.0 * N * (c["L"] + K),
                    flops=2.0 * M * N * c["L"] * (2 * c["I"] + 1) + 2.0 * M * N * q
                    + 2.0 * (M + N) * q * q)
    if kind == "project":
        return dict(bytes=rows + 8.0 * c["K"] * (N + M) + 16.0 * c["K"] * N,
                    flops=4.0 * N * M * c["K"] + N * gram(c["K"]))
    nq = sum(_requests(c))
    return dict(bytes=nq * (M / 4.0 + 8.0 * c["K"]) + 8.0 * (c["K"] + 2) * M, flops=nq * gram(c["K"]))


# ---------------------------------------------------------------- 64-bit results
def _signed(v):
    """Rows with their largest-|.| component positive."""
    return v * np.sign(v[np.arange(len(v)), np.abs(v).argmax(axis=1)])[:, None]


def _stats(g):
    """Counts and normalisation of code rows g [M, n] (device)."""
    n1 = (g == 1).sum(1)
    n2 = (g == 2).sum(1)
    n3 = (g == 3).sum(1)
    n = g.shape[1]
    c0 = n1 + 2 * n2
    c1 = 2 * (n - n3) - c0
    some = n3 < n
    mean = torch.where(some, c0.double() / (n - n3).clamp(min=1), 0.0)
    p = 0.5 * mean
    y = p * (1 - p)
    fancy = torch.where(y > 0, 1 / torch.sqrt(torch.where(y > 0, y, 1.0)), 1.0)
    fancy = torch.where(some, fancy, 0.0)
    status = torch.where(some, torch.where(torch.minimum(c0, c1) < 1, 1, 0), 2)
    return c0, c1, n3, mean, fancy, status


def _z(g, mean, fancy, keep):
    z = (g.double() - mean[:, None]) * fancy[:, None]
    z[(g == 3) | ~keep[:, None]] = 0.0
    return z


def _steps(M, n):
    step = max(1, CHUNK // n)
    return [slice(m, min(M, m + step)) for m in range(0, M, step)]


def _eig(x, k):
    if len(x) > 3000:  # minutes on the host
        ev, v = torch.linalg.eigh(x)
        ev, v = ev.cpu().numpy(), v[:, -k:].cpu().numpy()
    else:
        ev, v = np.linalg.eigh(x.cpu().numpy())
    return ev[::-1].copy(), _signed(v[:, ::-1][:, :k].T.copy())


def _loadings(g, stats, vec):
    c0, c1, nm, mean, fancy, status = stats
    keep = status == 0
    v = torch.from_numpy(vec).cuda()
    ff = torch.empty((len(v), len(g)), dtype=torch.float64, device="cuda")
    fxv = torch.zeros((len(v), g.shape[1]), dtype=torch.float64, device="cuda")
    for m in _steps(*g.shape):
        z = _z(g[m], mean[m], fancy[m], keep[m])
        ff[:, m] = 10 * (v @ z.t().contiguous())
        fxv += ff[:, m] @ z
    return ff, 1 / torch.sqrt((fxv * fxv).sum(1))


def _project(g, stats, ff, fx):
    """Normal equations and solutions of the samples of g [M, n]."""
    c0, c1, nm, mean, fancy, status = stats
    keep, k, n = status == 0, len(fx), g.shape[1]
    e = fx[:, None] * ff
    iu = torch.triu_indices(k, k)
    G = torch.zeros((len(iu[0]), n), dtype=torch.float64, device="cuda")
    r = torch.zeros((k, n), dtype=torch.float64, device="cuda")
    for m in _steps(*g.shape):
        obs = ((g[m] != 3) & keep[m, None]).double()
        G += (e[iu[0], m] * e[iu[1], m]) @ obs
        r += e[:, m] @ _z(g[m], mean[m], fancy[m], keep[m])
    A = torch.zeros((n, k, k), dtype=torch.float64, device="cuda")
    A[:, iu[0], iu[1]] = G.t()
    A[:, iu[1], iu[0]] = G.t()
    a = np.linalg.solve(A.cpu().numpy(), r.t().cpu().numpy()[:, :, None])[:, :, 0]
    return a.T.copy(), r.cpu().numpy()


def _exact_normal(c, seed):
    g = _geno(c, seed)
    M, n = g.shape
    pop = _pop(n)
    onehot = torch.nn.functional.one_hot(pop, NPOP).double()
    obs = (g != 3).double()
    val = torch.where(g == 3, 0, g).double()
    num, tot = obs @ onehot, val @ onehot
    fill = torch.where(num > 0, tot / num.clamp(min=1), float("nan"))[:, pop]
    y = torch.where(g == 3, fill, val)
    have = ~torch.isnan(y)
    y = torch.where(have, y, 0.0)
    mean = y.sum(1) / have.sum(1).clamp(min=1)
    p = 0.5 * mean
    v = p * (1 - p)
    fancy = torch.where(v > 0, 1 / torch.sqrt(torch.where(v > 0, v, 1.0)), 1.0)
    c0 = val.sum(1)
    c1 = 2 * obs.sum(1) - c0
    keep = torch.minimum(c0, c1) >= 1
    z = (y - mean[:, None]) * fancy[:, None]
    if c["weight"]:
        z *= torch.from_numpy(_weight(c, seed)).cuda()[:, None]
    z[~have | ~keep[:, None]] = 0.0
    x = z.t().contiguous() @ z
    scale = float(torch.trace(x)) / (n - 1)
    ev, vec = _eig(x / scale, K)
    return dict(c0=None, c1=None, nmiss=None, status=None, scale=scale,
                ynumsnps=float(keep.sum()), evals=ev, evecs=vec)


def _exact_fast(c, seed):
    g = _geno(c, seed)
    M, n = g.shape
    c0, c1, nm, mean, fancy, status = _stats(g)
    keep = status != 2
    x = torch.empty((M, n), dtype=torch.float64, device="cuda")
    for m in _steps(M, n):
        x[m] = _z(g[m], mean[m], fancy[m], keep[m]) / math.sqrt(2.0)
    om = np.random.Generator(np.random.PCG64(seed + 7)).standard_normal((n, c["L"]))
    a = torch.from_numpy(om).cuda()
    u = None
    for i in range(c["I"] + 1):
        q = x @ a
        if i < c["I"]:
            a = (q.t().contiguous() @ x).t().contiguous() / M
        # an orthonormal basis of all blocks, one block at a time, twice
        q = q / q.norm(dim=0)
        for _ in range(2):
            if u is not None:
                q = q - u @ (u.t().contiguous() @ q)
            q = torch.from_numpy(np.linalg.qr(q.cpu().numpy())[0]).cuda()
        u = q if u is None else torch.cat([u, q], dim=1)
    b = (u.t().contiguous() @ x).cpu().numpy()
    _, s, vt = np.linalg.svd(b, full_matrices=False)
    return dict(evals=s[:K] ** 2 / M, evecs=_signed(vt[:K].copy()))


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "eigh":
        ev, v = np.linalg.eigh(_covariance(c, seed))
        return dict(evals=ev[::-1].copy(), evecs=_signed(v[:, ::-1][:, :c["nvec"]].T.copy()))
    if kind == "normal":
        return _exact_normal(c, seed) if c["ldregress"] == 0 else None
    if kind == "fast":
        return _exact_fast(c, seed) if c["gen"] == "torch" else None
    g = _geno(c, seed)
    if kind in ("project", "serve"):
        st = _stats(g)
        ff, fx = _loadings(g, st, _axes(c, seed))
        if kind == "project":
            a, b = _project(g, st, ff, fx)
            return dict(ffvecs=ff.cpu().numpy(), fxscal=fx.cpu().numpy(), a=a, b=b, pstatus=None)
        a, _ = _project(_queries(c, seed).t().contiguous(), st, ff, fx)
        return dict(coords=(a * _eigscale(c)[:, None]).T.copy(), status=None)
    sel = torch.from_numpy(_kept(c, seed)).cuda().long()
    gs = g if len(sel) == c["N"] else g[:, sel]
    M, n = gs.shape
    st = _stats(gs)
    c0, c1, nm, mean, fancy, status = st
    x = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    for m in _steps(M, n):
        z = _z(gs[m], mean[m], fancy[m], status[m] == 0)
        x += z.t().contiguous() @ z
    scale = float(torch.trace(x)) / (n - 1)
    ev, vec = _eig(x / scale, K)
    if kind == "pass":
        return dict(scale=scale, evals=ev, evecs=vec)
    ff, fx = _loadings(gs, st, vec)
    a, b = _project(g, st, ff, fx)
    return dict(c0=None, c1=None, nmiss=None, status=None, mean=mean.cpu().numpy(),
                fancy=fancy.cpu().numpy(), scale=scale, evals=ev, evecs=vec,
                ffvecs=ff.cpu().numpy(), fxscal=fx.cpu().numpy(), a=a, b=b, pstatus=None)
