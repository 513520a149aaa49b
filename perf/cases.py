"""The measured workloads: what a program using this framework has it do.

Each case names its kind and its sizes; the kinds are

  job        the reference's own use: burn-in!, run-sampler!, sample! of a small correlated-Gaussian
             ensemble, then mean, variance and histogram of the draws
  run        run-sampler! of an ordinary ensemble (thousands to hundreds of thousands of walkers)
  posterior  a library posterior (binomial likelihood, beta prior) at the library's walker counts:
             burn-in!, the ensemble's mean, variance and histogram, sample!
  move       burn-in! and sample! of a large ensemble, where the move itself is memory traffic
  dataset    mean, variance and histogram of a data matrix on the GPU
  plot       what a plot of a library distribution needs: direct draws, their estimates, densities
  acor       autocorrelation of a recorded series
  logistic   a logistic regression declared by form: guarded reduced-precision chain and log
             densities of given points
  linear     a linear regression declared by form: run-sampler! and log densities of given points
  batch      many hierarchical beta-binomials in one launch: burn-in and a recorded run
  glm_batch  many fp8 logistic regressions in lockstep: burn-in and an accounted run

A chain continues from pass to pass, as a program's does; two runs of the same passes from the same
seed give the same positions.
"""
import math

import numpy as np
import torch

from bayadera_amd import _lib, engine, library, models

A = 2.0
WGS = 256
PRIOR_SD = 5.0
# guard of the accept test (log units) that each precision is used with
GUARDS = {"fp16": 6e-3, "fp16x2": 2e-3, "bf16x3": 2e-3}
PRECISIONS = {"fp16": _lib.BH_GLM_FP16, "fp16x2": _lib.BH_GLM_FP16X2, "bf16x3": _lib.BH_GLM_BF16X3,
              "fp32": _lib.BH_GLM_FP32, "fp64": _lib.BH_GLM_FP64}

_keep = {}


def _factory():
    if "factory" not in _keep:
        _keep["factory"] = engine.HipBayaderaFactory(0, WGS)
    return _keep["factory"]


def _library():
    if "library" not in _keep:
        _keep["library"] = library.Library(_factory())
    return _keep["library"]


def _compiled(model, dim):
    """The compiled sampler factory of a model, which a program keeps."""
    key = (model, dim)
    if key not in _keep:
        m = models.mvn_model(dim) if model == "mvn" else models.diag_gaussian_model(dim)
        _keep[key] = _factory().mcmc_factory(m)
    return _keep[key]


def listed():
    return [
        # the reference's own test ensemble: 1024 walkers on one work-group, steps bound by latency
        {"name": "job_1024x4", "kind": "job", "dim": 4, "walkers": 1024, "burn": 256, "steps": 1024,
         "columns": 1 << 18},
        # an ordinary ensemble of an odd dimension: launches of some microseconds each
        {"name": "run_65536x7", "kind": "run", "model": "mvn", "dim": 7, "walkers": 65536, "steps": 128,
         "partner": "flat"},
        # a library posterior with the library's default number of walkers
        {"name": "posterior_2p24", "kind": "posterior", "walkers": 1 << 24, "burn": 8},
        # a large ensemble with wide records
        {"name": "move_2p22x16", "kind": "move", "model": "mvn", "dim": 16, "walkers": 1 << 22, "burn": 8,
         "partner": "walker"},
        # the estimates of a large data matrix
        {"name": "dataset_16Mx4", "kind": "dataset", "rows": 1 << 24, "dim": 4},
        # the smallest calls: draws and densities for a plot
        {"name": "plot_65536", "kind": "plot", "n": 65536},
        # a long recorded run of two coordinates
        {"name": "acor_112640x2", "kind": "acor", "steps": 112640, "dim": 2},
        # the large logistic regression: one-term fp16 on the matrix cores, guarded
        {"name": "logistic_1Mx64", "kind": "logistic", "rows": 1_000_000, "dim": 64, "walkers": 16384,
         "precision": "fp16", "steps": 8, "points": 512},
        # a small one of odd row and point counts, two fp16 terms
        {"name": "logistic_50021x32", "kind": "logistic", "rows": 50021, "dim": 32, "walkers": 2048,
         "precision": "fp16x2", "steps": 32, "points": 1000},
        # linear regression, plain fp32
        {"name": "linear_100kx16", "kind": "linear", "rows": 100_000, "dim": 16, "walkers": 8192, "steps": 64,
         "points": 1024},
        # thousands of small hierarchical posteriors at once
        {"name": "batch_4096", "kind": "batch", "problems": 4096, "groups": 50, "walkers": 256, "burn": 8,
         "steps": 16, "state": "global"},
        # many fp8 logistic regressions of uneven sizes
        {"name": "glm_batch_64", "kind": "glm_batch", "problems": 64, "rows": 50000, "walkers": 2048, "burn": 2,
         "steps": 4, "precision": "fp16x2"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _walkers(rng, lo, hi):
    return max(lo, _log(rng, lo, hi) // (2 * WGS) * (2 * WGS))


def draw(rng):
    kind = rng.choice(["job", "run", "posterior", "move", "dataset", "plot", "acor", "logistic", "linear",
                       "batch", "glm_batch"])
    c = {"kind": kind}
    if kind == "job":
        w = rng.choice([512, 1024, 1536, 2048])
        c.update(dim=rng.randint(1, 5), walkers=w, burn=_log(rng, 64, 512), steps=_log(rng, 64, 1024),
                 columns=_log(rng, 1 << 12, 1 << 18))
    elif kind == "run":
        w = _walkers(rng, 4096 + 512, 1 << 17)
        c.update(model=rng.choice(["mvn", "diag"]), dim=rng.randint(1, 16), walkers=w, steps=_log(rng, 64, 192),
                 partner=rng.choice(["flat", "walker"]))
    elif kind == "posterior":
        c.update(walkers=_walkers(rng, 1 << 16, 1 << 24), burn=rng.randint(2, 8))
    elif kind == "move":
        dim = rng.randint(2, 32)
        c.update(model="mvn" if dim <= 16 else "diag", dim=dim, walkers=_walkers(rng, 1 << 18, (1 << 26) // dim),
                 burn=rng.randint(2, 8), partner=rng.choice(["flat", "walker"]))
    elif kind == "dataset":
        dim = rng.randint(1, 20)
        c.update(rows=_log(rng, 10_000, (1 << 26) // dim), dim=dim)
    elif kind == "plot":
        c.update(n=_log(rng, 1024, 1 << 22) * 4)
    elif kind == "acor":
        c.update(steps=_log(rng, 400, 200_000), dim=rng.randint(1, 8))
    elif kind == "logistic":
        c.update(rows=_log(rng, 10_000, 500_000), dim=rng.choice([32, 64]), walkers=_walkers(rng, 1024, 8192),
                 precision=rng.choice(["fp16", "fp16x2", "bf16x3"]), steps=rng.randint(4, 16),
                 points=rng.randint(100, 1500))
    elif kind == "linear":
        c.update(rows=_log(rng, 2_000, 150_000), dim=rng.randint(2, 32), walkers=_walkers(rng, 1024, 8192),
                 steps=rng.randint(50, 64), points=rng.randint(100, 2000))
    elif kind == "batch":
        c.update(problems=_log(rng, 64, 4096), groups=rng.randint(8, 50), walkers=rng.choice([128, 256, 512]),
                 burn=rng.randint(2, 8), steps=rng.randint(2, 16), state=rng.choice(["global", "lds"]))
    else:
        c.update(problems=rng.randint(4, 64), rows=_log(rng, 4_000, 50_000), walkers=rng.choice([512, 1024, 2048]),
                 burn=rng.randint(1, 2), steps=rng.randint(2, 4), precision=rng.choice(["fp16x2", "bf16x3"]))
    return c


# ---------------------------------------------------------------------------------------------
# inputs, made from the seed alone
# ---------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _gaussian_params(model, dim, seed):
    rng = np.random.default_rng([seed, dim])
    mu = rng.standard_normal(dim)
    if model == "mvn":
        a = rng.standard_normal((dim, dim))
        p = np.linalg.inv(a @ a.T + np.eye(dim)).reshape(-1)
    else:
        p = 1.0 / rng.uniform(0.5, 2.0, dim) ** 2
    return np.concatenate([mu, p]).astype(np.float32)


def _sampler(model, dim, walkers, seed, partner, warm):
    s = _compiled(model, dim).create_sampler(seed, walkers, _gaussian_params(model, dim, seed))
    s.set_partner(_lib.BH_PARTNER_FLAT if partner == "flat" else _lib.BH_PARTNER_WALKER)
    s.init_position(seed + 1, np.tile(np.array([-4.0, 4.0], np.float32), dim))
    s.burn_in(warm, A)
    return s


def _matrix(rows, dim, seed):
    """Draws as a sampler leaves them: correlated columns of different scales and offsets."""
    g = _generator(seed)
    x = torch.randn(rows, dim, generator=g, device="cuda")
    scale = torch.rand(dim, generator=g, device="cuda") * 3.0 + 0.25
    shift = torch.randn(dim, generator=g, device="cuda") * 2.0
    return (x * scale + 0.5 * x[:, :1] + shift).contiguous()


def _series(steps, dim, seed):
    """Ensemble means of a chain with autocorrelation times of some tens of steps (an AR(1) series per
    coordinate, by the powers of its coefficient in blocks)."""
    g = torch.Generator().manual_seed(int(seed))
    rho = 1.0 - 0.2 * torch.rand(dim, generator=g, dtype=torch.float64) - 0.02
    e = torch.randn(steps, dim, generator=g, dtype=torch.float64)
    x = e
    k = 1
    while k < 512:  # x_t = sum over j < 512 of rho^j e_(t-j)
        y = x.clone()
        y[k:] += x[:-k] * rho ** k
        x, k = y, 2 * k
    return (0.1 * x + 1.5).to(torch.float32).cuda()


def _logistic_data(rows, dim, points, seed):
    g = _generator(seed)
    x = (torch.randn(rows, dim, generator=g, device="cuda") / math.sqrt(dim)).to(torch.bfloat16)
    beta = torch.randn(dim, generator=g, device="cuda")
    eta = (x.float() * beta).sum(1)
    y = (torch.rand(rows, generator=g, device="cuda") < torch.sigmoid(eta)).to(torch.float32)
    # the posterior's sd per coordinate: Fisher information rows / dim * E[sigma'], 0.21 at eta ~ N(0, 1)
    sd = math.sqrt(dim / (0.21 * rows))
    p = beta + sd * torch.randn(points, dim, generator=g, device="cuda")
    return x, y, beta, sd, p.contiguous()


def _linear_data(rows, dim, points, seed):
    g = _generator(seed)
    x = torch.randn(rows, dim, generator=g, device="cuda")
    beta = torch.randn(dim, generator=g, device="cuda")
    y = (x * beta).sum(1) + 0.5 * torch.randn(rows, generator=g, device="cuda")
    centre = torch.cat([beta, torch.tensor([math.log(0.5)], device="cuda")])
    sd = 0.5 / math.sqrt(rows)
    p = centre + sd * torch.randn(points, dim + 1, generator=g, device="cuda")
    return x, y, centre, sd, p.contiguous()


def _hierarchical(problems, groups, seed):
    size = np.random.default_rng([problems, groups]).integers(min(5, groups), groups + 1, problems)
    rng = np.random.default_rng([seed, problems])
    n = np.round(np.exp(rng.uniform(math.log(10.0), math.log(1e5), (problems, groups))))
    theta = rng.beta(2.0, 5.0, (problems, groups))
    y = rng.binomial(n.astype(np.int64), theta).astype(np.float64)
    t = np.log((y + 0.5) / (n - y + 0.5))
    limits = np.zeros((problems, groups + 2, 2), np.float32)
    limits[:, 0] = [0.0, 1.5]
    limits[:, 1] = [0.5, 2.0]
    limits[:, 2:, 0] = t - 0.05
    limits[:, 2:, 1] = t + 0.05
    params = [np.concatenate([n[i, :k], y[i, :k], [10.0]]).astype(np.float32) for i, k in enumerate(size)]
    return params, [int(k) + 2 for k in size], limits


def _fp8_problems(problems, rows, seed):
    """Row counts log-uniform up to `rows`, 8 to 64 columns, e4m3 codes with a scale per column."""
    rng = np.random.default_rng([problems, rows])
    g = _generator(seed)
    codes, scales, labels = [], [], []
    limits = np.zeros((problems, 64, 2), np.float32)
    for p in range(problems):
        n = int(round(math.exp(rng.uniform(math.log(1000.0), math.log(rows)))))
        d = int(rng.choice([8, 16, 32, 64]))
        x = torch.randn(n, d, generator=g, device="cuda") / math.sqrt(d)
        s = x.abs().amax(0) / 448.0
        q = (x / s).to(torch.float8_e4m3fn)
        beta = torch.randn(d, generator=g, device="cuda")
        eta = (q.float() * s * beta).sum(1)
        labels.append((torch.rand(n, generator=g, device="cuda") < torch.sigmoid(eta)).float().cpu().numpy())
        codes.append(q.view(torch.uint8).cpu().numpy())
        scales.append(s.cpu().numpy())
        b, sd = beta.cpu().numpy(), math.sqrt(d / (0.21 * n))
        limits[p, :d, 0] = b - 2 * sd
        limits[p, :d, 1] = b + 2 * sd
    return models.GlmBatchModel(codes, scales, labels, PRIOR_SD), limits


def prepare(case, seed):
    c, fac, kind = case, _factory(), case["kind"]
    st = {"case": c}
    if kind == "job":
        st["sampler"] = _sampler("mvn", c["dim"], c["walkers"], seed, "flat", 16)
        st["draws"] = torch.empty(c["columns"], c["dim"], device="cuda")
    elif kind == "run":
        st["sampler"] = _sampler(c["model"], c["dim"], c["walkers"], seed, c["partner"], 16)
    elif kind == "posterior":
        rng = np.random.default_rng(seed)
        lib = _library()
        if "posterior" not in _keep:
            prior = lib.beta(2.0, 3.0)
            _keep["posterior"] = models.posterior_model(prior.model, "bb", lib.likelihood("binomial"))
        n = int(rng.integers(40, 400))
        k = int(rng.integers(n // 8, n - n // 8))
        prior = lib.beta(1.5 + rng.random(), 2.0 + rng.random())
        dist = library.Posterior(lib, _keep["posterior"], np.array([n, k], np.float32), prior)
        s = lib.mcmc_factory(dist.model).create_sampler(seed, c["walkers"], dist.params)
        s.init_position(seed + 1, np.asarray(dist.start_box(), np.float32))
        s.burn_in(16, A)
        st.update(sampler=s, draws=torch.empty(c["walkers"], 1, device="cuda"))
    elif kind == "move":
        st["sampler"] = _sampler(c["model"], c["dim"], c["walkers"], seed, c["partner"], 4)
        st["draws"] = torch.empty(c["walkers"], c["dim"], device="cuda")
    elif kind == "dataset":
        st["data"] = _matrix(c["rows"], c["dim"], seed)
    elif kind == "plot":
        # the distribution and the seed of its draws; the density is asked on an even grid
        mu, sigma = _plot_params(seed)
        dist = _library().gaussian(mu, sigma)
        x = torch.empty(c["n"], device="cuda")
        grid = torch.linspace(mu - 5 * sigma, mu + 5 * sigma, c["n"], device="cuda").reshape(-1, 1)
        st.update(seed=seed, direct=fac.direct_sampler_engine(dist.model), params=dist.params,
                  density=_library().distribution_engine(dist.model), draws=x, grid=grid,
                  pdf=torch.empty(c["n"], device="cuda"), log_pdf=torch.empty(c["n"], device="cuda"))
    elif kind == "acor":
        st["series"] = _series(c["steps"], c["dim"], seed)
    elif kind == "logistic":
        x, y, beta, sd, p = _logistic_data(c["rows"], c["dim"], c["points"], seed)
        model = models.glm_logistic_model(x.view(torch.int16).cpu().numpy().view(np.uint16), y.cpu().numpy(),
                                          PRIOR_SD)
        sf = fac.mcmc_factory(model)
        s = sf.create_sampler(seed, c["walkers"], np.zeros(1, np.float32))
        s.set_glm_precision(PRECISIONS[c["precision"]]).set_partner(_lib.BH_PARTNER_WALKER)
        s.set_glm_guard(GUARDS[c["precision"]])
        b = beta.cpu().numpy()
        s.init_position(seed + 1, np.stack([b - 2 * sd, b + 2 * sd], 1))
        s.burn_in(4, A)
        st.update(factory=sf, sampler=s, points=p, draws=torch.empty(c["walkers"], c["dim"], device="cuda"))
    elif kind == "linear":
        x, y, centre, sd, p = _linear_data(c["rows"], c["dim"], c["points"], seed)
        sf = fac.mcmc_factory(models.glm_gaussian_model(x.cpu().numpy(), y.cpu().numpy()))
        s = sf.create_sampler(seed, c["walkers"], np.zeros(1, np.float32))
        s.set_partner(_lib.BH_PARTNER_WALKER)
        b = centre.cpu().numpy()
        s.init_position(seed + 1, np.stack([b - 3 * sd, b + 3 * sd], 1))
        s.burn_in(4, A)
        st.update(factory=sf, sampler=s, points=p, draws=torch.empty(c["walkers"], c["dim"] + 1, device="cuda"))
    elif kind == "batch":
        params, dims, limits = _hierarchical(c["problems"], c["groups"], seed)
        key = ("hbb", c["groups"])
        if key not in _keep:
            _keep[key] = models.hbb_model(c["groups"])
        b = fac.batch(_keep[key], params, dims, [1] * len(dims), c["walkers"])
        if c["state"] == "global":
            b.set_state(_lib.BH_BATCH_STATE_GLOBAL)
        b.init_position(seed + 1, limits)
        b.burn_in(seed + 2, 4, A)
        st.update(batch=b, seed=seed, series=torch.empty(c["steps"] * sum(dims), device="cuda"))
    else:
        m, limits = _fp8_problems(c["problems"], c["rows"], seed)
        b = fac.glm_batch(m, c["walkers"]).set_precision(PRECISIONS[c["precision"]])
        b.init_position(seed + 1, limits)
        b.burn_in(seed + 2, 2, A)
        st.update(batch=b, seed=seed, series=torch.empty(c["steps"] * int(m.dims.sum()), device="cuda"))
    return st


def _plot_params(seed):
    rng = np.random.default_rng(seed)
    return float(np.float32(rng.uniform(-3.0, 3.0))), float(np.float32(rng.uniform(0.5, 2.0)))


# ---------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------
def _estimates(data):
    de = _factory().dataset_engine()
    h = de.histogram(data)
    return {"mean": de.data_mean(data), "variance": de.data_variance(data), "limits": h.limits, "pdf": h.pdf,
            "ranks": h.bin_ranks}


def _ran(r):
    ac = r["autocorrelation"]
    return {"acceptance": r["acceptance-rate"], "means": r["means"], "tau": ac.tau, "mean": ac.mean,
            "sigma": ac.sigma}


def run(st):
    c, kind = st["case"], st["case"]["kind"]
    if kind == "job":
        s = st["sampler"]
        s.burn_in(c["burn"], A)
        out = _ran(s.run_sampler(c["steps"], A))
        s.sample(c["columns"], out=st["draws"])
        out["draws"] = st["draws"]
        out["estimates"] = _estimates(st["draws"])
        return out
    if kind == "run":
        s = st["sampler"]
        out = _ran(s.run_sampler(c["steps"], A))
        out["positions"], out["logfn"], _ = s.state()
        return out
    if kind == "posterior":
        s = st["sampler"]
        s.burn_in(c["burn"], A)
        h = s.histogram()
        out = {"mean": s.mean(), "variance": s.variance(), "limits": h.limits, "pdf": h.pdf, "ranks": h.bin_ranks}
        out["draws"] = s.sample(out=st["draws"])
        return out
    if kind == "move":
        s = st["sampler"]
        s.burn_in(c["burn"], A)
        return s.sample(out=st["draws"])
    if kind == "dataset":
        return _estimates(st["data"])
    if kind == "plot":
        x = st["direct"].sample(st["seed"], st["params"], c["n"], out=st["draws"])
        out = _estimates(x)
        out["draws"] = x
        out["pdf_at"] = st["density"].density(st["params"], st["grid"], out=st["pdf"])
        out["log_pdf_at"] = st["density"].log_density(st["params"], st["grid"], out=st["log_pdf"])
        return out
    if kind == "acor":
        ac = _factory().acor_engine().acor(st["series"])
        return {"tau": ac.tau, "mean": ac.mean, "sigma": ac.sigma}
    if kind == "logistic":
        s = st["sampler"]
        s.burn_in(c["steps"], A)
        return {"acceptance": s.acc_rate(A), "draws": s.sample(out=st["draws"]),
                "log_density": st["factory"].log_density(st["points"], PRECISIONS[c["precision"]])}
    if kind == "linear":
        s = st["sampler"]
        out = _ran(s.run_sampler(c["steps"], A))
        out["draws"] = s.sample(out=st["draws"])
        out["log_density"] = st["factory"].log_density(st["points"], _lib.BH_GLM_FP32)
        return out
    b = st["batch"]
    b.burn_in(st["seed"] + 3, c["burn"], A)
    r = b.run(st["seed"] + 4, c["steps"], A, series=st["series"])
    return {"acceptance": r["acceptance-rate"], "mean": r["mean"], "sd": r["sd"], "series": st["series"]}


# ---------------------------------------------------------------------------------------------
# what one pass cannot do without
# ---------------------------------------------------------------------------------------------
def work(case):
    c, kind = case, case["kind"]

    def moves(walkers, dim, steps, density):
        # a walker-step reads its record, its partner's and its log density, and writes the accepted
        # third; about 100 integer operations for its draws, 6 per coordinate, and the density
        return walkers * steps * (8 * dim + 4 + (4 * dim + 4) / 3), walkers * steps * (100 + 6 * dim + density)

    def estimates(rows, dim):
        return 3 * 4 * rows * dim, 16 * rows * dim

    if kind == "job":
        s = -(-c["columns"] // c["walkers"])
        _, f = moves(c["walkers"], c["dim"], c["burn"] + c["steps"] + s, 2 * c["dim"] ** 2)
        eb, ef = estimates(c["columns"], c["dim"])
        return {"bytes": 4 * c["dim"] * (2 * c["walkers"] + c["steps"] + c["columns"]) + eb, "flops": f + ef}
    if kind == "run":
        d = c["dim"]
        b, f = moves(c["walkers"], d, c["steps"], 2 * d * d if c["model"] == "mvn" else 4 * d)
        return {"bytes": b, "flops": f}
    if kind == "posterior":
        b, f = moves(c["walkers"], 1, c["burn"] + 1, 20)
        return {"bytes": b + 12 * c["walkers"] + 8 * c["walkers"], "flops": f + 16 * c["walkers"]}
    if kind == "move":
        d = c["dim"]
        b, f = moves(c["walkers"], d, c["burn"] + 1, 2 * d * d if c["model"] == "mvn" else 4 * d)
        return {"bytes": b + 8 * d * c["walkers"], "flops": f}
    if kind == "dataset":
        b, f = estimates(c["rows"], c["dim"])
        return {"bytes": b, "flops": f}
    if kind == "plot":
        b, f = estimates(c["n"], 1)
        return {"bytes": b + 20 * c["n"], "flops": f + 60 * c["n"]}
    if kind == "acor":
        n = c["steps"] * c["dim"]
        return {"bytes": 4 * n, "flops": n * 2 * min(64, max(10, c["steps"] // 5))}
    if kind == "logistic":
        # per row and point: the product, then an exponential, a logarithm and their sums
        pairs = c["rows"] * (c["walkers"] * (c["steps"] + 2) + c["points"])
        half_steps = 2 * (c["steps"] + 2) + 1
        return {"bytes": half_steps * 2 * c["rows"] * c["dim"], "flops": pairs * (2 * c["dim"] + 6)}
    if kind == "linear":
        pairs = c["rows"] * (c["walkers"] * (c["steps"] + 1) + c["points"])
        half_steps = 2 * (c["steps"] + 1) + 1
        return {"bytes": half_steps * 4 * c["rows"] * (c["dim"] + 1), "flops": pairs * (2 * c["dim"] + 3)}
    if kind == "batch":
        d = (c["groups"] + min(5, c["groups"])) / 2 + 2
        steps = c["burn"] + c["steps"]
        ws = c["problems"] * c["walkers"]
        return {"bytes": ws * 4 * (2 * d + 2) + c["problems"] * c["steps"] * 4 * d,
                "flops": ws * steps * (100 + 6 * d + 24 * d)}
    mean_rows = (c["rows"] - 1000) / math.log(c["rows"] / 1000)
    steps = c["burn"] + c["steps"]
    return {"bytes": c["problems"] * mean_rows * 30 * 2 * steps,
            "flops": c["problems"] * mean_rows * c["walkers"] * steps * (2 * 30 + 6)}


# ---------------------------------------------------------------------------------------------
# the same in 64 bits, without the framework
# ---------------------------------------------------------------------------------------------
def _philox(counter, key):
    """Philox4x32-10 (Salmon, Moraes, Dror, Shaw, SC'11) on uint64 arrays holding 32-bit words."""
    mask = np.uint64(0xFFFFFFFF)
    c, k = [np.asarray(w, np.uint64) for w in counter], list(key)
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), p1 & mask,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), p0 & mask]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    return [(0.5 + (w >> np.uint64(9)).astype(np.float64)) * 2.0 ** -23 for w in c]


def _estimates64(x):
    """Of a float32 matrix; the ranks are an order of equal counts and have no such value."""
    n, m = x.shape
    lo, hi = x.min(0), x.max(0)
    pdf = np.zeros((m, WGS))
    for j in range(m):
        a = x[:, j].astype(np.float64)
        b = np.minimum(((a - lo[j]) / (float(hi[j]) - float(lo[j])) * WGS).astype(np.int64), WGS - 1)
        pdf[j] = np.bincount(b, minlength=WGS) * (WGS / n) / (float(hi[j]) - float(lo[j]))
    x64 = x.astype(np.float64)
    return {"mean": x64.mean(0), "variance": x64.var(0), "limits": np.stack([lo, hi], 1).astype(np.float64),
            "pdf": pdf, "ranks": None}


def _acor64(x, wgs):
    """Goodman's estimator as the reference groups it (amd_gcn.clj:216-267, amd-gcn-acor.cl): the sums of a
    level run over slices of wgs points; in its own slice a point past gsize - lag reads as zero."""
    n = x.size
    lag0 = max(min(min(n // 5, wgs), 64), 10)
    mu = x.mean()
    x = x - mu

    def level(v, lag, width):
        size = v.size
        v2 = v.copy()
        v2[max(size - lag, 0):] = 0.0
        c0 = float(np.dot(v2, v2))
        at = np.arange(size)
        tail = np.minimum(at // width * width + width, size)
        acc = np.zeros(size)
        for s in range(1, lag + 1):
            j = at + s
            inside = j < tail
            jj = np.minimum(j, size - 1)
            acc += np.where(inside, v2[jj], np.where(j < size, v[jj], 0.0))
        return c0, float(np.dot(v2, v2 + 2.0 * acc))

    c0, d = level(x, lag0, wgs)
    start, prev, stride, lag, size = c0, c0, 1, lag0, n
    while True:
        tau = d / (c0 if stride == 1 else prev)
        lag2 = lag if lag * 5 < size else max(size // 5, 10)
        if not (10 < lag2 and lag2 < tau * 5):
            scale = stride * (size - lag2)
            return d * (n - lag) / (scale * start), mu, math.sqrt(d / (scale * n))
        half = size // 2
        x = x[0:2 * half:2] + x[1:2 * half:2]
        prev = c0
        c0, d = level(x, lag2, min(wgs, half))
        stride, lag, size = 2 * stride, lag2, half


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "dataset":
        return _estimates64(_matrix(c["rows"], c["dim"], seed).cpu().numpy())
    if kind == "plot":
        mu, sigma = _plot_params(seed)
        i = np.arange(c["n"] // 4, dtype=np.uint64)
        one = np.ones_like(i)
        u = _philox([i, one * np.uint64(0xF00DCAFE), one * np.uint64(0xDEADBEEF), one * np.uint64(0xBEEFF00D)],
                    [int(seed) & 0xFFFFFFFF, 0xDECAFAAA])
        ra, rb = np.sqrt(-2.0 * np.log(u[1])), np.sqrt(-2.0 * np.log(u[3]))
        two_pi = 2.0 * math.pi
        z = np.stack([np.sin(two_pi * u[0]) * ra, np.cos(two_pi * u[0]) * ra, np.sin(two_pi * u[2]) * rb,
                      np.cos(two_pi * u[2]) * rb], 1).reshape(-1)
        x = mu + sigma * z
        out = _estimates64(x.astype(np.float32).reshape(-1, 1))
        grid = torch.linspace(mu - 5 * sigma, mu + 5 * sigma, c["n"], device="cuda").cpu().numpy().astype(np.float64)
        lp = -0.5 * ((grid - mu) / sigma) ** 2 - math.log(sigma) - 0.5 * math.log(2.0 * math.pi)
        # a draw that rounds to the other side of a bin's edge moves one count
        out.update(draws=x, pdf_at=np.exp(lp), log_pdf_at=lp)
        return out
    if kind == "acor":
        s = _series(c["steps"], c["dim"], seed).cpu().numpy().astype(np.float64)
        r = np.array([_acor64(s[:, j], WGS) for j in range(c["dim"])])
        return {"tau": r[:, 0], "mean": r[:, 1], "sigma": r[:, 2]}
    if kind == "logistic":
        x, y, _, _, p = _logistic_data(c["rows"], c["dim"], c["points"], seed)
        p = p.double()
        lp = -0.5 * (p * p).sum(1) / PRIOR_SD ** 2
        for r0 in range(0, c["rows"], 1 << 17):
            eta = x[r0:r0 + (1 << 17)].double() @ p.t()
            lp = lp + y[r0:r0 + (1 << 17)].double() @ eta - torch.nn.functional.softplus(
                eta, threshold=1e9).sum(0)
        return {"acceptance": None, "draws": None, "log_density": lp.cpu().numpy()}
    if kind == "linear":
        x, y, _, _, p = _linear_data(c["rows"], c["dim"], c["points"], seed)
        p = p.double()
        b, ls = p[:, :c["dim"]].contiguous(), p[:, c["dim"]]
        ss = torch.zeros(c["points"], dtype=torch.float64, device="cuda")
        for r0 in range(0, c["rows"], 1 << 15):
            res = y[r0:r0 + (1 << 15)].double()[:, None] - x[r0:r0 + (1 << 15)].double() @ b.t()
            ss = ss + (res * res).sum(0)
        lp = (-c["rows"] * (ls + 0.5 * math.log(2.0 * math.pi)) - 0.5 * torch.exp(-2.0 * ls) * ss
              - 0.5 * ((b * b).sum(1) / 100.0 + ls * ls))
        return {"acceptance": None, "means": None, "tau": None, "mean": None, "sigma": None, "draws": None,
                "log_density": lp.cpu().numpy()}
    return None  # a chain's positions are those of its own arithmetic
