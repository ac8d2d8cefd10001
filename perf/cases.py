"""The calls whose time counts: what a program that uses zeus_amd has it do.

A case is one call of a public entry point -- ``run_batch`` (one problem or
many), ``Zeus`` or ``evaluate`` -- on inputs drawn from a seed.  The objectives,
dimensions, boxes, start counts and PSO iterations are those of the package's
own workloads and tests.  Every start runs to its own end (requiredConverged
0): where an early stop takes effect depends on the timing of the GPU, so the
results of such a call differ from one call to the next.

What a call returns has to mean the same number under another order of
summation.  The Gaussian's iterates do, all the way to tol 1e-8.  The other
objectives amplify a rounding error a little in every iteration, so their
MAX_ITER and tolerance keep the results away from their own rounding noise,
and the gradient norm and the counts of starts are not compared where they
rest on it.  The minimum of Rosenbrock is 0: the value there is rounding
noise and its coordinates are what is returned.
"""
import math

import numpy as np
import torch

import zeus_amd as z

#: half width of the box, and the objective's class
BOX = {"rosenbrock": 5.0, "rastrigin": 5.12, "ackley": 32.768, "gaussian": 5.0,
       "dijet": 10.0, "mlp": 2.0}
CLASSES = {"rosenbrock": z.Rosenbrock, "rastrigin": z.Rastrigin, "ackley": z.Ackley}
PRNG = {"xorwow": z.PRNGType.XORWOW, "philox": z.PRNGType.PHILOX}
MAX_ITER = 10000


def solve(kind, dim, problems, starts, max_iter, tol, prng="philox", per_start=False,
          gradient="adjoint", size=0):
    """One call of run_batch on `problems` problems of one class; start counts
    fall from `starts` by up to a quarter (ragged batches)."""
    return {"call": "solve", "kind": kind, "dim": dim, "problems": problems, "starts": starts,
            "pso_iter": 10, "max_iter": max_iter, "tol": tol, "prng": prng,
            "per_start": per_start, "gradient": gradient, "size": size}


def listed():
    return [
        # the smallest call: a two-dimensional function, launches and latency
        {"name": "rosenbrock2_1024", **solve("rosenbrock", 2, 1, 1024, 100, 1e-8, "xorwow")},
        # many local minima, most starts end in one: the hit rate of the
        # global one is what a user asks
        {"name": "rastrigin20_2048", **solve("rastrigin", 20, 1, 2048, 100, 1e-4, "xorwow")},
        {"name": "ackley10_1000", **solve("ackley", 10, 1, 1000, 6, 1e-4)},
        # a long curved valley in 50 dimensions
        {"name": "rosenbrock50_700", **solve("rosenbrock", 50, 1, 700, 30, 1e-8)},
        # a batch of quadratic fits whose starts are all kept (spread of the
        # minimizers), ragged start counts
        {"name": "gaussian32_x6_all", **solve("gaussian", 32, 6, 1000, MAX_ITER, 1e-8,
                                              per_start=True)},
        # the 150-D quadratic at the benchmark's size, and a small call of it
        {"name": "gaussian150_4096", **solve("gaussian", 150, 1, 4096, MAX_ITER, 1e-8)},
        {"name": "gaussian150_100", **solve("gaussian", 150, 1, 100, MAX_ITER, 1e-8, "xorwow")},
        # one fit of a binned spectrum, and a batch of pseudo-experiments
        {"name": "dijet_1x256", **solve("dijet", 4, 1, 256, 8, 1e-8, "xorwow", size=100)},
        {"name": "dijet_64x256", **solve("dijet", 4, 64, 256, 8, 1e-8, size=100)},
        # training a small network from many starts
        {"name": "mlp_512", **solve("mlp", 321, 1, 512, 24, 1e-8, size=256)},
        # a mixed batch: every class at once
        {"name": "mixed_x24", "call": "mixed", "problems": 24, "layout": 42, "most": 2048},
        # a scan of the likelihood: values and gradients at given points
        {"name": "evaluate_dijet_16000", "call": "evaluate", "kind": "dijet", "dim": 4,
         "points": 16000, "gradient": "adjoint", "size": 100},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    which = rng.random()
    prng = rng.choice(["xorwow", "philox"])
    if which < 0.08:
        return {"call": "mixed", "problems": rng.randint(6, 24), "layout": rng.randrange(10**6),
                "most": _log_int(rng, 300, 2048)}
    if which < 0.18:
        kind, dim = rng.choice([("dijet", 4), ("rosenbrock", 10), ("rastrigin", 20),
                                ("gaussian", 32)])
        return {"call": "evaluate", "kind": kind, "dim": dim,
                "points": _log_int(rng, 1000, 16000),
                "gradient": rng.choice(["adjoint", "adjoint", "dual"]) if kind == "dijet"
                else "adjoint", "size": rng.randint(50, 200)}
    kind, dim = rng.choice([("rosenbrock", 2), ("rosenbrock", 10), ("rosenbrock", 50),
                            ("rastrigin", 2), ("rastrigin", 20), ("ackley", 10),
                            ("gaussian", 5), ("gaussian", 32), ("gaussian", 150),
                            ("gaussian", 150), ("dijet", 4), ("dijet", 4), ("mlp", 321)])
    if kind == "gaussian":
        many = rng.random() < 0.4
        return solve(kind, dim, rng.randint(2, 6) if many else 1,
                     _log_int(rng, 64, 700 if many else 4096), MAX_ITER, 1e-8, prng,
                     rng.random() < 0.3)
    if kind == "dijet":
        return solve(kind, dim, rng.choice([1, _log_int(rng, 2, 64)]), _log_int(rng, 64, 256),
                     rng.randint(5, 8), 1e-8, prng, False,
                     rng.choice(["adjoint", "adjoint", "adjoint", "dual"]),
                     rng.randint(50, 100))
    if kind == "mlp":
        return solve(kind, dim, 1, _log_int(rng, 64, 512), rng.randint(10, 24), 1e-8, prng,
                     size=rng.randint(100, 256))
    iters = {("rosenbrock", 2): (20, 100), ("rosenbrock", 10): (8, 12),
             ("rosenbrock", 50): (10, 30), ("rastrigin", 2): (30, 60),
             ("rastrigin", 20): (60, 100), ("ackley", 10): (4, 6)}[kind, dim]
    return solve(kind, dim, 1, _log_int(rng, 128, 2048 if dim < 50 else 1024),
                 rng.randint(*iters), 1e-8 if kind == "rosenbrock" else 1e-4, prng)


# --- inputs: plain data of one problem, from the seed alone -----------------------
def _specs(case, seed):
    """The problems of a case as plain records."""
    if case["call"] == "solve":
        return [dict(kind=case["kind"], dim=case["dim"],
                     n=case["starts"] - (7 * i) % max(1, case["starts"] // 4),
                     max_iter=case["max_iter"], tol=case["tol"], seed=seed + i, stream=i,
                     prng=case["prng"], pso_iter=case["pso_iter"],
                     data=_data(case["kind"], case["dim"], case["size"], seed, i))
                for i in range(case["problems"])]
    rng = np.random.default_rng(case["layout"])
    specs = []
    for i in range(case["problems"]):
        kind, dim, iters, tol = [("rosenbrock", 10, 12, 1e-8), ("rosenbrock", 50, 30, 1e-8),
                                 ("rastrigin", 20, 60, 1e-4), ("ackley", 10, 6, 1e-4),
                                 ("gaussian", 32, MAX_ITER, 1e-8),
                                 ("gaussian", 150, MAX_ITER, 1e-8)][int(rng.integers(0, 6))]
        n = int(round(math.exp(rng.uniform(math.log(128), math.log(case["most"])))))
        specs.append(dict(kind=kind, dim=dim, n=n, max_iter=iters, tol=tol, seed=seed + i,
                          stream=i, prng="xorwow", pso_iter=10,
                          data=_data(kind, dim, 0, seed, i)))
    return specs


def _data(kind, dim, size, seed, i):
    """Gaussian: C = A A^T / D + I.  Dijet: a falling spectrum of `size` bins
    with Poisson counts, 10^4 events expected.  MLP: noisy samples of sin 3x."""
    rng = np.random.default_rng((seed, i))
    if kind == "gaussian":
        a = rng.standard_normal((dim, dim))
        return a @ a.T / dim + np.eye(dim)
    if kind == "dijet":
        x = (1000.0 + (np.arange(size) + 0.5) * (6000.0 / size)) / 13000.0
        shape = (1 - x) ** 10 / x ** (5 + 0.1 * np.log(x))
        return np.stack([x, rng.poisson(1e4 * shape / shape.sum()).astype(np.float64)])
    if kind == "mlp":
        x = rng.uniform(-1, 1, size)
        return np.stack([x, np.sin(3 * x) + 0.1 * rng.standard_normal(size)])
    return None


def _objective(spec):
    kind, data = spec["kind"], spec["data"]
    if kind == "gaussian":
        f = z.Gaussian(data)
    elif kind == "dijet":
        f = z.LogLikelihood(data[1], data[0])
    elif kind == "mlp":
        f = z.Mlp(data[0], data[1])
    else:
        f = CLASSES[kind](spec["dim"])
    f.device_params()  # uploaded once, as a program that calls more than once does
    return f


def _box(kind):
    return (0.0 if kind == "dijet" else -BOX[kind]), BOX[kind]


def _points(case, seed):
    """Points of an evaluate case: inside the box, for the spectrum around its
    own parameters."""
    rng = np.random.default_rng((seed, 1))
    if case["kind"] == "dijet":
        return np.array([0.5, 10.0, 5.0, 0.1]) * rng.uniform(0.7, 1.3, (case["points"], 4))
    lo, hi = _box(case["kind"])
    return rng.uniform(lo, hi, (case["points"], case["dim"]))


def prepare(case, seed):
    if case["call"] == "evaluate":
        spec = dict(kind=case["kind"], dim=case["dim"],
                    data=_data(case["kind"], case["dim"], case["size"], seed, 0))
        return {"case": case, "f": _objective(spec), "points": _points(case, seed)}
    problems = []
    for s in _specs(case, seed):
        lo, hi = _box(s["kind"])
        problems.append(z.Problem(_objective(s), lo, hi, s["n"], s["max_iter"], s["pso_iter"], 0,
                                  s["tol"], s["seed"], s["kind"], stream=s["stream"],
                                  prng=PRNG[s["prng"]]))
    return {"case": case, "problems": problems}


def _outputs(case, results):
    """The results a case is read for (see the head of this file)."""
    out = {"coordinates": np.concatenate([r["x"] for r in results])}
    if case["call"] == "mixed" or (case["kind"], case["dim"]) != ("rosenbrock", 2):
        out["fval"] = np.array([r["fval"] for r in results])
    if case.get("kind") == "gaussian":
        out["gradient_norm"] = np.array([r["gnorm"] for r in results])
        out["claimed"] = np.array([r["claimed"] for r in results])
        out["iterations"] = np.array([r["sum_iter"] for r in results])
    if case.get("per_start"):
        for k in ("x", "fval", "status", "iter"):
            out["all_" + k] = np.concatenate([r["all"][k].reshape(-1) for r in results])
    return out


def run(state):
    case = state["case"]
    if case["call"] == "evaluate":
        f, g = z.evaluate(state["f"], state["points"], case["gradient"])
        return {"value": f, "gradient": g}
    probs = state["problems"]
    if len(probs) == 1 and not case["per_start"]:
        p = probs[0]
        res = [z.Zeus(p.f, p.lower, p.upper, p.N, p.MAX_ITER, p.PSO_ITER, p.requiredConverged,
                      p.fun_name, p.tolerance, p.seed, 0, prng=p.prng, stream=p.stream,
                      gradient=case["gradient"])]
    else:
        res = z.run_batch(probs, gradient=case.get("gradient", "adjoint"),
                          per_start=case.get("per_start", False))
    return _outputs(case, [dict(x=r.coordinates, fval=r.fval, gnorm=r.gradientNorm,
                                claimed=r.c.claimed, sum_iter=r.sum_iter, all=r.per_start)
                           for r in res])


# --- the work of a pass -----------------------------------------------------------
def _cost(kind, dim, size):
    """Floating-point operations of one value (a transcendental function as 20)."""
    return {"rosenbrock": 8 * dim, "rastrigin": 24 * dim, "ackley": 24 * dim + 60,
            "gaussian": 2 * dim * dim, "dijet": 45 * size,
            "mlp": 2 * 321 * size + 33 * 20 * size}[kind]


def work(case):
    """Operations: the PSO's values, and per BFGS iteration the line search's
    values, one gradient (as two values; the Gaussian's comes with the value),
    one product with the inverse Hessian and its rank-2 update.  Iterations and
    values per iteration are the usual ones of each class.  Bytes: parameters in,
    results out (the state of a start need not leave the chip)."""
    if case["call"] == "evaluate":
        per = _cost(case["kind"], case["dim"], case["size"])
        return {"bytes": 8.0 * case["points"] * (2 * case["dim"] + 1),
                "flops": 3.0 * per * case["points"]}
    flops = nbytes = 0.0
    for s in _specs({**case, "size": min(case.get("size", 0), 1)}, 0):
        kind, dim = s["kind"], s["dim"]
        cost = _cost(kind, dim, case.get("size", 0))
        iters, values = {"rosenbrock": (s["max_iter"], 4.0), "rastrigin": (s["max_iter"], 5.0),
                         "ackley": (s["max_iter"], 3.0),
                         "gaussian": ({5: 9, 32: 24}.get(dim, 27), 2.0),
                         "dijet": (s["max_iter"], 11.0), "mlp": (s["max_iter"], 1.6)}[kind]
        iters = min(iters, 40)
        grad = 0.0 if kind == "gaussian" else 2.0
        flops += s["n"] * (cost * (s["pso_iter"] + 2 + iters * (values + grad)) +
                           8.0 * dim * dim * iters)
        nbytes += 8.0 * ((dim * dim if kind == "gaussian" else 3 * case.get("size", 0)) + dim)
        if case.get("per_start"):
            nbytes += s["n"] * (8.0 * dim + 32)
    return {"bytes": nbytes, "flops": flops}


# --- the same results in plain numpy and torch ------------------------------------
def _philox(c0, c1, c2, c3, k0, k1):
    """Philox4x32-10 (Salmon et al., SC'11) on arrays of 64-bit words."""
    m = np.uint64(0xFFFFFFFF)
    c0, c1, c2, c3 = (np.asarray(c, np.uint64) for c in (c0, c1, c2, c3))
    for r in range(10):
        ka = np.uint64((k0 + r * 0x9E3779B9) & 0xFFFFFFFF)
        kb = np.uint64((k1 + r * 0xBB67AE85) & 0xFFFFFFFF)
        p0, p1 = np.uint64(0xD2511F53) * c0, np.uint64(0xCD9E8D57) * c2
        c0, c1, c2, c3 = ((p1 >> np.uint64(32)) ^ c1 ^ ka, p1 & m,
                          (p0 >> np.uint64(32)) ^ c3 ^ kb, p0 & m)
    return c0, c1, c2, c3


def _uniform(hi, lo):
    return (((hi << np.uint64(21)) | (lo >> np.uint64(11))) + np.uint64(1)).astype(
        np.float64) * 2.0**-53


class _Draws:
    """Pairs of uniforms of (start, coordinate) in the order a swarm takes them."""

    def __init__(self, spec):
        self.spec, self.t = spec, 0
        self.start = np.arange(spec["n"], dtype=np.uint64)[:, None]
        self.coord = np.arange(spec["dim"], dtype=np.uint64)[None, :]
        if spec["prng"] == "xorwow":  # Marsaglia 2003, a state per pair
            two, top = np.uint64(2), np.uint64(0xFFFFFFFF)
            a = _philox(two * self.coord, top, self.start, 0, spec["seed"], spec["stream"])
            b = _philox(two * self.coord + np.uint64(1), top, self.start, 0, spec["seed"],
                        spec["stream"])
            self.w = [*a, b[0]]
            self.d = b[1]

    def _next(self):
        m = np.uint64(0xFFFFFFFF)
        t = self.w[0] ^ (self.w[0] >> np.uint64(2))
        v = self.w[4]
        v = (v ^ ((v << np.uint64(4)) & m)) ^ (t ^ ((t << np.uint64(1)) & m))
        self.w = [*self.w[1:], v]
        self.d = (self.d + np.uint64(362437)) & m
        return (v + self.d) & m

    def pair(self):
        s = self.spec
        if s["prng"] == "xorwow":
            return [_uniform(self._next(), self._next()) for _ in range(2)]
        blk = np.uint64(self.t * s["dim"]) + self.coord
        self.t += 1
        o = _philox(blk, 0, self.start, 0, s["seed"], s["stream"])
        return _uniform(o[0], o[1]), _uniform(o[2], o[3])


def _value_and_gradient(spec, dev):
    """x (n x dim, float64) -> values, and values with gradients."""
    kind, dim = spec["kind"], spec["dim"]
    data = None if spec["data"] is None else torch.tensor(spec["data"], device=dev)
    w = 2 * math.pi
    if kind == "gaussian":
        def fg(x):
            g = x @ data
            return 0.5 * (x * g).sum(1), g
    elif kind == "rosenbrock":
        def fg(x):
            a, b = 1 - x[:, :-1], x[:, 1:] - x[:, :-1] ** 2
            g = torch.zeros_like(x)
            g[:, :-1] = -2 * a - 400 * x[:, :-1] * b
            g[:, 1:] += 200 * b
            return (a * a + 100 * b * b).sum(1), g
    elif kind == "rastrigin":
        def fg(x):
            return (10 * dim + (x * x - 10 * torch.cos(w * x)).sum(1),
                    2 * x + 10 * w * torch.sin(w * x))
    elif kind == "ackley":
        def fg(x):
            r = ((x * x).sum(1) / dim).sqrt()
            e1, e2 = torch.exp(-0.2 * r), torch.exp(torch.cos(w * x).sum(1) / dim)
            g = (4 * e1 / (dim * r))[:, None] * x + (w / dim * e2)[:, None] * torch.sin(w * x)
            return -20 * e1 - e2 + 20 + math.e, g
    elif kind == "dijet":
        x0, k = data[0], data[1]
        lg, l1, l0 = torch.lgamma(k + 1), torch.log1p(-x0), torch.log(x0)

        def fg(t):
            mean = t[:, :1] * (1 - x0) ** t[:, 1:2] / x0 ** (t[:, 2:3] + t[:, 3:4] * l0)
            wm = mean - k
            return ((mean + lg) - k * torch.log(mean)).sum(1), torch.stack(
                [(wm / t[:, :1]).sum(1), (wm * l1).sum(1), -(wm * l0).sum(1),
                 -(wm * l0 * l0).sum(1)], 1)
    else:
        px, py = data[0], data[1]

        def fg(t):
            n = t.shape[0]
            w1, b1 = t[:, 0:32:2], t[:, 1:32:2]
            m = t[:, 32:304].reshape(n, 16, 17)
            w2, b2, w3, b3 = m[:, :, :16], m[:, :, 16], t[:, 304:320], t[:, 320]
            h1 = torch.tanh(w1[:, :, None] * px + b1[:, :, None])
            h2 = torch.tanh(w2 @ h1 + b2[:, :, None])
            d = (w3[:, :, None] * h2).sum(1) + b3[:, None] - py
            dy = 2 / px.numel() * d
            d2 = dy[:, None] * w3[:, :, None] * (1 - h2 * h2)
            d1 = (w2.transpose(1, 2).contiguous() @ d2) * (1 - h1 * h1)
            g1 = torch.stack([(d1 * px).sum(2), d1.sum(2)], 2).reshape(n, 32)
            g2 = torch.cat([d2 @ h1.transpose(1, 2).contiguous(), d2.sum(2)[:, :, None]],
                           2).reshape(n, 272)
            return (d * d).mean(1), torch.cat(
                [g1, g2, (dy[:, None] * h2).sum(2), dy.sum(1)[:, None]], 1)
    return fg


def _first_min(v):
    return int(torch.nan_to_num(v, nan=math.inf).argmin())


def _swarm(spec, fg, dev):
    """Best positions of the swarm after its iterations (w 0.5, c1 1.2, c2 1.5)."""
    lo, hi = _box(spec["kind"])
    draws = _Draws(spec)

    def pair():
        return [torch.tensor(u, device=dev) for u in draws.pair()]
    u0, u1 = pair()
    vr = 0.1 * (hi - lo)
    x, v = lo + (hi - lo) * u0, -vr + 2 * vr * u1
    best, fb = x.clone(), fg(x)[0]
    m = _first_min(fb)
    gx, gv = best[m].clone(), float(fb[m])
    for _ in range(spec["pso_iter"]):
        u0, u1 = pair()
        v = 0.5 * v + 1.2 * u0 * (best - x) + 1.5 * u1 * (gx - x)
        x = x + v
        f = fg(x)[0]
        imp = f < fb
        fb = torch.where(imp, f, fb)
        best = torch.where(imp[:, None], x, best)
        m = _first_min(fb)
        if float(fb[m]) < gv:
            gx, gv = best[m].clone(), float(fb[m])
    return best


def _minimize(spec, dev):
    """BFGS with a backtracking line search (20 halvings, Armijo 0.1) from every
    start of the swarm, all starts side by side with dense inverse Hessians."""
    fg = _value_and_gradient(spec, dev)
    x = _swarm(spec, fg, dev)
    n, dim = x.shape
    f, g = fg(x)
    p = -g
    H = torch.eye(dim, device=dev, dtype=torch.float64).repeat(n, 1, 1)
    status = torch.full((n,), -1, device=dev, dtype=torch.int64)
    iters = torch.zeros_like(status)
    fval = f.clone()
    for it in range(spec["max_iter"]):
        live = status < 0
        if not bool(live.any()):
            break
        ddir = (g * p).sum(1)
        alpha = torch.ones_like(f)
        todo, f1 = live.clone(), f.clone()
        for _ in range(20):
            ft = fg(x + alpha[:, None] * p)[0]
            f1 = torch.where(todo, ft, f1)
            todo = todo & ~((ft <= f + 0.1 * alpha * ddir) & (ft < f))
            if not bool(todo.any()):
                break
            alpha = torch.where(todo, 0.5 * alpha, alpha)
        xt = x + alpha[:, None] * p
        ft, gn = fg(xt)
        f1 = torch.where(todo, ft, f1)
        s, y = xt - x, gn - g
        v = (H @ gn[:, :, None])[:, :, 0]
        u = v + p
        sy = (s * y).sum(1)
        upd = live & ~(sy.abs() < 1e-14)
        rho = 1 / torch.where(upd, sy, torch.ones_like(sy))
        a = (0.5 * (rho * rho * (y * u).sum(1) + rho))[:, None] * s - rho[:, None] * u
        a, s = (torch.where(upd[:, None], q, torch.zeros_like(q)) for q in (a, s))
        H += s[:, :, None] * a[:, None, :]
        H += a[:, :, None] * s[:, None, :]
        acc = live & (f1 < f)
        hg = torch.where(acc[:, None], v, -p)
        f = torch.where(acc, f1, f)
        x, g = (torch.where(acc[:, None], q, r) for q, r in ((xt, x), (gn, g)))
        p = -(hg + s * (a * g).sum(1)[:, None] + a * (s * g).sum(1)[:, None])
        nrm = (g * g).sum(1).sqrt()
        bad = live & ~(torch.isfinite(nrm) & torch.isfinite(f1))
        done = live & ~bad & (nrm < spec["tol"])
        fval = torch.where(bad, f1, torch.where(live, f, fval))
        status = torch.where(bad, 5, torch.where(done, 1, status))
        iters = torch.where(live, it + (status < 0).long(), iters)
    status = torch.where(status < 0, 0, status)
    m = _first_min(fval)
    gn = float((g * g).sum(1).sqrt()[m])
    return dict(x=x[m].cpu().numpy(), fval=float(fval[m]), gnorm=gn,
                claimed=int((status == 1).sum()), sum_iter=int(iters.sum()),
                all=dict(x=x.cpu().numpy(), fval=fval.cpu().numpy(),
                         status=status.cpu().numpy(), iter=iters.cpu().numpy()))


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    if case["call"] == "evaluate":
        spec = dict(kind=case["kind"], dim=case["dim"],
                    data=_data(case["kind"], case["dim"], case["size"], seed, 0))
        f, g = _value_and_gradient(spec, dev)(torch.tensor(_points(case, seed), device=dev))
        return {"value": f.cpu().numpy(), "gradient": g.cpu().numpy()}
    if case["call"] == "solve" and case["kind"] == "dijet" and case["problems"] > 16:
        return None  # too slow one problem after the other
    return _outputs(case, [_minimize(s, dev) for s in _specs(case, seed)])
