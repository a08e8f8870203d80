"""Performance cases of the framework: public calls on host arrays.

Each case is one call of ``estimate_mi``, ``pairwise_mi`` or
``estimate_entropy`` with the arrays a user's program holds (NumPy, float64
or integer labels), from the call to the returned array.  The sizes are those
of this repository's benchmark configurations and tests, and of the monthly,
daily and hourly series that lag scans are run on.

  listed()             the cases that are followed
  draw(rng)            another case of the same ranges
  prepare(case, seed)  the inputs
  run(state)           one call and its result
  work(case)           bytes and operations no implementation can do without
  exact(case, seed)    the result by brute force in 64 bits (small cases)
"""

import math
import warnings

import numpy as np
import torch

import ennemi_amd

# Brute force is left out beyond this many point pairs of all tasks together.
MOST_PAIRS = 2.5e10


def listed():
    return [
        # One pair of short series, as a tutorial or an interactive session
        # computes it: the latency of a call.
        {"name": "mi_300", "kind": "mi", "n": 300, "nx": 1, "lags": 1, "dz": 0, "k": 3,
         "nan": 0.0, "mask": 0.0},
        # One estimate of a middling sample.
        {"name": "mi_10k", "kind": "mi", "n": 10_000, "nx": 1, "lags": 1, "dz": 0, "k": 3,
         "nan": 0.0, "mask": 0.0},
        # Four drivers of a daily series over two weeks of lags, given a
        # condition, on the days that a mask selects.
        {"name": "lags_cond_mask", "kind": "mi", "n": 3_653, "nx": 4, "lags": 15, "dz": 1, "k": 3,
         "nan": 0.0, "mask": 0.5},
        # The masked lag scan: eight series with gaps, lags -48..48.
        {"name": "lag_scan_776", "kind": "mi", "n": 100_096, "nx": 8, "lags": 97, "dz": 0, "k": 3,
         "nan": 0.3, "mask": 0.0},
        # One conditional estimate with three conditions.
        {"name": "cond3_100k", "kind": "mi", "n": 100_000, "nx": 1, "lags": 1, "dz": 3, "k": 3,
         "nan": 0.0, "mask": 0.0},
        # The largest single estimate: two conditions, two million points.
        {"name": "cond2_2m", "kind": "mi", "n": 2_000_000, "nx": 1, "lags": 1, "dz": 2, "k": 5,
         "nan": 0.0, "mask": 0.0},
        # Many neighbours (smoother estimates), three variables.
        {"name": "mi_k100", "kind": "mi", "n": 20_011, "nx": 3, "lags": 1, "dz": 0, "k": 100,
         "nan": 0.0, "mask": 0.0},
        # Every pair of a wide data set, a tenth of its columns rounded.
        {"name": "pairs_64", "kind": "pairs", "n": 50_000, "nvar": 64, "dz": 0, "k": 3, "nan": 0.0},
        # Pairs of a small data set with gaps, given a condition.
        {"name": "pairs_cond", "kind": "pairs", "n": 5_003, "nvar": 12, "dz": 1, "k": 3, "nan": 0.1},
        # Joint entropy of four variables.
        {"name": "entropy_4d", "kind": "entropy", "n": 100_000, "d": 4, "dz": 0, "k": 3},
        # Continuous variables against class labels.
        {"name": "classes_1m", "kind": "classes", "n": 1_000_000, "nx": 3, "classes": 16, "dz": 0, "k": 3},
        # Two discrete variables.
        {"name": "discrete_1m", "kind": "discrete", "n": 1_000_000, "levels": 50, "dz": 0},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["mi", "mi", "mi", "pairs", "entropy", "classes", "discrete"])
    k = rng.choice([2, 3, 3, 3, 4, 5, 7, 10, 20, 40, 100])
    if kind == "mi":
        dz = rng.choice([0, 0, 0, 1, 1, 2, 3])
        n = _log_int(rng, 300, 100_096 if dz < 3 else 60_000)
        if dz == 0 and rng.random() < 0.15:
            n = _log_int(rng, 100_000, 1_000_000)
        nx, lags = rng.randint(1, 8), rng.choice([1, 3, 12, 25, 49, 97])
        # Points of all tasks: as many as the lag scan's, fewer where the
        # neighbour search has more dimensions or longer lists.
        most = {0: 5e7, 1: 4e6, 2: 1e6, 3: 2e5}[dz] / (1 if k <= 7 else 4 if k <= 20 else 16)
        while n * nx * lags > most and nx * lags > 1:
            if nx >= lags:
                nx -= 1
            else:
                lags = max(1, lags // 2)
        if n > most:
            n = int(most)
        if n - lags < 16 * k:   # masks and gaps leave a third of the rows
            k = 3
        return {"kind": "mi", "n": n, "nx": nx, "lags": lags, "dz": dz, "k": k,
                "nan": rng.choice([0.0, 0.0, 0.05, 0.3]), "mask": rng.choice([0.0, 0.0, 0.5])}
    if kind == "pairs":
        dz = rng.choice([0, 0, 1])
        nvar = rng.randint(3, 64)
        most = (8e7 if dz == 0 else 2e6) / (1 if k <= 7 else 4 if k <= 20 else 16)
        n = max(300, min(_log_int(rng, 300, 50_000), int(most / (nvar * (nvar - 1) / 2))))
        return {"kind": "pairs", "n": n, "nvar": nvar, "dz": dz, "k": k if n >= 16 * k else 3,
                "nan": rng.choice([0.0, 0.0, 0.1])}
    if kind == "entropy":
        d = rng.randint(1, 5)
        return {"kind": "entropy", "n": _log_int(rng, 300, 100_000 if d <= 4 else 30_000), "d": d,
                "dz": rng.choice([0, 0, 1]) if d <= 3 else 0, "k": min(k, 20)}
    if kind == "classes":
        dz = rng.choice([0, 0, 1])
        return {"kind": "classes", "n": _log_int(rng, 1_000, 1_000_000 if dz == 0 else 50_000),
                "nx": rng.randint(1, 3), "classes": rng.randint(2, 20), "dz": dz, "k": min(k, 10)}
    return {"kind": "discrete", "n": _log_int(rng, 300, 1_000_000), "levels": rng.randint(2, 60),
            "dz": rng.choice([0, 0, 1])}


def _series(rng, n, m):
    """m coupled AR(1) series of length n (coefficients 0.3-0.9, each driven
    by the next one with 0.2): sum over j of A^j e(t - j), by doubling."""
    burn = 256
    a = np.diag(np.linspace(0.3, 0.9, m) if m > 1 else np.array([0.6]))
    for j in range(m - 1):
        a[j, j + 1] = 0.2
    s = rng.normal(size=(n + burn, m))
    power, step = a, 1
    while step < burn:
        s[step:] += s[:-step] @ power.T
        power, step = power @ power, 2 * step
    return s[burn:]


def _data(case, seed):
    """The arrays of a case, as a dict of NumPy arrays and options."""
    rng = np.random.default_rng([20, seed])
    n, kind = case["n"], case["kind"]
    if kind == "mi":
        nx, lags, dz = case["nx"], case["lags"], case["dz"]
        s = _series(rng, n, 1 + nx + dz)
        y, x = s[:, 0].copy(), s[:, 1:1 + nx].copy()
        z = s[:, 1 + nx:].copy() if dz else None
        if case["nan"]:
            for j in range(nx):
                x[rng.random(n) < rng.uniform(0.0, case["nan"]), j] = np.nan
        mask = rng.random(n) < case["mask"] if case["mask"] else None
        lag = np.arange(lags) - lags // 2
        return {"y": y, "x": x[:, 0].copy() if nx == 1 else x, "lag": lag, "cond": z, "mask": mask,
                "drop_nan": case["nan"] > 0, "cond_lag": 1 if dz and lags > 1 else 0}
    if kind == "pairs":
        nvar, dz = case["nvar"], case["dz"]
        data = np.empty((n, nvar))
        for c in range(nvar):
            if c % 4 == 0:
                data[:, c] = rng.standard_t(3, size=n)
            elif c % 4 == 1:
                data[:, c] = rng.uniform(-1, 1, size=n)
            elif c % 4 == 2:
                data[:, c] = np.sin(data[:, c - 2]) + 0.3 * rng.normal(size=n)
            else:
                data[:, c] = rng.lognormal(0, 1, size=n)
        for c in range(0, nvar, 10):
            data[:, c] = np.round(data[:, c], 2)
        z = data[:, :dz] + rng.normal(size=(n, dz)) if dz else None
        if case["nan"]:
            for c in range(nvar):
                data[rng.random(n) < rng.uniform(0.0, case["nan"]), c] = np.nan
            if dz:
                z = np.where(np.isnan(z), 0.0, z)
        return {"data": data, "cond": z, "drop_nan": case["nan"] > 0}
    if kind == "entropy":
        d, dz = case["d"], case["dz"]
        a = np.random.default_rng(7).normal(size=(d + dz, d + dz))
        v = rng.normal(size=(n, d + dz)) @ a.T + 0.7 * rng.normal(size=(n, d + dz))
        return {"x": v[:, :d].copy(), "cond": v[:, d:].copy() if dz else None}
    if kind == "classes":
        nx, classes, dz = case["nx"], case["classes"], case["dz"]
        p = (np.arange(classes) + 1.0) ** -1.1
        y = rng.choice(classes, size=n, p=p / p.sum())
        z = rng.normal(size=(n, dz)) if dz else None
        mu = 2.0 * np.cos(2 * np.pi * (np.arange(classes)[:, None] + np.arange(nx)) / classes)
        x = mu[y] + rng.normal(size=(n, nx))
        if dz:
            x += 0.5 * z[:, :1]
        return {"y": y, "x": x[:, 0].copy() if nx == 1 else x, "cond": z}
    levels, dz = case["levels"], case["dz"]
    x = rng.integers(0, levels, size=n)
    y = (x + rng.geometric(0.4, size=n)) % levels
    z = rng.integers(0, 4, size=(n, dz)) if dz else None
    return {"x": x, "y": y, "cond": z}


def prepare(case, seed):
    # A program that marks its variables knows the warnings of small classes.
    warnings.filterwarnings("ignore", message=".*many unique values.*")
    return {"kind": case["kind"], "k": case.get("k", 3), **_data(case, seed)}


def run(s):
    kind = s["kind"]
    if kind == "mi":
        return ennemi_amd.estimate_mi(s["y"], s["x"], s["lag"], k=s["k"], cond=s["cond"], cond_lag=s["cond_lag"],
                                      mask=s["mask"], drop_nan=s["drop_nan"])
    if kind == "pairs":
        return ennemi_amd.pairwise_mi(s["data"], k=s["k"], cond=s["cond"], drop_nan=s["drop_nan"])
    if kind == "entropy":
        return ennemi_amd.estimate_entropy(s["x"], k=s["k"], multidim=True, cond=s["cond"])
    if kind == "classes":
        return ennemi_amd.estimate_mi(s["y"], s["x"], k=s["k"], cond=s["cond"], discrete_y=True)
    return ennemi_amd.estimate_mi(s["y"], s["x"], cond=s["cond"], discrete_x=True, discrete_y=True)


def _shape(case):
    """(estimates, columns of one, columns of input, values of output)."""
    kind, dz = case["kind"], case["dz"]
    if kind == "mi":
        t = case["nx"] * case["lags"]
        return t, 2 + dz, 1 + case["nx"] + dz, t
    if kind == "pairs":
        v = case["nvar"]
        return v * (v - 1) // 2, 2 + dz, v + dz, v * v
    if kind == "entropy":
        return (2 if dz else 1), case["d"] + dz, case["d"] + dz, 1
    if kind == "classes":
        return case["nx"], 1 + dz, 1 + case["nx"] + dz, case["nx"]
    return 1, 2 + dz, 2 + dz, 1


def work(case):
    """Input read and output written once; per point of an estimate, the
    distances to its k neighbours and itself (difference and maximum in each
    column) and a comparison per column and level of a search."""
    n, k = case["n"], case.get("k", 0)
    tasks, cols, inputs, outputs = _shape(case)
    per_point = cols * (2.0 * (k + 1) + math.log2(n))
    return {"bytes": 8.0 * (n * inputs + outputs), "flops": tasks * n * per_point}


# The estimates by brute force over all pairs, in 64 bits.

def _psi(v):
    """The estimators' digamma series at positive integers (float64)."""
    y = v.to(torch.float64)
    p = torch.log(y) - y ** -6 * (y ** 2 * (y ** 2 * (y / 2 + 1 / 12) - 1 / 120) + 1 / 252)
    p = torch.where(y == 1, torch.full_like(p, -0.5772156649015331), p)
    return torch.full_like(p, math.inf) if bool((y == 0).any()) else p


def _psi1(v):
    return float(_psi(torch.tensor([v], dtype=torch.float64))[0])


def _dist(q, p):
    """Maximum-norm distances (rows of q, rows of p)."""
    d = (q[:, :1] - p[:, 0][None, :]).abs_()
    for c in range(1, p.shape[1]):
        d = torch.maximum(d, (q[:, c:c + 1] - p[:, c][None, :]).abs_())
    return d


def _blocks(n):
    step = max(1, (1 << 26) // max(1, n))
    return [(a, min(n, a + step)) for a in range(0, n, step)]


def _radii(p, k):
    n = len(p)
    return torch.cat([_dist(p[a:b], p).topk(k + 1, dim=1, largest=False).values[:, k] if k + 1 <= n else
                      torch.full((b - a,), math.inf, dtype=torch.float64, device=p.device) for a, b in _blocks(n)])


def _count(p, q, eps):
    r = eps - 1e-12
    return torch.cat([(_dist(q[a:b], p) <= r[a:b, None]).sum(dim=1) for a, b in _blocks(len(q))])


def _cuda(*cols):
    return torch.from_numpy(np.column_stack(cols).astype(np.float64)).cuda()


def _rescaled(x, y, z, draw_x=True, draw_y=True):
    """Standardised columns plus the estimators' fixed low-amplitude noise."""
    rng = np.random.default_rng(2_718281828)
    if draw_x:
        x = (x - x.mean()) / x.std()
        x = x + rng.normal(0.0, 1e-10, x.shape)
    if draw_y:
        y = (y - y.mean()) / y.std()
        y = y + rng.normal(0.0, 1e-10, y.shape)
    if z is not None:
        z = (z - z.mean(axis=0)) / z.std(axis=0)
        z = z + rng.normal(0.0, 1e-10, z.shape)
    return x, y, z


def _mi(x, y, z, k):
    x, y, z = _rescaled(x, y, z)
    n = len(x)
    if z is None:
        p = _cuda(x, y)
        eps = _radii(p, k)
        a, b = _count(p[:, :1], p[:, :1], eps), _count(p[:, 1:], p[:, 1:], eps)
        return _psi1(n) + _psi1(k) - float((_psi(a) + _psi(b)).mean())
    p = _cuda(x, y, z)
    eps = _radii(p, k)
    xz, yz, zz = torch.cat([p[:, :1], p[:, 2:]], 1), p[:, 1:], p[:, 2:]
    return _psi1(k) - float((_psi(_count(xz, xz, eps)) + _psi(_count(yz, yz, eps)) - _psi(_count(zz, zz, eps))).mean())


def _ross(x, labels, z, k):
    n = len(x)
    x, _, z = _rescaled(x, None, z, draw_y=False)
    full = _cuda(x) if z is None else _cuda(x, z)
    zz = None if z is None else _cuda(z)
    values, lab = np.unique(labels), torch.from_numpy(labels).cuda()
    total, term = 0.0, 0.0
    for v in values:
        at = (lab == int(v)).nonzero()[:, 0]
        p = full[at]
        eps = _radii(p, k)
        if z is None:
            total += float(_psi(_count(full, p, eps)).sum())
            term += _psi1(len(p)) * (len(p) / n)
        else:
            own = _psi(_count(zz[at], zz[at], eps))
            total += float((_psi(_count(full, p, eps)) + own - _psi(_count(zz, zz[at], eps))).sum())
    if z is None:
        return _psi1(n) + _psi1(k) - total / n - term
    return _psi1(k) - total / n


def _entropy(v, k):
    p = _cuda(v)
    return _psi1(len(v)) - _psi1(k) + v.shape[1] * (float(torch.log(_radii(p, k)).mean()) + math.log(2.0))


def _plugin_mi(x, y):
    n = len(x)
    nx, ny = np.bincount(x), np.bincount(y)
    pair = np.bincount(x.astype(np.int64) * len(ny) + y, minlength=len(nx) * len(ny)).reshape(len(nx), len(ny))
    i, j = np.nonzero(pair)
    c = pair[i, j].astype(np.float64)
    return float(np.sum(c * np.log(n * c / (nx[i].astype(np.float64) * ny[j])))) / n


def exact(case, seed):
    d, n, k, kind = _data(case, seed), case["n"], case.get("k", 3), case["kind"]
    tasks, cols, _, _ = _shape(case)
    if kind != "discrete":
        # About 100 bytes of traffic a pair, more for long neighbour lists.
        cost = 1.0 + 0.25 * (cols - 2) + k / 20
        if float(n) * n * tasks * cost > MOST_PAIRS:
            return None
    if kind == "mi":
        x, y, z = d["x"].reshape(n, -1), d["y"], d["cond"]
        lag, cl = d["lag"], d["cond_lag"]
        hi, lo = max(int(lag.max()), cl, 0), min(int(lag.min()), cl, 0)
        out = np.empty((len(lag), x.shape[1]))
        for i, g in enumerate(lag):
            for j in range(x.shape[1]):
                xs, ys = x[hi - g:n - g + lo, j], y[hi:n + lo]
                zs = None if z is None else z[hi - cl:n - cl + lo]
                keep = np.ones(len(xs), dtype=bool) if d["mask"] is None else d["mask"][hi:n + lo].copy()
                if d["drop_nan"]:
                    keep &= ~np.isnan(xs)
                out[i, j] = _mi(xs[keep], ys[keep], None if zs is None else zs[keep], k)
        return out
    if kind == "pairs":
        data, z = d["data"], d["cond"]
        out = np.full((case["nvar"], case["nvar"]), np.nan)
        for i in range(case["nvar"]):
            for j in range(i + 1, case["nvar"]):
                keep = ~(np.isnan(data[:, i]) | np.isnan(data[:, j]))
                out[i, j] = out[j, i] = _mi(data[keep, i], data[keep, j], None if z is None else z[keep], k)
        return out
    if kind == "entropy":
        if d["cond"] is None:
            return np.asarray(_entropy(d["x"], k))
        return np.asarray(_entropy(np.column_stack((d["x"], d["cond"])), k) - _entropy(d["cond"], k))
    if kind == "classes":
        x = d["x"].reshape(n, -1)
        return np.array([[_ross(x[:, j], d["y"], d["cond"], k) for j in range(x.shape[1])]])
    if d["cond"] is None:
        return np.array([[_plugin_mi(d["x"], d["y"])]])
    g = d["cond"][:, 0]
    return np.array([[sum(float((g == v).sum()) * _plugin_mi(d["x"][g == v], d["y"][g == v])
                          for v in np.unique(g)) / n]])
