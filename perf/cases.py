"""Performance cases: what users of this package have it do, over the sizes they do it at.

Four kinds of work, all on one GPU and through the public entry points:

  call      evaluate the interpolant at a batch of points (`ip(x)`)
  jacobian  the dense Jacobian (`ip.gradient(x)`)
  step      forward and backward through `ip.differentiable(x)`
  serve     requests of mixed sizes against several resident interpolants (`NativeServer`)

A case is a dict of plain values: the kind, the node family, the input dimension `d`, the budget `t`
of the index set (k_j = log((2 + j) / log 2)), the number of outputs `o`, of points `p`, and the
precision.  `n`, the size of the index set that `t` gives, is there for the reader.
"""

import math
import random

import numpy as np
import torch

from smolyax_amd import nodes
from smolyax_amd.interpolation import SmolyakBarycentricInterpolator
from smolyax_amd.serving import NativeServer
from smolyax_amd.workloads import k_rule

# Budgets t by (d, |Lambda|) of the benchmark's configurations and of the reference's runtime grid
T_D10_N1000 = 8.831424
T_D1000_N10000 = 8.22451968
T_D160_N10000 = 8.56884
T_D40_N10000 = 9.44952
T_D200_N5000 = 7.85360448
T_D100_N10000 = 8.7492300


def listed():
    return [
        # A first look at a small problem, a handful of points per call inside another program's
        # loop (the smallest batch of the reference's benchmark): launches and host work.
        dict(name="few_points_fp64", kind="call", nodes="leja", d=10, t=T_D10_N1000, n=1000, o=1,
             p=50, precision="fp64"),
        # The headline: a scalar quantity of interest of a 1000-dimensional parameter, a Monte
        # Carlo batch, in the faster precision and in the default one.
        dict(name="scalar_mixed", kind="call", nodes="leja", d=1000, t=T_D1000_N10000, n=9999, o=1,
             p=16384, precision="mixed"),
        dict(name="scalar_fp64", kind="call", nodes="leja", d=1000, t=T_D1000_N10000, n=9999, o=1,
             p=16384, precision="fp64"),
        # The far corner of the reference's own runtime grid (160 inputs, 160 outputs, 5000 points).
        dict(name="vector_fp64", kind="call", nodes="leja", d=160, t=T_D160_N10000, n=10002, o=160,
             p=5000, precision="fp64"),
        # Gaussian inputs, a few outputs, a batch of the same grid.
        dict(name="hermite_few_outputs_fp64", kind="call", nodes="hermite", d=40, t=T_D40_N10000,
             n=9994, o=10, p=500, precision="fp64"),
        # A surrogate with a vector-valued output, in the faster precision.
        dict(name="vector_mixed", kind="call", nodes="leja", d=200, t=T_D200_N5000, n=5000, o=256,
             p=8192, precision="mixed"),
        # A surrogate whose output is a field: dense contraction, FP32 and BF16.
        dict(name="field_mixed", kind="call", nodes="leja", d=100, t=T_D100_N10000, n=9986, o=4096,
             p=4096, precision="mixed"),
        dict(name="field_bf16", kind="call", nodes="leja", d=100, t=T_D100_N10000, n=9986, o=4096,
             p=4096, precision="bf16"),
        # Sensitivities of the scalar quantity, and of the vector at a ragged number of points.
        dict(name="jacobian_scalar", kind="jacobian", nodes="leja", d=1000, t=T_D1000_N10000,
             n=9999, o=1, p=4096, precision="fp64"),
        dict(name="jacobian_vector", kind="jacobian", nodes="leja", d=200, t=T_D200_N5000, n=5000,
             o=256, p=999, precision="fp64"),
        # The interpolant as a layer of a program that trains or inverts through it.
        dict(name="step_fp64", kind="step", nodes="leja", d=200, t=T_D200_N5000, n=5000, o=256,
             p=8192, precision="fp64"),
        # A serving process: 32 requests of 1 to 4096 points that are pending at once, against 8
        # resident interpolants on Gauss-Hermite nodes.
        dict(name="serve_mix", kind="serve", resident=8, requests=32, spec=0, precision="mixed"),
    ]


# ------------------------------------------------------------------------------------------------
# drawn cases

def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _budget(d, n):
    """t with |Lambda| close to n (bisection on the count of the index set)."""
    lo, hi = 1.0, 2.0
    while len(_index_set(d, hi, n)) < n:
        hi *= 1.3
    for _ in range(14):
        mid = 0.5 * (lo + hi)
        if len(_index_set(d, mid, n + 1)) > n:
            hi = mid
        else:
            lo = mid
    return round(lo, 6)


def draw(rng):
    kind = rng.choice(["call", "call", "call", "jacobian", "step", "serve"])
    if kind == "serve":
        return dict(kind=kind, resident=rng.randint(3, 8), requests=rng.randint(8, 32),
                    spec=rng.randrange(1, 1 << 20), precision="mixed")
    d = _log_int(rng, 10, 1000)
    n = _log_int(rng, 100, 10000 if d >= 40 else 2000)
    outputs = rng.choice(["one", "few", "many"])
    if kind == "call":
        family = rng.choice(["leja", "leja", "hermite"])
        precision = rng.choice(["fp64", "fp64", "mixed"] if family == "hermite" else
                               ["fp64", "fp64", "newton-fp64", "mixed", "bf16"])
        o = 1 if outputs == "one" else _log_int(rng, 2, 15) if outputs == "few" else \
            _log_int(rng, 16, 2048)
        p = _log_int(rng, 1, 16384)
        # multiply-adds of the contraction, kept below those of the listed cases of the precision
        most = {"fp64": 6e9 if o >= 16 else 2e8, "newton-fp64": 4e10, "mixed": 1e11,
                "bf16": 1.6e11}[precision]
        p = max(1, min(p, int(most / (n * o))))
    elif kind == "jacobian":
        family, precision = "leja", "fp64"
        o = 1 if outputs == "one" else _log_int(rng, 2, 8) if outputs == "few" else \
            _log_int(rng, 9, 512)
        p = max(1, min(_log_int(rng, 1, 4096), int(4e8 / (8 * d * o)), int(2e9 / (n * o))))
    else:
        family, precision = "leja", rng.choice(["fp64", "newton-fp64", "mixed"])
        o = 1 if outputs == "one" else _log_int(rng, 2, 512)
        p = max(1, min(_log_int(rng, 16, 8192), int((6e9 if o >= 16 else 2e8) / (n * o))))
    t = _budget(d, n)
    return dict(kind=kind, nodes=family, d=d, t=t, n=len(_index_set(d, t)), o=o, p=p,
                precision=precision)


# ------------------------------------------------------------------------------------------------
# inputs

def _function(family, d, o, seed):
    """The target, seeded: exp(-c . x) for one output on [-1, 1]^d, else sin(A x + b)."""
    rng = np.random.default_rng(seed)
    if o == 1 and family == "leja":
        c = rng.uniform(0.5, 1.5, (d, 1)) / (np.arange(d)[:, None] + 1.0) ** 2
        return lambda x: np.exp(-(np.asarray(x) @ c))
    a = rng.standard_normal((d, o)) / (np.arange(d)[:, None] + 1.0) ** 2
    b = rng.uniform(0.0, 2.0 * np.pi, o)
    return lambda x: np.sin(np.asarray(x) @ a + b)


def _points(family, p, d, seed):
    """Uniform on [-1, 1]^d (Leja) or N(0, I) (Gauss-Hermite), FP64, on the GPU."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    if family == "leja":
        return torch.rand((p, d), dtype=torch.float64, device="cuda", generator=gen) * 2.0 - 1.0
    return torch.randn((p, d), dtype=torch.float64, device="cuda", generator=gen)


def _interpolant(family, d, t, o, seed, precision):
    node_gen = nodes.Leja(dim=d) if family == "leja" else \
        nodes.GaussHermite(scaling=np.full(d, np.sqrt(2.0)))
    ip = SmolyakBarycentricInterpolator(d_out=o, node_gen=node_gen, k=k_rule(d), t=t,
                                        precision=precision)
    ip.set_f(f=_function(family, d, o, seed), vectorized=True)
    return ip


def _serving(case):
    """Resident interpolants (d, t, o) and requests (interpolant, points) of a serving case: d,
    |Lambda|, o and the batch sizes log-uniform over the ranges of the serving workload."""
    rng = random.Random(case["spec"])
    resident = []
    for _ in range(case["resident"]):
        d = _log_int(rng, 8, 500)
        t = _budget(d, _log_int(rng, 50, min(4000, 60 * d)))
        resident.append((d, t, _log_int(rng, 1, 1024)))
    requests = [(rng.randrange(case["resident"]), _log_int(rng, 1, 4096))
                for _ in range(case["requests"])]
    return resident, requests


def prepare(case, seed):
    if case["kind"] == "serve":
        resident, requests = _serving(case)
        ips = {f"ip{i}": _interpolant("hermite", d, t, o, seed * 100 + i, case["precision"])
               for i, (d, t, o) in enumerate(resident)}
        xs = [(f"ip{i}", _points("hermite", p, resident[i][0], seed * 100 + r))
              for r, (i, p) in enumerate(requests)]
        return dict(kind="serve", server=NativeServer(ips), requests=xs)
    ip = _interpolant(case["nodes"], case["d"], case["t"], case["o"], seed, case["precision"])
    x = _points(case["nodes"], case["p"], case["d"], seed)
    state = dict(kind=case["kind"], ip=ip, x=x)
    if case["kind"] == "step":
        state["x"] = x.requires_grad_()
        state["w"] = _cotangent(case, seed)
    return state


def _cotangent(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed + 1)
    return torch.randn((case["p"], case["o"]), dtype=torch.float64, device="cuda", generator=gen)


def run(state):
    if state["kind"] == "call":
        return state["ip"](state["x"])
    if state["kind"] == "jacobian":
        return state["ip"].gradient(state["x"])
    if state["kind"] == "step":
        y = state["ip"].differentiable(state["x"])
        (gx,) = torch.autograd.grad(y, state["x"], state["w"])
        return y.detach(), gx
    server = state["server"]
    reqs = [server.submit(name, x) for name, x in state["requests"]]
    server.drain()
    server.completed.clear()
    return [r.y for r in reqs]


def _call_work(d, n, o, p, coefficient_bytes):
    return dict(bytes=8.0 * p * d + 8.0 * p * o + coefficient_bytes * n * o,
                flops=p * n * (1.0 + 2.0 * o))


def work(case):
    """The polynomial has |Lambda| terms: one product per term and point, one multiply-add per
    term, point and output; per (term, factor) pair the same for a derivative."""
    if case["kind"] == "serve":
        resident, requests = _serving(case)
        total = dict(bytes=0.0, flops=0.0)
        for i, p in requests:
            d, t, o = resident[i]
            w = _call_work(d, len(_index_set(d, t)), o, p, 4)
            total = {key: total[key] + w[key] for key in total}
        return total
    d, o, p = case["d"], case["o"], case["p"]
    terms = _index_set(d, case["t"])
    n, pairs = len(terms), sum(len(nu) for nu in terms)
    size = {"fp64": 8, "newton-fp64": 8, "mixed": 4, "bf16": 2}[case["precision"]]
    if case["kind"] == "call":
        return _call_work(d, n, o, p, size)
    if case["kind"] == "jacobian":
        return dict(bytes=8.0 * p * d + 8.0 * p * o * d + 8.0 * n * o,
                    flops=p * pairs * (1.0 + 2.0 * o))
    fwd = _call_work(d, n, o, p, size)
    # backward: the cotangents and the coefficients contracted to one weight per term and point,
    # then two operations per (term, factor) pair
    return dict(bytes=fwd["bytes"] + 16.0 * p * d + 8.0 * p * o + size * n * o,
                flops=fwd["flops"] + p * (2.0 * n * o + 2.0 * pairs))


# ------------------------------------------------------------------------------------------------
# the same interpolants from their definition, in 64 bits

def _index_set(d, t, stop=None):
    """Multi-indices ((dim, degree), ...) with sum k_j nu_j < t; `stop`: no more than that many."""
    k = k_rule(d).tolist()
    found, stack = [], [(0, float(t), ())]
    while stack:
        i, rest, nu = stack.pop()
        found.append(nu)
        if stop is not None and len(found) >= stop:
            break
        while i < d and k[i] < rest:
            m = 1
            while m * k[i] < rest:
                stack.append((i + 1, rest - m * k[i], nu + ((i, m),)))
                m += 1
            i += 1
    return found


def _leja_nodes(m):
    x = [0.0, 1.0, -1.0, 1 / math.sqrt(2), -1 / math.sqrt(2)]
    while len(x) <= m:
        j = len(x)
        x.append(-x[j - 1] if j % 2 == 0 else math.sqrt((x[(j + 1) // 2] + 1) / 2))
    return np.array(x[: m + 1])


def _newton_basis(xi, x, m):
    """prod_{r < m} (x - xi_r) / (xi_m - xi_r) and its derivative."""
    h, dh = torch.ones_like(x), torch.zeros_like(x)
    for r in range(m):
        c = 1.0 / (xi[m] - xi[r])
        dh = (dh * (x - xi[r]) + h) * c
        h = h * (x - xi[r]) * c
    return h, dh


class _Newton:
    """Leja interpolant as a Newton sum over the index set: H (terms x points) and surpluses S."""

    def __init__(self, d, t, f, x):
        dev = x.device
        self.terms = sorted(_index_set(d, t), key=len)
        row = {nu: i for i, nu in enumerate(self.terms)}
        top = max((m for nu in self.terms for _, m in nu), default=0)
        xi = _leja_nodes(top)
        grid = np.full((len(self.terms), d), xi[0])
        for i, nu in enumerate(self.terms):
            for j, m in nu:
                grid[i, j] = xi[m]
        s = torch.as_tensor(f(grid), device=dev).reshape(len(self.terms), -1).clone()
        self.pairs = {}   # (dim, degree) -> rows that hold the factor, the same rows without it
        for i, nu in enumerate(self.terms):
            for pos, (j, m) in enumerate(nu):
                rows, rest = self.pairs.setdefault((j, m), ([], []))
                rows.append(i)
                rest.append(row[nu[:pos] + nu[pos + 1:]])
        for j, m in sorted(self.pairs):
            rows, rest = self.pairs[j, m]
            for r in range(m):
                h = math.prod((xi[m] - xi[q]) / (xi[r] - xi[q]) for q in range(r))
                lower = rest if r == 0 else \
                    [row[tuple(sorted(self.terms[b] + ((j, r),)))] for b in rest]
                s[rows] -= h * s[lower]
        self.s = s
        tab, self.slope, at = [], {}, {}
        for j, m in self.pairs:
            h, dh = _newton_basis(xi, x[:, j], m)
            at[j, m] = len(tab)
            tab.append(h)
            self.slope[j, m] = dh
        self.h = torch.ones((len(self.terms), x.shape[0]), dtype=torch.float64, device=dev)
        tab = torch.stack(tab) if tab else None
        for size in range(1, max(map(len, self.terms)) + 1):
            rows = [i for i, nu in enumerate(self.terms) if len(nu) == size]
            self.h[rows] = self.h[[row[self.terms[i][:-1]] for i in rows]] * \
                tab[[at[self.terms[i][-1]] for i in rows]]

    def value(self):
        return self.h.t() @ self.s

    def by_dim(self):
        """(dim, rows, derivatives of the rows' products with respect to that dim)."""
        dims = {}
        for (j, m), (rows, rest) in self.pairs.items():
            dims.setdefault(j, []).append((rows, self.h[rest] * self.slope[j, m]))
        for j, parts in dims.items():
            yield j, sum((rows for rows, _ in parts), []), torch.cat([dd for _, dd in parts])


def _hermite_value(d, t, f, x):
    """Gauss-Hermite interpolant as the combination of its tensor-product interpolants."""
    zeta = {}
    for nu in _index_set(d, t):
        for mask in range(1 << len(nu)):
            low = tuple((j, m - (mask >> b & 1)) for b, (j, m) in enumerate(nu)
                        if m - (mask >> b & 1) > 0)
            zeta[low] = zeta.get(low, 0) + (-1) ** bin(mask).count("1")
    xi, basis = {}, {}
    y, used = None, [(nu, z) for nu, z in zeta.items() if z]
    centre = math.sqrt(2.0) * np.polynomial.hermite.hermgauss(1)[0][0]
    for at in range(0, len(used), 256):
        part, grids = used[at: at + 256], []
        for nu, _ in part:
            axes = []
            for j, m in nu:
                if m not in xi:
                    xi[m] = math.sqrt(2.0) * np.polynomial.hermite.hermgauss(m + 1)[0]
                if (j, m) not in basis:
                    rows = []
                    for a in range(m + 1):
                        b = torch.ones_like(x[:, j])
                        for q in range(m + 1):
                            if q != a:
                                b = b * ((x[:, j] - xi[m][q]) / (xi[m][a] - xi[m][q]))
                        rows.append(b)
                    basis[j, m] = torch.stack(rows)
                axes.append(xi[m])
            mesh = np.meshgrid(*axes, indexing="ij") if axes else []
            grid = np.full((math.prod(len(a) for a in axes), d), centre)
            for (j, _), g in zip(nu, mesh):
                grid[:, j] = g.reshape(-1)
            grids.append(grid)
        values = torch.as_tensor(f(np.concatenate(grids)), device=x.device)
        weights = []
        for nu, z in part:
            w = torch.full((1, x.shape[0]), float(z), dtype=torch.float64, device=x.device)
            for j, m in nu:
                w = (w[:, None, :] * basis[j, m][None]).reshape(-1, x.shape[0])
            weights.append(w)
        add = torch.cat(weights).t() @ values.reshape(len(values), -1)
        y = add if y is None else y + add
    return y


def exact(case, seed):
    if case["kind"] == "serve":
        resident, requests = _serving(case)
        out = []
        for r, (i, p) in enumerate(requests):
            d, t, o = resident[i]
            out.append(_hermite_value(d, t, _function("hermite", d, o, seed * 100 + i),
                                      _points("hermite", p, d, seed * 100 + r)))
        return out
    d, t, o = case["d"], case["t"], case["o"]
    f = _function(case["nodes"], d, o, seed)
    x = _points(case["nodes"], case["p"], d, seed)
    if case["nodes"] == "hermite":
        return _hermite_value(d, t, f, x)
    newton = _Newton(d, t, f, x)
    if case["kind"] == "call":
        return newton.value()
    if case["kind"] == "jacobian":
        jac = torch.zeros((case["p"], o, d), dtype=torch.float64, device=x.device)
        for j, rows, dd in newton.by_dim():
            jac[:, :, j] = dd.t() @ newton.s[rows]
        return jac
    weight = newton.s @ _cotangent(case, seed).t().contiguous()
    gx = torch.zeros_like(x)
    for j, rows, dd in newton.by_dim():
        gx[:, j] = (weight[rows] * dd).sum(0)
    return newton.value(), gx
