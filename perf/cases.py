"""Performance cases of the transfer framework.

Each case is one call pattern of a user's program through the public Python
entry points, on clouds resident in device memory:

* ``transfer``: build a moving-least-squares operator for new clouds and
  apply it (the coupling step of a moving mesh);
* ``apply``: apply an operator that the program keeps (a fixed mesh);
* ``adjoint``: the differentiable transfer, forward and backward;
* ``batch``: rebuild a batch of uneven operators after its points moved, and
  apply it;
* ``knn``: the neighbour search on its own;
* ``nearest``: build and apply the nearest-neighbour operator;
* ``spline``: build and apply the radial-basis spline operator.

Clouds: ``cube`` (uniform, targets inside the sources' box), ``graded``
(density falling away from a corner by orders of magnitude, as a refined
mesh) and ``shell`` (a thin spherical shell).
"""
import math

import numpy as np
import torch

import datatransferkit_amd as dtk
from datatransferkit_amd.autograd import mls_transfer

_BASIS = {"constant": 1, "linear": 4, "quadratic": 10}
_CASE = {
    "path": "transfer", "cloud": "cube", "n_src": 0, "n_tgt": 0, "fields": 1,
    "basis": "linear", "k": 0, "rbf": "wendland0", "precision": "fp64",
    "solver": "classical", "geometry": "float", "truncation": "absolute",
}


def _case(**kw):
    return dict(_CASE, **kw)


def listed():
    fast = dict(precision="fp32_bulk", solver="cholesky")
    return [
        # the operator's defaults on a cloud of a small component: a call
        # whose launches count more than its work
        _case(name="small_default", n_src=1003, n_tgt=1201),
        # the defaults at the size of a surface mesh
        _case(name="linear_10k", n_src=10_000, n_tgt=10_000),
        # the drop-in solver with the quadratic basis and its own k
        _case(name="quadratic_dropin", n_src=120_011, n_tgt=80_021, fields=4,
              basis="quadratic", k=10, rbf="wendland2"),
        # the headline transfer of the benchmark
        _case(name="quadratic_1m_fp32", n_src=1_000_000, n_tgt=1_000_000, fields=4,
              basis="quadratic", k=32, rbf="wendland2", **fast),
        # all-double accuracy: a finer target mesh than the sources
        _case(name="quadratic_double", n_src=150_001, n_tgt=300_007, fields=3,
              basis="quadratic", k=16, rbf="wendland4", geometry="double",
              solver="cholesky"),
        # an ill-conditioned surface: truncated systems in mixed precision
        _case(name="shell_fp32", cloud="shell", n_src=300_000, n_tgt=300_000, fields=4,
              basis="quadratic", k=32, rbf="wendland4", truncation="relative", **fast),
        # a kept operator applied every time step
        _case(name="apply_kept", path="apply", n_src=500_000, n_tgt=700_001, fields=4,
              basis="quadratic", k=32, rbf="wendland2", solver="cholesky"),
        # an optimisation step through the transfer
        _case(name="adjoint_100k", path="adjoint", n_src=200_000, n_tgt=100_000,
              fields=8, basis="quadratic", k=16, rbf="wendland2", geometry="double",
              solver="cholesky"),
        # many uneven operators rebuilt from moved points in a time loop
        _case(name="batch_rebuild", path="batch", problems=512, n_src=8192, n_tgt=0,
              rbf="wendland2", **fast),
        # neighbour lists of a refined mesh
        _case(name="knn_graded", path="knn", cloud="graded", n_src=100_003, n_tgt=90_001,
              k=64),
        # nearest-neighbour transfer at full size
        _case(name="nearest_1m", path="nearest", n_src=1_000_000, n_tgt=1_000_000,
              fields=4),
        # a spline transfer: a Krylov solve over the sources
        _case(name="spline_150k", path="spline", n_src=150_000, n_tgt=200_003),
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    fast = dict(precision="fp32_bulk", solver="cholesky")
    rbf = rng.choice(["wendland0", "wendland2", "wendland4"])
    kind = rng.choice(["default", "dropin", "fp32", "fp32", "double", "shell", "apply",
                       "adjoint", "batch", "knn", "knn", "nearest", "spline"])
    if kind == "default":
        return _case(n_src=_size(rng, 500, 200_000), n_tgt=_size(rng, 500, 200_000),
                     fields=rng.randint(1, 4), rbf=rbf, k=rng.choice([0, 0, 8]))
    if kind == "dropin":
        return _case(n_src=_size(rng, 2000, 150_000), n_tgt=_size(rng, 2000, 75_000),
                     fields=rng.randint(1, 4), basis="quadratic",
                     k=rng.choice([10, 16, 32]), rbf=rbf)
    if kind == "fp32":
        return _case(n_src=_size(rng, 2000, 1_000_000), n_tgt=_size(rng, 2000, 900_000),
                     fields=rng.randint(1, 4), basis=rng.choice(["linear", "quadratic"]),
                     k=rng.choice([16, 24, 32]), rbf=rbf, **fast)
    if kind == "double":
        return _case(n_src=_size(rng, 2000, 300_000), n_tgt=_size(rng, 2000, 300_000),
                     fields=rng.randint(1, 4), basis=rng.choice(["linear", "quadratic"]),
                     k=rng.choice([16, 20, 32]), rbf=rbf, geometry="double",
                     solver="cholesky")
    if kind == "shell":
        return _case(cloud="shell", n_src=_size(rng, 20_000, 300_000),
                     n_tgt=_size(rng, 20_000, 300_000), fields=rng.randint(1, 4),
                     basis="quadratic", k=32, rbf="wendland4", truncation="relative",
                     **fast)
    if kind == "apply":
        solver = rng.choice(["fp64", "fp32"])
        return _case(path="apply", n_src=_size(rng, 2000, 500_000),
                     n_tgt=_size(rng, 2000, 700_000), fields=rng.randint(1, 8),
                     basis="quadratic", k=rng.choice([16, 24, 32]), rbf=rbf,
                     **(dict(solver="cholesky") if solver == "fp64" else fast))
    if kind == "adjoint":
        return _case(path="adjoint", n_src=_size(rng, 2000, 200_000),
                     n_tgt=_size(rng, 2000, 100_000), fields=rng.randint(1, 8),
                     basis=rng.choice(["linear", "quadratic"]), k=rng.choice([16, 24]),
                     rbf="wendland2", geometry="double", solver="cholesky")
    if kind == "batch":
        form = fast if rng.random() < 0.7 else dict(solver="cholesky")
        return _case(path="batch", problems=_size(rng, 16, 512),
                     n_src=_size(rng, 512, 8192), n_tgt=0, rbf="wendland2", **form)
    if kind == "knn":
        return _case(path="knn", cloud=rng.choice(["cube", "graded"]),
                     n_src=_size(rng, 1000, 100_000), n_tgt=_size(rng, 1000, 100_000),
                     k=rng.choice([1, 5, 10, 20, 32, 50, 64]),
                     geometry=rng.choice(["float", "float", "double"]))
    if kind == "nearest":
        return _case(path="nearest", n_src=_size(rng, 2000, 1_000_000),
                     n_tgt=_size(rng, 2000, 1_000_000), fields=rng.randint(1, 4))
    return _case(path="spline", n_src=_size(rng, 2000, 120_000),
                 n_tgt=_size(rng, 2000, 150_000))


# ------------------------------------------------------------------ inputs
def _cloud(kind, n, gen, target):
    """n points [n, 3] float64 of a cloud; target: the targets' variant."""
    def u(*shape):
        return torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen)

    if kind == "cube":
        p = u(n, 3)
        return 0.05 + 0.9 * p if target else p
    if kind == "graded":
        return u(n, 3) ** 3
    v = torch.randn((n, 3), dtype=torch.float64, device="cuda", generator=gen)
    v = v / v.norm(dim=1, keepdim=True)
    return v * (1 + (2 * u(n, 1) - 1) * (2e-4 if target else 5e-4))


def _values(p, fields, gen):
    """Smooth fields at the points [fields, n], with a little noise."""
    x, y, z = p[:, 0], p[:, 1], p[:, 2]
    t = 2 * math.pi
    f = [torch.sin(t * x) * torch.cos(t * y) + z * z,
         torch.cos(t * x + 0.3) * torch.sin(2 * t * z) + 0.5 * y,
         x * y * z + torch.sin(3 * t * y),
         torch.cos(t * (x + y + z)) + x * x - y]
    v = torch.stack([f[i % 4] * (1 + i // 4) for i in range(fields)])
    return v + 1e-6 * torch.randn(v.shape, dtype=v.dtype, device=v.device, generator=gen)


def _options(case):
    o = dict(basis=case["basis"], rbf=case["rbf"], k=case["k"],
             precision=case["precision"], geometry=case["geometry"],
             solver=case["solver"], truncation=case["truncation"])
    return o


def _batch_sizes(case):
    """Uneven problems: source counts log-uniform up to the case's, targets
    half to twice as many, neighbour counts above the basis size. The sizes
    are those of the program, the same for every seed."""
    rng = np.random.default_rng(case["problems"])
    out = []
    for _ in range(case["problems"]):
        ns = int(round(math.exp(rng.uniform(math.log(64), math.log(case["n_src"])))))
        nt = int(round(ns * rng.uniform(0.5, 2.0)))
        basis = "linear" if rng.random() < 0.5 else "quadratic"
        k = int(rng.choice([10, 16, 32, 64] if basis == "linear" else [16, 32, 64]))
        out.append((ns, nt, basis, min(k, ns)))
    return out


def _batch_inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    sizes = _batch_sizes(case)
    ns, nt = [s[0] for s in sizes], [s[1] for s in sizes]
    n = len(sizes)

    def expand(v, counts):
        return torch.repeat_interleave(v, torch.tensor(counts, device="cuda"), dim=0)

    a = torch.eye(3, dtype=torch.float64, device="cuda") + 0.25 * torch.randn(
        (n, 3, 3), dtype=torch.float64, device="cuda", generator=gen).clamp(-1, 1)
    b = torch.randn((n, 3), dtype=torch.float64, device="cuda", generator=gen)

    def points(counts):
        p = torch.rand((sum(counts), 3), dtype=torch.float64, device="cuda", generator=gen)
        return ((expand(a, counts) * p[:, None, :]).sum(-1) + expand(b, counts)).contiguous()

    src, tgt = points(ns), points(nt)
    x = torch.sin(2 * src[:, 0]) * torch.cos(src[:, 1]) + src[:, 2] ** 2
    return sizes, ns, nt, src, tgt, x.contiguous()


def prepare(case, seed):
    if case["path"] == "batch":
        sizes, ns, nt, src, tgt, x = _batch_inputs(case, seed)
        op = dtk.MovingLeastSquaresBatch.from_concatenated(
            src, tgt, ns, nt, [s[2] for s in sizes], [s[3] for s in sizes],
            rbf=case["rbf"], precision=case["precision"], solver=case["solver"])
        y = torch.zeros(sum(nt), dtype=torch.float64, device="cuda")
        return {"case": case, "op": op, "x": x, "y": y, "src": src, "tgt": tgt}
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    src = _cloud(case["cloud"], case["n_src"], gen, False)
    tgt = _cloud(case["cloud"], case["n_tgt"], gen, True)
    st = {"case": case, "src": src, "tgt": tgt}
    if case["path"] == "knn":
        return st
    dtype = torch.float32 if case["precision"] == "fp32_bulk" else torch.float64
    st["x"] = _values(src, case["fields"], gen).to(dtype)
    st["y"] = torch.zeros((case["fields"], case["n_tgt"]), dtype=dtype, device="cuda")
    if case["path"] == "apply":
        st["op"] = dtk.MovingLeastSquaresOperator(src, tgt, **_options(case))
    if case["path"] == "adjoint":
        st["ybar"] = torch.randn((case["fields"], case["n_tgt"]), dtype=torch.float64,
                                 device="cuda", generator=gen)
    return st


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "transfer":
        op = dtk.MovingLeastSquaresOperator(state["src"], state["tgt"], **_options(case))
        return op.apply(state["x"], state["y"])
    if path == "apply":
        return state["op"].apply(state["x"], state["y"])
    if path == "adjoint":
        opts = _options(case)
        del opts["geometry"]
        x = state["x"].detach().requires_grad_(True)
        t = state["tgt"].detach().requires_grad_(True)
        y = mls_transfer(state["src"], t, x, **opts)
        y.backward(state["ybar"])
        return {"y": y.detach(), "x_grad": x.grad, "target_grad": t.grad}
    if path == "batch":
        state["op"].rebuild()
        return state["op"].apply_concatenated(state["x"], state["y"])
    if path == "knn":
        idx, dist = dtk.knn(state["src"], state["tgt"], case["k"],
                            geometry=case["geometry"], with_distances=True)
        return {"indices": idx, "distances": dist}
    make = dtk.NearestNeighborOperator if path == "nearest" else dtk.SplineOperator
    op = make(state["src"], state["tgt"], geometry=case["geometry"])
    return op.apply(state["x"], state["y"])


def work(case):
    """Points, values and results once each; the solves' operations."""
    m = _BASIS[case["basis"]]
    k = case["k"] or m
    ns, nt, f = case["n_src"], case["n_tgt"], case["fields"]
    vb = 4 if case["precision"] == "fp32_bulk" else 8
    path = case["path"]

    def setup(m, k):
        return 25 * k + k * m * (m + 1) + 2 * (m ** 3 // 3) + m * (m + 1) + k * (2 * m + 1)

    if path == "batch":
        sizes = _batch_sizes(case)
        return {"bytes": float(sum(32 * s + 32 * t for s, t, _, _ in sizes)),
                "flops": float(sum(t * (setup(_BASIS[b], k) + 10 * k)
                                   for _, t, b, k in sizes))}
    points = 24.0 * (ns + nt)
    if path == "knn":
        return {"bytes": points + 12.0 * nt * k, "flops": 8.0 * nt * k}
    values = float(vb * f * (ns + nt))
    if path == "apply":
        return {"bytes": values + nt * k * (4.0 + vb), "flops": 2.0 * nt * k * f}
    if path == "nearest":
        return {"bytes": points + values, "flops": 8.0 * nt}
    if path == "spline":
        return {"bytes": points + values, "flops": 8.0 * 4 * (ns + nt)}
    flops = nt * (setup(m, k) + 8.0 * k + 2.0 * k * f)
    if path == "adjoint":
        return {"bytes": points + 2 * values + 24.0 * nt, "flops": 2 * flops}
    return {"bytes": points + values, "flops": flops}


# ------------------------------------------- the same results in 64 bits
def _brute(src, tgt, k):
    idx = torch.empty((len(tgt), k), dtype=torch.int64, device=src.device)
    step = max(1, int(1e8) // len(src))
    for i in range(0, len(tgt), step):
        t = tgt[i:i + step]
        d = (t[:, None, 0] - src[None, :, 0]).square_()
        for a in (1, 2):
            d += (t[:, None, a] - src[None, :, a]).square_()
        idx[i:i + step] = d.topk(k, dim=1, largest=False).indices
    return idx


def _neighbours(src, tgt, k, uniform):
    """The k nearest sources of every target (as a set)."""
    n = len(src)
    if n < 20_000 or not uniform:
        return _brute(src, tgt, k)
    lo = src.min(0).values
    ext = src.max(0).values - lo
    h = float((ext.prod() * (0.5 * k + 3) / n) ** (1 / 3))
    dims = torch.floor(ext / h).long() + 1

    def cell(p):
        c = torch.floor((p - lo) / h).long()
        return torch.minimum(torch.clamp(c, min=0), dims - 1)

    def flat(c):
        return (c[:, 0] * dims[1] + c[:, 1]) * dims[2] + c[:, 2]

    ids = flat(cell(src))
    order = torch.argsort(ids)
    count = torch.bincount(ids, minlength=int(dims.prod()))
    first = torch.cumsum(count, 0) - count
    width = int(count.max())
    off = torch.stack(torch.meshgrid(*[torch.arange(-1, 2, device=src.device)] * 3,
                                     indexing="ij"), -1).reshape(-1, 3)
    lane = torch.arange(width, device=src.device)
    idx = torch.empty((len(tgt), k), dtype=torch.int64, device=src.device)
    far = torch.empty(len(tgt), dtype=torch.float64, device=src.device)
    step = max(1, int(3e7) // (27 * width))
    for i in range(0, len(tgt), step):
        t = tgt[i:i + step]
        c = cell(t)[:, None, :] + off[None]
        ok = ((c >= 0) & (c < dims)).all(-1)
        q = flat(torch.where(ok[..., None], c, 0).reshape(-1, 3)).reshape(ok.shape)
        valid = (ok[..., None] & (lane < count[q][..., None])).reshape(len(t), -1)
        s = (first[q][..., None] + lane).clamp(max=n - 1).reshape(len(t), -1)
        s = order[s]
        d = (src[s] - t[:, None, :]).square().sum(-1)
        d = torch.where(valid, d, math.inf)
        v, j = d.topk(k, dim=1, largest=False)
        idx[i:i + step] = s.gather(1, j)
        far[i:i + step] = v[:, -1]
    miss = torch.nonzero(far > h * h).flatten()
    if len(miss):
        idx[miss] = _brute(src, tgt[miss], k)
    return idx


def _phi(rbf, r):
    q = 1 - r
    if rbf == "wendland0":
        return q ** 2
    if rbf == "wendland2":
        return q ** 4 * (4 * r + 1)
    return q ** 6 * (35 * r * r + 18 * r + 3)


def _solve(a, b):
    """x of a x = b for batches of small positive definite matrices."""
    m = b.shape[1]
    rows = []
    for _ in range(m):
        rows.append((a[:, 0], b[:, 0]))
        f = a[:, 1:, 0] / a[:, 0, :1]
        b = b[:, 1:] - f * b[:, :1]
        a = a[:, 1:, 1:] - f[..., None] * a[:, :1, 1:]
    x = []
    for r, v in reversed(rows):
        for j, xj in enumerate(x):
            v = v - r[:, j + 1] * xj
        x.insert(0, v / r[:, 0])
    return torch.stack(x, 1)


def _coefficients(src, tgt, idx, m, rbf, geometry):
    """The rows of the operator; the monomials in units of the radius, which
    changes no coefficient."""
    rel = src[idx] - tgt[:, None, :]
    if geometry == "float":
        rel = rel.float().double()
    d = rel.square().sum(-1).sqrt()
    radius = 1.1 * d.max(dim=1, keepdim=True).values
    w = _phi(rbf, d / radius)
    x, y, z = (rel / radius[..., None]).unbind(-1)
    p = [torch.ones_like(x)]
    if m >= 4:
        p += [x, y, z]
    if m >= 10:
        p += [x * x, x * y, x * z, y * y, y * z, z * z]
    p = torch.stack(p, -1)
    a = (p[..., None] * (w[..., None] * p)[:, :, None, :]).sum(1)
    e = torch.zeros((len(tgt), m), dtype=p.dtype, device=p.device)
    e[:, 0] = 1
    a0 = _solve(a, e)
    # one step of refinement
    a0 = a0 + _solve(a, e - (a * a0[:, None, :]).sum(-1))
    return (p * a0[:, None, :]).sum(-1) * w


def _rounded(p, geometry):
    return p.float().double() if geometry == "float" else p


def _spline_exact(src, tgt, x):
    """y = (Q + N) z with [[M, P], [P^T, 0]] z = [x; 0], by GMRES with
    reorthogonalisation, restarted to the rounding of 64 bits."""
    n = len(src)
    fs, ft = _rounded(src, "float"), _rounded(tgt, "float")

    def rows(pts, fpts):
        idx = _neighbours(fs, fpts, 4, True)
        d = (src[idx] - pts[:, None, :]).float().double().square().sum(-1).sqrt()
        return idx, _phi("wendland0", d / (1.1 * d.max(dim=1, keepdim=True).values))

    (mi, mv), (ni, nv) = rows(src, fs), rows(tgt, ft)
    one = torch.ones((n, 1), dtype=torch.float64, device=src.device)
    p = torch.cat([one, fs], 1)
    q = torch.cat([torch.ones((len(tgt), 1), dtype=torch.float64, device=src.device), ft], 1)

    def system(z):
        s, c = z[:n], z[n:]
        return torch.cat([(mv * s[mi]).sum(1) + p @ c, p.T @ s])

    b = torch.cat([x, torch.zeros(4, dtype=torch.float64, device=src.device)])
    z = torch.zeros_like(b)
    for _ in range(4):
        r = b - system(z)
        beta = r.norm()
        if float(beta / b.norm()) < 1e-14:
            break
        v = torch.empty((161, n + 4), dtype=torch.float64, device=src.device)
        hess = torch.zeros((161, 160), dtype=torch.float64, device=src.device)
        v[0] = r / beta
        for j in range(160):
            w = system(v[j])
            for _ in range(2):
                c = v[:j + 1] @ w
                w = w - c @ v[:j + 1]
                hess[:j + 1, j] += c
            hess[j + 1, j] = w.norm()
            v[j + 1] = w / hess[j + 1, j]
        rhs = np.zeros(161)
        rhs[0] = float(beta)
        yk = np.linalg.lstsq(hess.cpu().numpy(), rhs, rcond=None)[0]
        z = z + torch.from_numpy(yk).to(v) @ v[:160]
    return (nv * z[:n][ni]).sum(1) + q @ z[n:]


def exact(case, seed):
    path, geometry = case["path"], case["geometry"]
    m = _BASIS[case["basis"]]
    if path == "batch":
        sizes, ns, nt, src, tgt, x = _batch_inputs(case, seed)
        out, s0, t0 = [], 0, 0
        for a, b, basis, k in sizes:
            s, t, v = src[s0:s0 + a], tgt[t0:t0 + b], x[s0:s0 + a]
            idx = _brute(_rounded(s, "float"), _rounded(t, "float"), k)
            c = _coefficients(s, t, idx, _BASIS[basis], case["rbf"], "float")
            out.append((c * v[idx]).sum(1))
            s0, t0 = s0 + a, t0 + b
        return torch.cat(out)
    if case["cloud"] == "shell":
        return None  # truncated at a threshold: decided by rounding
    if case["k"] <= m and path == "transfer":
        return None  # square systems: near the truncation threshold
    # the inputs of prepare, drawn in its order
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    src = _cloud(case["cloud"], case["n_src"], gen, False)
    tgt = _cloud(case["cloud"], case["n_tgt"], gen, True)
    k = min(case["k"] or (1 if path == "nearest" else m), case["n_src"])
    uniform = case["cloud"] == "cube"
    fs, ft = _rounded(src, geometry), _rounded(tgt, geometry)
    if path == "knn":
        idx = _neighbours(fs, ft, k, uniform)
        d = (fs[idx] - ft[:, None, :]).square().sum(-1).sqrt()
        return {"indices": None, "distances": d.sort(dim=1).values}
    x = _values(src, case["fields"], gen)
    if case["precision"] == "fp32_bulk":
        x = x.float().double()
    if path == "spline":
        return torch.stack([_spline_exact(src, tgt, f) for f in x])
    idx = _neighbours(fs, ft, k, uniform)
    if path == "nearest":
        return x[:, idx[:, 0]]
    if path == "adjoint":
        ybar = torch.randn((case["fields"], case["n_tgt"]), dtype=torch.float64,
                           device="cuda", generator=gen)
        xv, tv = x.requires_grad_(True), tgt.requires_grad_(True)
        c = _coefficients(src, tv, idx, m, case["rbf"], geometry)
        y = torch.stack([(c * f[idx]).sum(1) for f in xv])
        gx, gt = torch.autograd.grad(y, (xv, tv), ybar)
        return {"y": y.detach(), "x_grad": gx, "target_grad": gt}
    step = 25_000
    y = []
    for i in range(0, len(tgt), step):
        j = idx[i:i + step]
        c = _coefficients(src, tgt[i:i + step], j, m, case["rbf"], geometry)
        y.append(torch.stack([(c * f[j]).sum(1) for f in x]))
    return torch.cat(y, 1)
