"""The work a user of this package has it do, as measurable cases.

Every case goes through the public Python entry points (sgtsne_amd): the front
end (kNN and perplexity equalisation), a whole embedding call, iterations of
one job on the device, the evaluation of the gradient's terms and the cost, and
a batch of jobs advanced together.  Sizes and data follow this repository's
own workloads: 50-D Gaussian mixtures, 40 clusters of power-law sizes at
1.3 M points, sparse 784-D clusters, jobs and requests of 500 to 200,000
points in two and three dimensions.

Kinds (the fields of a case):
  steps   one resident job: set_Y, `iters` iterations, get_Y (n, d, phase, format)
  terms   gradient terms and KL divergence of an embedding (n, d)
  run     the drop-in call from P to Y (n, d, iters)
  front   points to P: exact kNN and perplexity equalisation (n, dim, data)
  batch   `jobs` jobs admitted from their points or graphs (source), `iters` iterations, Y read back
`phase` start: the reference's N(0, 1e-4^2) start (early exaggeration, smallest
grid); late: an embedding spread over its clusters (the grids of a run's second
half).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpu-sg-sne_amd"))
import sgtsne_amd as S  # noqa: E402

K, U = 90, 30.0  # neighbours and perplexity of every workload


def listed():
    return [
        # the smallest request of the serving stream: launches and the host round trip
        dict(name="steps_2k", kind="steps", n=2011, d=2, phase="start", format=4, iters=10),
        # the 10-cluster mixture (N = 10,000, 50-D), early exaggeration
        dict(name="steps_10k", kind="steps", n=10000, d=2, phase="start", format=4, iters=20),
        # N = 60,000 in the hybrid ELL + COO format of the sparse workload
        dict(name="steps_60k_hybrid", kind="steps", n=60000, d=2, phase="start", format=3, iters=10),
        # the second half of a 60,000-point run: a large 2-D grid
        dict(name="steps_60k_late", kind="steps", n=60000, d=2, phase="late", format=4, iters=15),
        # the largest request of the serving stream, in 3-D, late
        dict(name="steps_200k_3d", kind="steps", n=200003, d=3, phase="late", format=4, iters=10),
        # the headline workload: 1.3 M points, early exaggeration
        dict(name="steps_1300k", kind="steps", n=1300000, d=2, phase="start", format=4, iters=20),
        # watching a run: gradient terms and cost of the current embedding
        dict(name="terms_50k", kind="terms", n=50021, d=2),
        # a small whole call: context, upload, iterations, result
        dict(name="run_1k", kind="run", n=1203, d=2, iters=10),
        # the front end of a mid-sized 50-D job
        dict(name="front_20k_50d", kind="front", n=20011, dim=50, data="mixture"),
        # the front end on sparse 784-D data (more dimensions than the filtered search takes)
        dict(name="front_6k_784d", kind="front", n=6007, dim=784, data="sparse"),
        # many small 2-D jobs as one batch, admitted from their points
        dict(name="batch_2d", kind="batch", jobs=16, lo=500, hi=8000, d=2, source="points", phase="start", iters=8),
        # a few 3-D jobs as one batch, admitted from their graphs with the embeddings of an earlier run
        dict(name="batch_3d", kind="batch", jobs=6, lo=2000, hi=20000, d=3, source="graph", phase="late", iters=10),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "terms", "run", "front", "batch"])
    d = rng.choice([2, 2, 3])
    if kind == "steps":
        n = _log_uniform(rng, 700, 300000)
        return dict(kind=kind, n=n, d=d, phase=rng.choice(["start", "late"]), format=3 if rng.random() < 0.15 else 4,
                    iters=rng.randint(6, 10) if n < 5000 else rng.randint(8, 16))
    if kind == "terms":
        return dict(kind=kind, n=_log_uniform(rng, 700, 200000), d=d)
    if kind == "run":
        return dict(kind=kind, n=_log_uniform(rng, 500, 20000), d=d, iters=rng.randint(6, 10))
    if kind == "front":
        if rng.random() < 0.25:
            return dict(kind=kind, n=_log_uniform(rng, 700, 8000), dim=784, data="sparse")
        return dict(kind=kind, n=_log_uniform(rng, 500, 60000), dim=rng.choice([10, 30, 50, 50, 64, 100, 128]),
                    data="mixture")
    late = rng.random() < 0.5
    return dict(kind=kind, jobs=rng.randint(4, 16), lo=rng.choice([500, 1000]), hi=_log_uniform(rng, 3000, 12000), d=d,
                source="graph" if late else "points", phase="late" if late else "start",
                iters=rng.randint(6, 8))


# ---- inputs -------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _labels(n, weights, g):
    """Cluster of every point: about weights[c] of the points in cluster c, shuffled."""
    return torch.multinomial(weights, n, replacement=True, generator=g)


def _mixture(n, dim, seed, clusters=None):
    """Gaussian clusters with a decaying spectrum (as the power-law workload's):
    X [n][dim], the labels, each cluster's share and the coordinates within the cluster."""
    g = _gen(seed)
    if clusters is None:
        clusters = 40 if n > 100000 else 10
    w = torch.arange(1, clusters + 1, device="cuda", dtype=torch.float64) ** -(1.5 if n > 100000 else 0.3)
    w /= w.sum()
    lab = _labels(n, w, g)
    sd = torch.arange(1, dim + 1, device="cuda", dtype=torch.float32) ** -0.5
    z = torch.randn(n, dim, device="cuda", generator=g)
    centre = 4.0 * torch.randn(clusters, dim, device="cuda", generator=g)
    X = torch.empty(n, dim, device="cuda")
    for c in range(clusters):
        q, _ = torch.linalg.qr(torch.randn(dim, dim, device="cuda", generator=g))
        at = torch.nonzero(lab == c).flatten()
        X[at] = (z[at] * sd) @ q.T + centre[c]
    return X.cpu().numpy(), lab, w, z


def _sparse(n, dim, seed, clusters=10, density=0.19):
    """Clusters that each use their own 19 % of the dimensions, values U[0, 255]."""
    g = _gen(seed)
    lab = torch.randint(clusters, (n,), device="cuda", generator=g)
    support = torch.rand(clusters, dim, device="cuda", generator=g) < density
    X = 255.0 * torch.rand(n, dim, device="cuda", generator=g) * support[lab]
    return X.cpu().numpy()


def _radius(n, d):
    """Half the width of a finished embedding of n points."""
    return 50.0 * (n / 1e4) ** 0.35 if d == 2 else 10.0 * (n / 1e4) ** 0.3


def _start(n, d, seed):
    return (1e-4 * np.random.default_rng(seed).standard_normal((n, d))).astype(np.float32)


def _spread(n, d, lab, w, z, seed):
    """An embedding late in a run: clusters side by side, each spread along its
    points' leading coordinates."""
    g = _gen(seed + 1)
    R = _radius(n, d)
    c = torch.randn(w.numel(), d, device="cuda", generator=g)
    c = c / c.norm(dim=1, keepdim=True) * (0.8 * R * torch.rand(w.numel(), 1, device="cuda", generator=g) ** (1.0 / d))
    r = (0.3 * R * (w / w.max()) ** (1.0 / d)).float()
    Y = c[lab] + r[lab][:, None] * z[:, :d].clamp(-2.5, 2.5) / 2.5 + 0.01 * R * torch.randn(n, d, device="cuda",
                                                                                         generator=g)
    return Y.cpu().numpy()


def _sizes(case):
    """The sizes of a batch's jobs, log-uniform over its range."""
    rng = np.random.default_rng(case["jobs"] * 100003 + case["hi"])
    j = case["jobs"]
    at = (np.arange(j) + rng.uniform(0, 1, j)) / j
    return [int(v) for v in np.exp(np.log(case["lo"]) + at * (np.log(case["hi"]) - np.log(case["lo"])))]


def _points(n, d, phase, seed, clusters=None):
    """Points of a job and the embedding it starts from."""
    X, lab, w, z = _mixture(n, 50, seed, clusters)
    return X, _spread(n, d, lab, w, z, seed) if phase == "late" else _start(n, d, seed)


def _to_graph(X):
    I, D = S.knn_exact(X, K)
    return S.perplexityEqualization(I, D, X.shape[0], K, U)


def _graph(case, seed):
    X, Y0 = _points(case["n"], case["d"], case.get("phase", "late" if case["kind"] == "terms" else "start"), seed)
    return _to_graph(X), Y0


def _batch_inputs(case, seed):
    jobs = [_points(n, case["d"], case["phase"], 1000 * seed + i, 5 + i % 8) for i, n in enumerate(_sizes(case))]
    return [(_to_graph(X), Y0) for X, Y0 in jobs] if case["source"] == "graph" else jobs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "front":
        X = _sparse(case["n"], case["dim"], seed) if case["data"] == "sparse" else _mixture(case["n"], case["dim"], seed)[0]
        return dict(case=case, X=X)
    if kind == "batch":
        jobs = _batch_inputs(case, seed)
        points = sum(Y0.shape[0] for _, Y0 in jobs)
        params = S.tsneparams(d=case["d"], maxIter=case["iters"], layout=S.LAYOUT_AOS)
        return dict(case=case, jobs=jobs, batch=S.Batch(params, case["jobs"], points, 2 * K * points))
    P, Y0 = _graph(case, seed)
    if kind == "run":
        return dict(case=case, P=P, Y0=Y0, params=S.tsneparams(d=case["d"], maxIter=case["iters"], layout=S.LAYOUT_AOS))
    ctx = S.Context(S.tsneparams(d=case["d"], format=case.get("format", S.FORMAT_CSR_SEG)))
    ctx.upload_P(P)
    if kind == "terms":
        ctx.set_Y(Y0)
    return dict(case=case, ctx=ctx, Y0=Y0)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "steps":
        ctx = state["ctx"]
        ctx.set_Y(state["Y0"])
        ctx.step(case["iters"])
        return ctx.get_Y()
    if kind == "terms":
        Fa, Fr, Z, _ = state["ctx"].terms()
        return dict(Fattr=Fa, Frep=Fr, Z=Z, kl=state["ctx"].kl())
    if kind == "run":
        return S.sgtsne(state["P"], state["params"], y_in=state["Y0"])
    if kind == "front":
        I, D = S.knn_exact(state["X"], K)
        P = S.perplexityEqualization(I, D, case["n"], K, U)
        return dict(I=I, D=D, col=P.col, val=P.val)
    b = state["batch"]
    if case["source"] == "points":
        ids = [b.add_points(X, k=K, u=U, y_in=Y0, max_iter=case["iters"]) for X, Y0 in state["jobs"]]
    else:
        ids = [b.add(P, y_in=Y0, max_iter=case["iters"]) for P, Y0 in state["jobs"]]
    b.step(case["iters"] + 1)
    out = [b.get_Y(j) for j in ids]
    for j in ids:
        b.remove(j)
    return out


def _side(n, d, phase):
    return 16 if phase == "start" else max(16, int(2 * _radius(n, d) / (0.7 if d == 2 else 1.2)) + 2)


def work(case):
    """What a pass cannot do without: P (its symmetric part has about 1.63 times
    the nonzeros of the kNN graph) and the point state once per iteration, the
    grid and the transforms; for the front end X in, I, D, col and val out, and
    one multiply-add per coordinate of every pair."""
    kind, d = case["kind"], case.get("d", 2)

    def iteration(n, side):
        nnz, cells = 1.63 * K * n, side ** d
        return (8.0 * nnz + 4 * (n + 1) + 52.0 * d * n + 16.0 * (d + 1) * cells,
                nnz * (5 * d + 2) + n * 2.0 * (2 * d + 3) * 4 ** d + 5.0 * (2 * d + 3) * (2 ** d * cells) * math.log2(2 ** d * cells + 1))

    def front(n, dim):
        return 4.0 * n * dim + n * (K + 1) * 12.0 + n * K * 8.0, 2.0 * n * n * dim

    if kind == "front":
        b, f = front(case["n"], case["dim"])
    elif kind == "terms":
        b, f = iteration(case["n"], _side(case["n"], d, "late"))
        b, f = b + 8 * 1.63 * K * case["n"], 2 * f
    elif kind == "batch":
        b = f = 0.0
        for n in _sizes(case):
            ib, jf = iteration(n, _side(n, d, case["phase"]))
            pts = case["source"] == "points"
            b += (4.0 * n * 50 if pts else 8.0 * K * n) + 8.0 * n * d + case["iters"] * ib
            f += (2.0 * n * n * 50 if pts else 0.0) + case["iters"] * jf
    else:
        b, f = iteration(case["n"], _side(case["n"], d, case.get("phase", "start")))
        b, f = case["iters"] * b + 8.0 * d * case["n"], case["iters"] * f
        if kind == "run":
            b += 8.0 * K * case["n"]
    return dict(bytes=b, flops=f)


# ---- the same results in 64 bits ------------------------------------------------

_SIZES = [8, 9, 10, 11, 12, 13, 14, 15, 16, 20, 25, 26, 28, 32, 33, 35, 36, 39, 40, 42, 44, 45, 48, 49, 50, 52, 54, 55, 56,
          60, 63, 64, 65, 66, 70, 72, 75, 77, 78, 80, 84, 88, 90, 91, 96, 98, 99, 100, 104, 105, 108, 110, 112, 117, 120,
          125, 126, 130, 132, 135, 140, 144, 147, 150, 154, 156, 160, 165, 168, 175, 176, 180, 182, 189, 192, 195, 196,
          198, 200, 208, 210, 216, 220, 224, 225, 231, 234, 240, 245, 250, 252, 260, 264, 270, 273, 275, 280, 288, 294,
          297, 300, 308, 312, 315, 320, 325, 330, 336, 343, 350, 351, 352, 360, 364, 375, 378, 385, 390, 392, 396, 400,
          416, 420, 432, 440, 441, 448, 450, 455, 462, 468, 480, 490, 495, 500, 504, 512]  # getBestGridSize


def _knn64(X):
    X = torch.from_numpy(X).cuda().double()
    n, dim = X.shape
    D = torch.empty(n, K + 1, dtype=torch.float64, device="cuda")
    I = torch.empty(n, K + 1, dtype=torch.int64, device="cuda")
    step = max(1, int(6e7 / (n * dim)))
    for i in range(0, n, step):
        d2 = (X[i:i + step, None, :] - X[None]).square().sum(2)
        D[i:i + step], I[i:i + step] = torch.topk(d2, K + 1, largest=False, sorted=True)
    return I, D


def _perplexity64(D):
    """Bisection of the precision to |H - log u| < 1e-5, from 1, as the method defines it."""
    D = D[:, 1:]
    n = D.shape[0]
    beta = torch.ones(n, dtype=torch.float64, device="cuda")
    lo, hi = torch.full_like(beta, -math.inf), torch.full_like(beta, math.inf)
    done = torch.zeros(n, dtype=torch.bool, device="cuda")
    P = torch.empty_like(D)
    for _ in range(200):
        e = torch.exp(-beta[:, None] * D)
        s = e.sum(1)
        diff = beta * (D * e).sum(1) / s + s.log() - math.log(U)
        P = torch.where(done[:, None], P, e / s[:, None])
        done = done | (diff.abs() < 1e-5)
        if bool(done.all()):
            break
        up, down = ~done & (diff > 0), ~done & (diff <= 0)
        lo, hi = torch.where(up, beta, lo), torch.where(down, beta, hi)
        beta = torch.where(up, torch.where(hi.isinf(), 2 * beta, (beta + hi) / 2), beta)
        beta = torch.where(down, torch.where(lo.isinf(), beta / 2, (beta + lo) / 2), beta)
    return P


def _symmetric64(n, col, val):
    """(P + P^T) / sum: rows ascending, columns and values."""
    row = torch.arange(n, device="cuda").repeat_interleave(K)
    key, at = torch.sort(torch.cat([row * n + col, col * n + row]))
    v = torch.cat([val, val])[at]
    new = torch.ones_like(key, dtype=torch.bool)
    new[1:] = key[1:] != key[:-1]
    out = torch.zeros(int(new.sum()), dtype=torch.float64, device="cuda").index_add_(0, torch.cumsum(new, 0) - 1, v)
    key = key[new]
    return key // n, key % n, out / out.sum()


def _attractive64(P, Y, kl_z=None):
    row, col, val = P
    n, d = Y.shape
    F, kl = torch.zeros_like(Y), 0.0
    tiny = float(np.finfo(np.float32).tiny)
    for i in range(0, row.numel(), 1 << 25):
        r, c, p = row[i:i + (1 << 25)], col[i:i + (1 << 25)], val[i:i + (1 << 25)]
        df = Y[r] - Y[c]
        q = 1.0 / (1.0 + df.square().sum(1))
        F.index_add_(0, r, (p * q)[:, None] * df)
        if kl_z is not None:
            kl += float((p * torch.log((p + tiny) / (q / kl_z + tiny))).sum())
    return F, kl


def _repulsive64(Y):
    """Interpolated repulsion (not divided by Z) and Z."""
    n, d = Y.shape
    lo, hi = Y.min(0).values, Y.max(0).values
    maxy = float((hi - lo).max())
    grid = max(math.ceil(maxy / (0.7 if d == 2 else 1.2)), 14)
    ng = next((s for s in _SIZES if grid + 2 <= s), 512)
    grid = ng - 2
    t = ((Y - lo) * ((grid - 1) / maxy)).clamp(0.0, math.nextafter(grid - 1.0, 0.0))
    f = t.floor().long()
    dl = t - f
    g1 = lambda x: ((0.5 * x - 1.0) * x - 0.5) * x + 1.0  # noqa: E731
    g2 = lambda x: ((-x / 6.0 + 1.0) * x - 11.0 / 6.0) * x + 1.0  # noqa: E731
    w = torch.stack([g2(1.0 + dl), g1(dl), g1(1.0 - dl), g2(2.0 - dl)], 2)  # [n][d][4]
    yc = Y - 0.5 * (lo + hi)
    q = torch.cat([torch.ones(n, 1, dtype=torch.float64, device="cuda"), yc], 1)
    V = torch.zeros(d + 1, *([ng] * d), dtype=torch.float64, device="cuda")
    step = max(1, int(1e8 / ng ** (d - 1)))
    for i in range(0, n, step):  # dense weights along each axis: V_c = sum_i q_ic w_i(x) w_i(y) ...
        m = min(step, n - i)
        W = [torch.zeros(m, ng, dtype=torch.float64, device="cuda").scatter_(
            1, f[i:i + m, a:a + 1] + torch.arange(4, device="cuda"), w[i:i + m, a]) for a in range(d)]
        rest = W[1] if d == 2 else (W[1][:, :, None] * W[2][:, None, :]).reshape(m, ng * ng)
        for c in range(d + 1):
            V[c] += ((W[0] * q[i:i + m, c:c + 1]).T @ rest).reshape(V[c].shape)
    h = maxy / (grid - 1)
    L = 2 * ng
    r = torch.arange(L, device="cuda", dtype=torch.float64)
    r = torch.minimum(r, L - r) * h
    r2 = sum(x.square() for x in torch.meshgrid(*([r] * d), indexing="ij"))
    ax = list(range(-d, 0))
    Vh = torch.fft.rfftn(V, s=[L] * d, dim=ax)
    cut = (slice(None),) + (slice(0, ng),) * d
    Phi = torch.fft.irfftn(Vh * torch.fft.rfftn((1 + r2) ** -2), s=[L] * d, dim=ax)[cut]
    psi = torch.fft.irfftn(Vh[:1] * torch.fft.rfftn(1 / (1 + r2)), s=[L] * d, dim=ax)[cut]
    flat = torch.cat([Phi, psi]).reshape(d + 2, -1).T.contiguous()
    at = torch.zeros(n, d + 2, dtype=torch.float64, device="cuda")
    for node in range(4 ** d):
        idx, ww = torch.zeros_like(f[:, 0]), torch.ones_like(dl[:, 0])
        for a in range(d):
            o = node // 4 ** a % 4
            idx, ww = idx * ng + f[:, a] + o, ww * w[:, a, o]
        at += ww[:, None] * flat[idx]
    return yc * at[:, :1] - at[:, 1:d + 1], float(at[:, d + 1].sum()) - n


def _iterate64(P, Y0, iters):
    Y = torch.from_numpy(Y0).cuda().double()
    Y = Y - Y.mean(0)
    u, gain = torch.zeros_like(Y), torch.ones_like(Y)
    for _ in range(iters):
        Fa, _ = _attractive64(P, Y)
        Fr, Z = _repulsive64(Y)
        dy = 12.0 * Fa - Fr / Z
        gain = torch.where(dy.sign() != u.sign(), gain + 0.2, gain * 0.8).clamp(min=0.01)
        u = 0.5 * u - 200.0 * gain * dy
        Y = Y + u
        Y = Y - Y.mean(0)
    return Y.cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "front":
        X = prepare(case, seed)["X"]
        D = _knn64(X)[1]
        return dict(I=None, D=D.cpu().numpy(), col=None, val=_perplexity64(D).reshape(-1).cpu().numpy())
    if kind == "batch":
        out = []
        for src, Y0 in _batch_inputs(case, seed):
            if case["source"] == "points":
                I, D = _knn64(src)
                col, val = I[:, 1:].reshape(-1), _perplexity64(D).reshape(-1)
            else:
                col, val = torch.from_numpy(src.col).cuda().long(), torch.from_numpy(src.val).cuda().double()
            out.append(_iterate64(_symmetric64(Y0.shape[0], col, val), Y0, case["iters"]))
        return out
    P, Y0 = _graph(case, seed)  # P is an input of these
    P = _symmetric64(case["n"], torch.from_numpy(P.col).cuda().long(), torch.from_numpy(P.val).cuda().double())
    if kind == "terms":
        Y = torch.from_numpy(Y0).cuda().double()
        Y = Y - Y.mean(0)
        Fr, Z = _repulsive64(Y)
        Fa, kl = _attractive64(P, Y, Z)
        return dict(Fattr=Fa.cpu().numpy(), Frep=(Fr / Z).cpu().numpy(), Z=Z, kl=kl)
    return _iterate64(P, Y0, case["iters"])
