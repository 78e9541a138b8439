"""The work a user of tbslas_amd has it do, as cases that can be timed and checked.

Kinds (``case["kind"]``), each one pass through public entry points:

eval      ``Tree.eval`` at a user's points (probes, samples for a picture,
          another code's nodes): any order, from a handful to millions.
traj      ``traj_rk2``: particles carried through a velocity tree.
step      a short run: the initial condition set, then ``semilag_insitu``
          steps, then the coefficients read.  One tracer, or many that share
          the trajectories (``dof``).
vjp       one differentiable step through ``torch.autograd``: forward,
          cotangents of concentration and velocity.
grid      the tricubic variant: one ``grid_semilag_insitu`` step and the
          new samples read at their points.
batch     many small problems in one ``Batch``: steps between snapshots,
          then every problem's state.
refit     ``Tree.set_grid_values`` and back (``Tree.grid_values``): nodal
          values of another solver taken into the tree and returned.

The FP64 arithmetic is the entry points' default.  The FP32 modes' results
are kept in float32, the precision their coefficients are read with.
Inputs are made with torch from the seed alone; leaf lists depend on the
case alone, so a case's outputs have one shape.
"""
import math

import numpy as np
import torch

CENTRE = (0.7, 0.5, 0.5)  # where refined trees are fine and clouds gather


# --- leaf lists ---------------------------------------------------------

def _compact3(c):
    r = np.zeros_like(c)
    for b in range(21):
        r |= ((c >> (3 * b)) & 1) << b
    return r


def leaf_list(depth, radius):
    """The uniform tree of ``depth``; with ``radius`` > 0, its leaves whose
    centres are nearer than that to CENTRE split once (Morton order)."""
    c = np.arange(8 ** depth, dtype=np.int64)
    a = np.stack([_compact3(c), _compact3(c >> 1), _compact3(c >> 2)], 1)
    d = np.full(len(c), depth, dtype=np.int64)
    if radius > 0:
        mid = (a + 0.5) / 2.0 ** depth
        split = ((mid - np.array(CENTRE)) ** 2).sum(1) < radius ** 2
        reps = np.where(split, 8, 1)
        child = np.arange(reps.sum()) - np.repeat(np.cumsum(reps) - reps, reps)
        a, d, s = np.repeat(a, reps, 0), np.repeat(d, reps), np.repeat(split, reps)
        bits = np.stack([child & 1, (child >> 1) & 1, child >> 2], 1)
        a = np.where(s[:, None], 2 * a + bits, a)
        d = d + s
    return a.astype(np.uint32), d.astype(np.uint8)


def num_leaves(case):
    return len(leaf_list(case["depth"], case.get("radius", 0.0))[1])


def ncoef(q):
    return (q + 1) * (q + 2) * (q + 3) // 6


def _triangle(q):
    """(i, j, k) of the packed coefficients, i(z) -> j(y) -> k(x)."""
    t = [(i, j, k) for i in range(q + 1) for j in range(q + 1 - i) for k in range(q + 1 - i - j)]
    return torch.tensor(t, dtype=torch.int64, device="cuda").T


# --- fields, made from the seed -----------------------------------------

def _rng(seed, what):
    return np.random.RandomState((1000003 * int(seed) + what) % (2 ** 32))


def velocity_field(seed, flow, k=0):
    """A smooth periodic flow with random phases ("waves"), or a rigid
    rotation about a random axis through the middle ("spin"); k: snapshot."""
    r = _rng(seed, 1)
    a, b, c, d = (float(x) for x in r.uniform(0.3, 5.9, 4))
    z, phi, amp = r.uniform(-0.9, 0.9), r.uniform(0, 2 * math.pi), r.uniform(0.8, 1.2) * (1 + 0.05 * k)
    if flow == "spin":
        s = math.sqrt(1 - z * z)
        w = [2 * math.pi * v for v in (s * math.cos(phi), s * math.sin(phi), z)]

        def spin(p):
            x, y, u = (p[:, i] - 0.5 for i in range(3))
            return torch.stack([w[1] * u - w[2] * y, w[2] * x - w[0] * u, w[0] * y - w[1] * x], 1)
        return spin
    t = 2 * math.pi

    def waves(p):
        x, y, u = t * p[:, 0] + a, t * p[:, 1] + b, t * p[:, 2] + c
        return amp * torch.stack([x.sin() * y.cos() * u.cos(), -x.cos() * y.sin() * u.cos(),
                                  0.25 * (t * p[:, 0] + d).sin() * y.cos()], 1)
    return waves


def blob_field(seed, dof, sigma, what=2):
    """Gaussian blobs, the first near CENTRE, the others about it."""
    r = _rng(seed, what)
    mid = np.array(CENTRE) + r.uniform(-0.01, 0.01, (dof, 3)) + (np.arange(dof) > 0)[:, None] * r.uniform(-0.2, 0.2, (dof, 3))
    sig = sigma * r.uniform(0.9, 1.1, dof)

    def blobs(p):
        return torch.stack([torch.exp(-((p - torch.tensor(m, device=p.device)) ** 2).sum(1) / (2 * s * s))
                            for m, s in zip(mid, sig)], 1)
    return blobs


def fit(field, anchor, depth, q, dof):
    """Chebyshev coefficients [L][dof][Nc] of field: values at first-kind
    nodes, one-axis transforms, the triangle kept."""
    d = q + 1
    th = (torch.arange(d, dtype=torch.float64, device="cuda") + 0.5) * math.pi / d
    xi = -torch.cos(th)
    F = _cheb(xi, d).T * (2.0 / d)
    F[0] *= 0.5
    i, j, k = _triangle(q)
    s = torch.tensor(0.5 ** depth.astype(np.float64), device="cuda")
    lo = torch.tensor(anchor.astype(np.float64), device="cuda") * s[:, None]
    u = 0.5 * xi + 0.5
    node = torch.stack([g.reshape(-1) for g in torch.meshgrid(u, u, u, indexing="ij")][::-1], 1)
    out = torch.empty((len(depth), dof, ncoef(q)), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 24) // (d ** 3 * dof))
    for a in range(0, len(depth), step):
        p = (lo[a:a + step, None] + node * s[a:a + step, None, None]).reshape(-1, 3)
        v = field(p).reshape(-1, d, d, d, dof)
        for _ in range(3):  # z, y, x in turn: each transformed axis goes last
            v = torch.tensordot(v, F, dims=([1], [1]))
        out[a:a + step] = v[:, :, i, j, k]
    return out


# --- 64-bit arithmetic without the framework ----------------------------

def _cheb(x, d):
    """T_0..T_{d-1} at x; zero outside [-1, 1]."""
    inside = (x.abs() <= 1).to(x.dtype)
    xx = x * inside
    t = [inside, xx]
    for _ in range(2, d):
        t.append(2 * xx * t[-1] - t[-2])
    return torch.stack(t[:d], -1)


def _wrap(p):
    p = torch.where(p < 0, p + 1, p)
    return torch.where(p >= 1, p - 1, p)


def _spread3(c):
    r = torch.zeros_like(c)
    for b in range(21):
        r |= ((c >> b) & 1) << (3 * b)
    return r


class Leaves:
    """Leaf list with keys, for lookups in torch."""

    def __init__(self, anchor, depth):
        self.a = torch.tensor(anchor.astype(np.int64), device="cuda")
        self.d = torch.tensor(depth.astype(np.int64), device="cuda")
        self.key = self._key(self.a << (21 - self.d)[:, None])
        self.scale = 2.0 ** self.d.to(torch.float64)

    @staticmethod
    def _key(c):
        return _spread3(c[:, 0]) | (_spread3(c[:, 1]) << 1) | (_spread3(c[:, 2]) << 2)

    def find(self, p):
        c = (p.detach() * 2097152.0).floor().clamp(0, 2097151).to(torch.int64)
        return torch.searchsorted(self.key, self._key(c), right=True) - 1

    def unit(self, p, leaf):
        s = self.scale[leaf][:, None]
        return (p - self.a[leaf].to(torch.float64) / s) * s


def _eval(lv, coef, q, p):
    leaf = lv.find(p)
    t = _cheb(2.0 * lv.unit(p, leaf) - 1.0, q + 1)
    i, j, k = _triangle(q)
    basis = t[:, 2][:, i] * t[:, 1][:, j] * t[:, 0][:, k]
    return (coef[leaf] * basis[:, None, :]).sum(-1)


def _in_chunks(f, p, per):
    step = max(1024, (1 << 27) // per)
    return torch.cat([f(p[a:a + step]) for a in range(0, len(p), step)])


def _stretched(q):
    d = q + 1
    s = 1.0 / math.cos(0.5 * math.pi / d)
    c = [-math.cos((i + 0.5) * math.pi / d) * s * 0.5 + 0.5 for i in range(d)]
    return torch.tensor(c, dtype=torch.float64, device="cuda")


def _node_basis(q):
    """B [P][Nc]: the triangle basis at the stretched nodes, x fastest."""
    t = _cheb((2 * _stretched(q) - 1).clamp(-1, 1), q + 1)
    i, j, k = _triangle(q)
    return (t[:, None, None, i] * t[None, :, None, j] * t[None, None, :, k]).reshape(-1, ncoef(q))


def _points_of(lv, node):
    g = torch.stack([x.reshape(-1) for x in torch.meshgrid(node, node, node, indexing="ij")][::-1], 1)
    ln = (1.0 / lv.scale)[:, None, None]
    return (lv.a.to(torch.float64)[:, None] * ln + g * ln).reshape(-1, 3)


def _departures(vel, p, t0, t1, nrk, periodic, g, times=None):
    """Midpoint substeps from t0 to t1; vel(k, p): snapshot k's values."""
    tau, t = (t1 - t0) / nrk, t0
    wrap = _wrap if periodic else (lambda x: x)
    for _ in range(nrk):
        p = wrap(p)
        h = wrap(p + 0.5 * tau * _functor(vel, p, t, 1, g, times))
        p = p + tau * _functor(vel, h, t + 0.5 * tau, 2, g, times)
        t += tau
    return p


def _functor(vel, p, t, stage, g, times):
    if g == "prev":  # extrapolated from the current and the previous snapshot
        return vel(0, p) if stage == 1 else 1.5 * vel(0, p) - 0.5 * vel(1, p)
    if g == "set":  # cubic Hermite in time through four snapshots
        v, x = [vel(k, p) for k in range(4)], times
        m1 = (v[2] - v[1]) * 0.5 / (x[2] - x[1]) + (v[1] - v[0]) * 0.5 / (x[1] - x[0])
        m2 = (v[3] - v[2]) * 0.5 / (x[3] - x[2]) + (v[2] - v[1]) * 0.5 / (x[2] - x[1])
        h = x[2] - x[1]
        s = (t - x[1]) / h
        return ((2 * s ** 3 - 3 * s ** 2 + 1) * v[1] + (s ** 3 - 2 * s * s + s) * h * m1
                + (3 * s * s - 2 * s ** 3) * v[2] + (s ** 3 - s * s) * h * m2)
    v = vel(0, p)
    return v * time_factor(t) if g == "cos" else v


def time_factor(t):
    return math.cos(math.pi * t)


# --- inputs --------------------------------------------------------------

def _snapshots(case):
    return {"prev": 2, "set": 4}.get(case.get("g"), 1)


def _times(case):
    return [-0.5 * case["dt"] + case["dt"] * (k - 1) for k in range(4)]


def _inputs(case, seed):
    """(anchor, depth, velocity coefficients per snapshot, concentration
    coefficients) of a Chebyshev case."""
    a, d = leaf_list(case["depth"], case.get("radius", 0.0))
    q = case["q"]
    vel = [fit(velocity_field(seed, case["flow"], -k), a, d, q, 3) for k in range(_snapshots(case))] if "flow" in case else None
    conc = fit(blob_field(seed, case["dof"], case["sigma"]), a, d, q, case["dof"]) if "sigma" in case else None
    return a, d, vel, conc


def _cloud(case, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) * 7 + 5)
    p = torch.rand((case["n"], 3), dtype=torch.float64, device="cuda", generator=g)
    if case["points"] == "cloud":  # particles about CENTRE
        p = 0.5 + 0.12 * torch.randn((case["n"], 3), dtype=torch.float64, device="cuda", generator=g)
        p = (p + torch.tensor(CENTRE, device="cuda") - 0.5).clamp(0.0, 0.999)
    return p


def _batch_problems(case, seed):
    """Problem p's (leaves, degree, velocity, concentration, dt)."""
    r, out = np.random.RandomState(case["n"] * 31 + case["depth"]), []
    for p in range(case["n"]):
        depth, q = case["depth"] - int(r.randint(0, 2)), (6, 8, 10)[p % 3]
        a, d = leaf_list(max(1, depth), 0.0)
        s = int(seed) * 1009 + p
        out.append((a, d, q, fit(velocity_field(s, "waves"), a, d, q, 3),
                    fit(blob_field(s, 1, 0.12), a, d, q, 1), 1e-3 * (1 + p % 4)))
    return out


def prepare(case, seed):
    import tbslas_amd as tb
    from tbslas_amd.batch import Batch

    kind, s = case["kind"], {"case": case}
    if kind == "batch":
        vel, conc, dt = [], [], []
        for a, d, q, v, c, h in _batch_problems(case, seed):
            vel.append(_tree(tb, a, d, q, v))
            conc.append(_tree(tb, a, d, q, c))
            dt.append(h)
        torch.cuda.synchronize()
        s["batch"] = Batch(vel, conc, dt, bc=1)
        s["batch"].tune()
        return s
    if kind == "grid":
        a, d = leaf_list(case["depth"], case.get("radius", 0.0))
        s["points"], v, c = _grid_inputs(case, seed, Leaves(a, d))
        s["vel"], s["conc"] = tb.Grid(a, d, case["n"], 3), tb.Grid(a, d, case["n"], 1)
        s["vel"].set_samples(v)
        s["conc"].set_samples(c)
        s["c0"] = c
        s["dep"] = torch.empty_like(s["points"])
        return s
    a, d, vel, conc = _inputs(case, seed)
    q = case["q"]
    if kind == "refit":
        s["tree"] = tb.Tree(a, d, q, case["dof"])
        s["vals"] = _nodal_values(case, seed, len(d))
        return s
    if kind == "eval":
        s["tree"] = _tree(tb, a, d, q, conc)
        s["pts"] = _cloud(case, seed)
        return s
    trees = [_tree(tb, a, d, q, v) for v in vel]
    if kind == "vjp":
        s["v"], s["c"] = vel[0].requires_grad_(), conc.requires_grad_()
        s["vel"], s["conc"] = trees[0], tb.Tree(a, d, q, case["dof"])
        s["lam"] = _cotangent(conc, seed)
        return s
    if case.get("g") == "prev":
        s["vel"] = tb.Velocity.extrap(*trees)
    elif case.get("g") == "set":
        s["vel"] = tb.Velocity.set(trees, _times(case))
    else:
        s["vel"] = tb.Velocity.tree(trees[0], time_factor if case.get("g") == "cos" else None)
    if kind == "traj":
        s["pts"] = _cloud(case, seed)
    else:
        s["conc"], s["c0"] = _tree(tb, a, d, q, conc), conc
    return s


def _tree(tb, a, d, q, coef):
    t = tb.Tree(a, d, q, coef.shape[1])
    t.set_coeffs(coef)
    return t


def _cotangent(conc, seed):
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 17)
    return torch.randn(conc.shape, dtype=torch.float64, device="cuda", generator=g)


def _nodal_values(case, seed, L):
    g = torch.Generator(device="cuda").manual_seed(int(seed) + 11)
    return torch.randn((L, case["dof"], (case["q"] + 1) ** 3), dtype=torch.float64, device="cuda", generator=g)


def _grid_inputs(case, seed, lv):
    n = case["n"]
    p = _points_of(lv, torch.arange(n, dtype=torch.float64, device="cuda") / (n - 1))
    v = velocity_field(seed, "waves")(p).reshape(-1, n ** 3, 3).transpose(1, 2).contiguous()
    return p, v, blob_field(seed, 1, 0.08)(p).reshape(-1, 1, n ** 3).contiguous()


def _kept(case, t):
    """What the program keeps of a result: float32 in the FP32 modes."""
    return t if case["mode"] == "fp64" else t.float()


def run(s):
    import tbslas_amd as tb
    from tbslas_amd.adjoint import semilag_step

    case = s["case"]
    kind = case["kind"]
    if kind == "eval":
        return _kept(case, s["tree"].eval(s["pts"], case["bc"], case["mode"]))
    if kind == "traj":
        return tb.traj_rk2(s["vel"], s["pts"], 0.0, -case["dt"], case["nrk"], case["bc"])
    if kind == "refit":
        s["tree"].set_grid_values(s["vals"])
        return s["tree"].get_coeffs_device(), s["tree"].grid_values()
    if kind == "step":
        s["conc"].set_coeffs(s["c0"])
        for k in range(case["steps"]):
            tb.semilag_insitu(s["vel"], s["conc"], 1 + k, case["dt"], case["nrk"], case["bc"], case["mode"])
        return _kept(case, s["conc"].get_coeffs_device())
    if kind == "vjp":
        s["c"].grad = s["v"].grad = None
        out = semilag_step(s["c"], s["v"], s["vel"], s["conc"], 1, case["dt"], case["bc"])
        out.backward(s["lam"])
        return out.detach(), s["c"].grad, s["v"].grad
    if kind == "grid":
        s["conc"].set_samples(s["c0"])
        tb.grid_semilag_insitu(s["vel"], s["conc"], 1, case["dt"], 1, case["bc"], case["mode"], dep=s["dep"])
        return s["dep"], _kept(case, s["conc"].eval(s["points"], case["bc"], case["mode"]))
    b = s["batch"]
    b.step(case["steps"])
    # the state is FP32; coeffs() widens it
    return [b.coeffs(p).astype(np.float32) for p in range(case["n"])]


# --- exact values ----------------------------------------------------------

#: point-terms that the 64-bit evaluation below does in about ten seconds
MOST = 2.5e11


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        probs = _batch_problems(case, seed)
        if sum(len(p[1]) * (p[2] + 1) ** 3 * ncoef(p[2]) for p in probs) * case["steps"] > MOST / 3:
            return None
        return [_steps(Leaves(a, d), q, [v], c, h, case["steps"], 1, 1, None, None, stationary=True)
                for a, d, q, v, c, h in probs]
    if kind == "grid":
        return _exact_grid(case, seed)
    q = case["q"]
    nc, P = ncoef(q), (q + 1) ** 3
    points = case.get("n") or num_leaves(case) * P
    terms = {"eval": case.get("dof", 1), "refit": 1, "traj": 2 * case.get("nrk", 1) * 3,
             "vjp": 24, "step": case.get("steps", 1) * (case.get("dof", 1) + 6 * case.get("nrk", 1) * _snapshots(case))}[kind]
    if points * nc * (1 + terms / 4) > MOST:
        return None
    a, d, vel, conc = _inputs(case, seed)
    lv = Leaves(a, d)
    if kind == "refit":
        vals = _nodal_values(case, seed, len(d))
        B = _node_basis(q)
        coef = vals @ torch.linalg.pinv(B).T
        return coef, coef @ B.T
    if kind == "eval":
        p = _cloud(case, seed)
        return _in_chunks(lambda x: _eval(lv, conc, q, _wrap(x) if case["bc"] else x), p, nc * case["dof"])
    if kind == "traj":
        return _in_chunks(lambda x: _departures(lambda k, y: _eval(lv, vel[k], q, y), x, 0.0, -case["dt"], case["nrk"],
                                                case["bc"], case.get("g"), _times(case)), _cloud(case, seed), 4 * nc)
    if kind == "step":
        return _steps(lv, q, vel, conc, case["dt"], case["steps"], case["nrk"], case["bc"], case.get("g"), _times(case))
    # vjp: cotangents of the values at the departure points, chunk by chunk
    pinv = torch.linalg.pinv(_node_basis(q))
    out = _steps(lv, q, vel, conc, case["dt"], 1, 1, case["bc"], None, None)
    u = (_cotangent(conc, seed) @ pinv).transpose(1, 2).reshape(-1, conc.shape[1])
    v, c = vel[0].requires_grad_(), conc.requires_grad_()
    p = _points_of(lv, _stretched(q))
    step = (1 << 25) // (nc * 4)
    for b in range(0, len(p), step):
        x = _departures(lambda k, y: _eval(lv, v, q, y), p[b:b + step], case["dt"], 0.0, 1, case["bc"], None)
        (_eval(lv, c, q, _wrap(x) if case["bc"] else x) * u[b:b + step]).sum().backward()
    return out, c.grad, v.grad


def _steps(lv, q, vel, conc, dt, steps, nrk, periodic, g, times, stationary=False):
    pinv = torch.linalg.pinv(_node_basis(q))
    p, nc, dof = _points_of(lv, _stretched(q)), ncoef(q), conc.shape[1]
    for k in range(steps):
        t0 = dt if stationary else (1 + k) * dt

        def value(x):
            dep = _departures(lambda m, y: _eval(lv, vel[m], q, y), x, t0, t0 - dt, nrk, periodic, g, times)
            return _eval(lv, conc, q, _wrap(dep) if periodic else dep)
        vals = _in_chunks(value, p, nc * max(4, dof)).reshape(-1, (q + 1) ** 3, dof)
        conc = vals.transpose(1, 2) @ pinv.T
    return conc


def _exact_grid(case, seed):
    a, d = leaf_list(case["depth"], case.get("radius", 0.0))
    lv, n = Leaves(a, d), case["n"]
    if len(d) * n ** 3 > 4e7:
        return None
    p, v, c = _grid_inputs(case, seed, lv)
    wrap = _wrap if case["bc"] else (lambda x: x)

    def interp(s, x):
        leaf = lv.find(x)
        u = lv.unit(x, leaf)
        inside = ((u >= 0) & (u <= 1)).all(1)
        t = u * (n - 1)
        first = (t.long() - 1).clamp(0, n - 4)
        t = t - first
        w = []
        for i in range(4):
            m = torch.ones_like(t)
            for j in range(4):
                if i != j:
                    m = m * (t - j) / (i - j)
            w.append(m)
        flat = s.reshape(-1)
        out = torch.zeros((len(x), s.shape[1]), dtype=torch.float64, device="cuda")
        for k in range(s.shape[1]):
            base = (leaf * s.shape[1] + k) * n ** 3 + first[:, 0] + n * (first[:, 1] + n * first[:, 2])
            for z in range(4):
                for y in range(4):
                    for e in range(4):
                        out[:, k] += w[e][:, 0] * w[y][:, 1] * w[z][:, 2] * flat[base + e + n * (y + n * z)]
        return out * inside[:, None]

    def vel_at(_, x):
        return interp(v, x)
    dep = _in_chunks(lambda x: wrap(_departures(vel_at, x, case["dt"], 0.0, 1, case["bc"], None)), p, 256)
    new = _in_chunks(lambda x: interp(c, x), dep, 256).reshape(-1, 1, n ** 3).contiguous()
    return dep, _in_chunks(lambda x: interp(new, wrap(x)), p, 256)


# --- what a pass cannot do without ------------------------------------------

def _refit_flops(q):
    d = q + 1
    return 2.0 * (1.5 * d ** 4 + ncoef(q) * d + ncoef(q) ** 2)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        r, by, fl = np.random.RandomState(case["n"] * 31 + case["depth"]), 0.0, 0.0
        for p in range(case["n"]):
            L, q = 8 ** max(1, case["depth"] - int(r.randint(0, 2))), (6, 8, 10)[p % 3]
            nc = ncoef(q)
            by += case["steps"] * L * nc * 4 * 5 + L * nc * 4
            fl += case["steps"] * L * ((q + 1) ** 3 * (27 * (q + 1) + 14 * nc + 18) + _refit_flops(q))
        return {"bytes": by, "flops": fl}
    L = num_leaves(case)
    if kind == "grid":
        N = L * case["n"] ** 3
        w = 4 if case["mode"] == "fp32" else 8
        return {"bytes": N * (4 * w + 8 + 24 + 24 + w), "flops": N * (2 * 696 + 2 * 280 + 18.0)}
    q, dof, nrk = case["q"], case.get("dof", 3), case.get("nrk", 1)
    nc, P = ncoef(q), (q + 1) ** 3
    w = 8 if case.get("mode", "fp64") == "fp64" else 4
    if kind == "eval":
        return {"bytes": case["n"] * (24.0 + w * dof) + L * dof * nc * w, "flops": case["n"] * (9.0 * (q + 1) + 2 * dof * nc)}
    if kind == "traj":
        return {"bytes": case["n"] * 48.0 + L * 3 * nc * 8, "flops": case["n"] * nrk * (18.0 * (q + 1) + 12 * nc + 18)}
    if kind == "refit":
        return {"bytes": 8.0 * L * dof * (2 * P + nc), "flops": L * dof * (2 * _refit_flops(q) - 2.0 * nc ** 2)}
    trees = _snapshots(case)
    fwd = L * (P * (nrk * (1 + trees) * (9.0 * (q + 1) + 6 * nc) + 9 * (q + 1) + 2 * nc * dof + 18 * nrk) + dof * _refit_flops(q))
    if kind == "vjp":  # each of the step's contractions again, and for both cotangents
        return {"bytes": 8.0 * L * nc * (2 * 3 + 4 * dof), "flops": 3 * fwd}
    return {"bytes": case["steps"] * w * L * nc * (3.0 * trees + 2 * dof), "flops": case["steps"] * fwd}


# --- the cases ---------------------------------------------------------------

def listed():
    return [
        # a few probes read from a small tree: one launch, its latency
        {"name": "eval_1009_probes_q6", "kind": "eval", "depth": 2, "q": 6, "dof": 1, "sigma": 0.2, "n": 1009,
         "points": "uniform", "bc": 0, "mode": "fp64"},
        # a vector field sampled at a million unordered points (a picture, a coupled code's nodes)
        {"name": "eval_1m_scattered_q8", "kind": "eval", "depth": 4, "radius": 0.2, "q": 8, "dof": 3, "sigma": 0.1, "n": 1000003,
         "points": "uniform", "bc": 1, "mode": "fp64"},
        # a cloud of particles carried through a time-dependent flow, four substeps
        {"name": "traj_300k_particles_q8", "kind": "traj", "depth": 4, "q": 8, "flow": "waves", "g": "cos", "dt": 0.02, "nrk": 4,
         "n": 300007, "points": "cloud", "bc": 1},
        # the smallest step of a test or a coarse start: launches count
        {"name": "step_64_leaves_q6", "kind": "step", "depth": 2, "q": 6, "dof": 1, "sigma": 0.06, "flow": "spin", "dt": 0.0314,
         "nrk": 1, "steps": 1, "bc": 0, "mode": "fp64"},
        # an ordinary run: uniform tree, rigid rotation, free space
        {"name": "step_4096_leaves_q8", "kind": "step", "depth": 4, "q": 8, "dof": 1, "sigma": 0.06, "flow": "spin", "dt": 0.0314,
         "nrk": 1, "steps": 2, "bc": 0, "mode": "fp64"},
        # the headline: the adaptive tree of about 36,000 leaves at degree 14, FP32 with the FP64 head
        {"name": "step_36k_leaves_q14_fp32h", "kind": "step", "depth": 5, "radius": 0.155, "q": 14, "dof": 1, "sigma": 0.04,
         "flow": "waves", "g": "cos", "dt": 1e-3, "nrk": 1, "steps": 1, "bc": 1, "mode": "fp32h"},
        # the same path in the default precision on a smaller refined tree
        {"name": "step_5k_leaves_q14_fp64", "kind": "step", "depth": 4, "radius": 0.19, "q": 14, "dof": 1, "sigma": 0.05,
         "flow": "waves", "g": "cos", "dt": 2e-3, "nrk": 1, "steps": 1, "bc": 1, "mode": "fp64"},
        # 64 tracers on one set of trajectories
        {"name": "step_64_tracers_q8_fp32", "kind": "step", "depth": 4, "q": 8, "dof": 64, "sigma": 0.08, "flow": "waves", "dt": 5e-3,
         "nrk": 1, "steps": 1, "bc": 1, "mode": "fp32"},
        # an ensemble of small problems, eight steps between snapshots
        {"name": "batch_24_problems", "kind": "batch", "n": 24, "depth": 4, "steps": 8},
        # a training step: forward and both cotangents
        {"name": "vjp_4096_leaves_q8", "kind": "vjp", "depth": 4, "q": 8, "dof": 1, "sigma": 0.08, "flow": "waves", "dt": 5e-3, "bc": 1},
        # the cubic variant on 8^3 samples per leaf
        {"name": "grid_32k_leaves_n8_fp64", "kind": "grid", "depth": 5, "n": 8, "dt": 2e-3, "bc": 1, "mode": "fp64"},
        # another solver's nodal vector field taken in and handed back
        {"name": "refit_4096_leaves_q10_dof3", "kind": "refit", "depth": 4, "q": 10, "dof": 3},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


#: arithmetic of a drawn case at most: below the largest listed one's
DRAWN_FLOPS = 4e11


def draw(rng):
    while True:
        c = _draw(rng)
        cost = work(c)["flops"] * (2.0 if c.get("mode", "fp64") == "fp64" else 1.0)
        if cost <= DRAWN_FLOPS and (c["kind"] == "grid" or "q" not in c or num_leaves(c) * (c["q"] + 1) ** 3 * max(c.get("dof", 1), 3) <= 4e8):
            return c


def _draw(rng):
    kind = rng.choice(["eval", "eval", "traj", "step", "step", "step", "tracers", "vjp", "grid", "batch", "refit"])
    depth, radius = rng.randint(1, 5), rng.choice([0.0, round(rng.uniform(0.1, 0.3), 3)])
    flow = {"flow": rng.choice(["waves", "waves", "spin"]), "dt": round(math.exp(rng.uniform(math.log(5e-4), math.log(2e-2))), 5)}
    bc = 0 if flow["flow"] == "spin" else 1
    q = rng.choice([3, 4, 5, 6, 7, 8, 8, 9, 10, 11, 12, 13, 14, 14])
    sigma = round(rng.uniform(0.06, 0.15), 3)
    if kind == "eval":
        return {"kind": kind, "depth": depth, "radius": radius, "q": q, "dof": rng.choice([1, 1, 3]), "sigma": sigma,
                "n": _log(rng, 100, 3000000), "points": rng.choice(["uniform", "cloud"]), "bc": rng.choice([0, 1]),
                "mode": rng.choice(["fp64", "fp64", "fp32", "fp32h"])}
    if kind == "traj":
        return {"kind": kind, "depth": depth, "radius": radius, "q": q, "flow": "waves", "dt": flow["dt"],
                "g": rng.choice(["", "cos", "prev"]), "nrk": rng.randint(1, 5), "n": _log(rng, 1000, 1000000),
                "points": rng.choice(["uniform", "cloud"]), "bc": 1}
    if flow["flow"] == "spin":
        sigma = 0.06  # nothing at the faces, where free space cuts off
    if kind == "step":
        g = rng.choice(["", "", "cos", "prev", "set"])
        return {"kind": kind, "depth": depth, "radius": radius, "q": q, "dof": rng.choice([1, 1, 1, 2]), "sigma": sigma,
                **flow, "g": g, "nrk": rng.choice([1, 1, 2]), "steps": rng.choice([1, 2, 3]), "bc": bc,
                "mode": rng.choice(["fp64", "fp64", "fp32", "fp32h"])}
    if kind == "tracers":
        return {"kind": "step", "depth": min(depth, 4), "radius": 0.0, "q": rng.choice([4, 6, 7, 8]),
                "dof": rng.choice([16, 32, 48, 64]), "sigma": sigma, "flow": "waves", "dt": flow["dt"], "g": "", "nrk": 1,
                "steps": 1, "bc": 1, "mode": rng.choice(["fp32", "fp64"])}
    if kind == "vjp":
        return {"kind": kind, "depth": min(depth, 4), "radius": radius, "q": rng.choice([4, 5, 6, 7, 8, 8, 9, 10]), "dof": 1, "sigma": sigma,
                "flow": "waves", "dt": flow["dt"], "bc": 1}
    if kind == "grid":
        return {"kind": kind, "depth": depth, "radius": radius, "n": rng.choice([5, 6, 8, 8, 10]), "dt": flow["dt"], "bc": 1,
                "mode": rng.choice(["fp64", "fp64", "fp32"])}
    if kind == "batch":
        return {"kind": kind, "n": rng.randint(3, 24), "depth": rng.choice([3, 4]), "steps": rng.randint(2, 12)}
    return {"kind": "refit", "depth": depth, "radius": radius, "q": q, "dof": rng.choice([1, 3, 3, 8])}
