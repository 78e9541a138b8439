"""The velocity cotangent of an in-situ step by value: against torch's
autograd through the same step written out in float64 (locate, the triangle
basis, RK2, the pinv refit), at every class of degree, over one and two RK2
substeps, in TBX_FP64 and TBX_EXACT, and with more leaves among a workgroup's
points than its table of leaves holds.

Bar: 1e-11 of the largest entry.  An entry sums products of at most 969
coefficients with basis derivatives (up to q^2 = 256 times the basis) in
FP64: 969 x 256 x 1.1e-16 = 2.7e-11 if every rounding pointed one way, and
roundings of some hundred such products do not."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

TOL = 1e-11


def _cheb(x, d):
    import torch

    inside = (x.abs() <= 1).to(x.dtype)
    x = x * inside
    t = [inside, x]
    for _ in range(2, d):
        t.append(2 * x * t[-1] - t[-2])
    return torch.stack(t[:d], -1)


def _triangle(q):
    import torch

    t = [(i, j, k) for i in range(q + 1) for j in range(q + 1 - i) for k in range(q + 1 - i - j)]
    return torch.tensor(t, device="cuda").T


def _value(tree, coeff, p, bc):
    # p as the call sees it; locate wraps by itself
    import torch

    leaf = tree.locate(p.detach().contiguous(), bc).long()
    a = torch.tensor(tree.anchor.astype(np.float64), device="cuda")[leaf]
    s = torch.tensor(2.0 ** tree.depth.astype(np.float64), device="cuda")[leaf][:, None]
    w = _wrap(p) if bc else p
    t = _cheb(2.0 * (w - a / s) * s - 1.0, tree.q + 1)
    i, j, k = _triangle(tree.q)
    return (coeff[leaf] * (t[:, 2][:, i] * t[:, 1][:, j] * t[:, 0][:, k])[:, None, :]).sum(-1)


def _wrap(p):
    import torch

    p = torch.where(p < 0, p + 1, p)
    return torch.where(p >= 1, p - 1, p)


def _reference(tb, vel, conc, vc, cc, lam, dt, nsub, bc):
    import torch

    M = torch.tensor(tb.pt2coeff_matrix(vel.q), device="cuda").reshape(conc.P, conc.nc)  # [P][Nc]
    u = (lam @ M.T).transpose(1, 2).reshape(-1, conc.dof)
    v = vc.clone().requires_grad_()
    pts = conc.grid_points()
    tau, step = -dt / nsub, max(256, (1 << 24) // (4 * vel.nc))
    for b in range(0, len(pts), step):
        x = pts[b:b + step]
        for _ in range(nsub):
            x = _wrap(x) if bc else x
            h = x + 0.5 * tau * _value(vel, v, x, bc)
            x = x + tau * _value(vel, v, h, bc)
        (_value(conc, cc, x, bc) * u[b:b + step]).sum().backward()
    return v.grad


def _field(tb, leaves, q, dof, seed, decay, size):
    import torch

    deg = np.array([i + j + k for i in range(q + 1) for j in range(q + 1 - i)
                    for k in range(q + 1 - i - j)])
    c = size * np.random.default_rng(seed).standard_normal((len(leaves[1]), dof, tb.ncoef(q))) * decay ** deg
    return tb.Tree(*leaves, q, dof, c), torch.tensor(c, device="cuda")


def _check(tb, leaves, q, dof, mode, nsub, bc, size, dt):
    import torch

    from tbslas_amd.adjoint import semilag_insitu_vjp

    vel, vc = _field(tb, leaves, q, 3, q, 0.5, size)
    conc, cc = _field(tb, leaves, q, dof, 100 + q, 0.3, 1.0)
    lam = torch.tensor(np.random.default_rng(q + 7).standard_normal(cc.shape), device="cuda")
    want = _reference(tb, vel, conc, vc, cc, lam, dt, nsub, bc)
    got = torch.zeros_like(vc)
    semilag_insitu_vjp(vel, conc, 1, dt, lam, bc, mode, grad_vel=got, num_rk_step=nsub)
    assert float((got - want).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("mode", ["fp64", "exact"])
@pytest.mark.parametrize("q", [1, 2, 3, 4, 5, 8, 10, 11, 13, 15, 16])
def test_across_degrees(tb, q, mode):
    _check(tb, tb.uniform_leaves(1), q, 1 + q % 2, mode, 1 + (q < 9), 1, 1.0, 0.02)


@pytest.mark.parametrize("mode", ["fp64", "exact"])
@pytest.mark.parametrize("q,depth", [(1, 3), (2, 3), (3, 3), (6, 2), (7, 3)])
def test_many_leaves_in_a_workgroup(tb, q, depth, mode):
    # velocities that differ from leaf to leaf throw a workgroup's points all
    # over the tree
    _check(tb, tb.uniform_leaves(depth), q, 1, mode, 2, 1, 1.0, 0.2)
