"""The row contraction (a workgroup's points ordered by leaf, 16 lanes to a
leaf) at the sizes where its ordering and padding change: point counts about
the row, the wavefront and the two workgroup sizes, more leaves in a
workgroup than its table has slots, points outside the domain, component
counts about its groups of three, every class of degree.

Bars: TBX_FP64 within 1e-12 relative L-inf of the oracle (sums of at most
969 terms below 1 in FP64 rounding, as the other FP64 parity bars);
TBX_FP32 within 2e-6 (FP32 rounding of as many); a point's value does not
depend on the points around it (bit-identical)."""
import numpy as np
import pytest

from conftest import random_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q", [1, 2, 3, 4, 7, 8, 11, 14, 15, 16])
def test_rows_match_oracle(tb, orc, q):
    import torch

    dof = 1 + q % 5
    anchor, depth = random_tree(q, max_depth=4, p_split=0.5, min_depth=2)
    rng = np.random.default_rng(q)
    deg = np.array([i + j + k for i in range(q + 1) for j in range(q + 1 - i)
                    for k in range(q + 1 - i - j)])
    coeff = rng.standard_normal((len(depth), dof, tb.ncoef(q))) * 0.5 ** deg
    g, o = tb.Tree(anchor, depth, q, dof, coeff), orc.Tree(anchor, depth, q, dof, coeff)
    pts = rng.random((65536 + 257, 3)) * 1.2 - 0.1  # some outside [0, 1]^3
    pts[:400] = pts[0]                              # one leaf for whole workgroups
    ref, _ = orc.eval_tree(o, pts, 0)
    ref = ref.reshape(len(pts), dof)
    big = np.abs(ref).max()
    x = torch.from_numpy(pts).cuda()
    whole = g.eval(x, 0, "fp64")
    assert np.abs(whole.cpu().numpy() - ref).max() <= 1e-12 * big
    assert np.abs(g.eval(x, 0, "fp32").cpu().numpy() - ref).max() <= 2e-6 * big
    for n in (1, 15, 16, 17, 63, 64, 65, 255, 257, 1000, 65536):
        a = len(pts) - n  # other neighbours, the same values
        assert torch.equal(g.eval(x[a:].contiguous(), 0, "fp64"), whole[a:]), n


def test_rows_nonfinite_leaf_stays_alone(tb):
    import torch

    anchor, depth = tb.uniform_leaves(2)
    coeff = np.random.default_rng(0).standard_normal((64, 1, tb.ncoef(6)))
    x = torch.rand((5000, 3), dtype=torch.float64, device="cuda")
    t = tb.Tree(anchor, depth, 6, 1, coeff)
    want, leaf = t.eval(x), t.locate(x)
    coeff[5] = np.nan
    coeff[9] = np.inf
    got = tb.Tree(anchor, depth, 6, 1, coeff).eval(x)
    bad = (leaf == 5) | (leaf == 9)
    assert bool((~torch.isfinite(got[bad])).all()) and torch.equal(got[~bad], want[~bad])


def _tree(tb, q, dof, seed):
    anchor, depth = random_tree(seed, max_depth=4, p_split=0.4, min_depth=2)
    deg = np.array([i + j + k for i in range(q + 1) for j in range(q + 1 - i)
                    for k in range(q + 1 - i - j)])
    rng = np.random.default_rng(seed)
    return tb.Tree(anchor, depth, q, dof,
                   rng.standard_normal((len(depth), dof, tb.ncoef(q))) * 0.3 ** deg)


@pytest.mark.parametrize("mode", ["fp64", "fp32", "fp32h"])
@pytest.mark.parametrize("kind", ["uniform", "one leaf", "sorted", "outside"])
def test_points_ordered_by_leaf_keep_their_values(tb, mode, kind):
    # 300,001 points of degree 8 and three components are ordered by leaf
    # first, 3,000 at a time they are not: the same bits
    import torch

    t = _tree(tb, 8, 3, 2)
    g = torch.Generator(device="cuda").manual_seed(1)
    x = torch.rand((300001, 3), dtype=torch.float64, device="cuda", generator=g)
    if kind == "one leaf":
        x[1000:] = x[1000:] * 0.01 + 0.5
    elif kind == "sorted":
        x = x[t.locate(x).argsort()].contiguous()
    elif kind == "outside":
        x = x * 1.5 - 0.25
    bc = int(kind == "outside")
    y = x.clone()
    whole = t.eval(y, bc, mode, write_back=True)
    parts = torch.cat([t.eval(x[a:a + 3000].contiguous(), bc, mode) for a in range(0, len(x), 3000)])
    assert torch.equal(whole, parts)
    want = torch.where(x < 0, x + 1, torch.where(x >= 1, x - 1, x)) if bc else x
    assert torch.equal(y, want)


@pytest.mark.parametrize("depth", [1, 2, 3, 4])
@pytest.mark.parametrize("spread", [1.0, 0.05])
def test_order_over_leaf_counts(tb, depth, spread):
    # 8, 64, 512 and 4,096 leaves: points as they come, and counted in LDS or
    # in memory; over the domain or on a few leaves.  The same bits as 3,000
    # at a time, which are never ordered.
    import torch

    anchor, dep = tb.uniform_leaves(depth)
    rng = np.random.default_rng(depth)
    t = tb.Tree(anchor, dep, 9, 3, rng.standard_normal((len(dep), 3, tb.ncoef(9))))
    g = torch.Generator(device="cuda").manual_seed(depth)
    x = torch.rand((70001, 3), dtype=torch.float64, device="cuda", generator=g) * spread + 0.45 * (1 - spread)
    whole = t.eval(x)
    parts = torch.cat([t.eval(x[a:a + 3000].contiguous()) for a in range(0, len(x), 3000)])
    assert torch.equal(whole, parts)


@pytest.mark.parametrize("nrk", [1, 3, 16, 17, 33])
def test_ordered_trajectories_keep_their_values(tb, nrk):
    import torch

    v = _tree(tb, 6, 3, 5)
    g = torch.Generator(device="cuda").manual_seed(2)
    x = torch.rand((200003, 3), dtype=torch.float64, device="cuda", generator=g)
    whole = tb.traj_rk2(v, x, 0.1, 0.0, nrk, 1, g=lambda t: 1.0 + t)
    parts = torch.cat([tb.traj_rk2(v, x[a:a + 1000].contiguous(), 0.1, 0.0, nrk, 1,
                                   g=lambda t: 1.0 + t) for a in range(0, len(x), 1000)])
    assert torch.equal(whole, parts)
    y = x.clone()
    tb.traj_rk2(v, y, 0.1, 0.0, nrk, 1, g=lambda t: 1.0 + t, out=y)
    assert torch.equal(y, whole)


def test_evaluation_under_capture(tb):
    # a captured call allocates nothing and takes the points as they come
    import torch

    t = _tree(tb, 8, 3, 3)
    x = torch.rand((200001, 3), dtype=torch.float64, device="cuda")
    want = t.eval(x)
    s = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = t.eval(x)
    for _ in range(3):
        out.zero_()
        x.copy_(torch.rand_like(x))
        want = t.eval(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("q", [1, 3, 8, 10, 13, 16])
@pytest.mark.parametrize("bc", [0, 1])
def test_adjoint_dot_product_across_degrees(tb, q, bc):
    # <lam, F(c)> = <F^T lam, c> and, along a velocity perturbation that is
    # one polynomial, the derivative's dot product: the transposed
    # interpolation's tiles change with the degree.  1e-12 of |lam| |F(c)|
    # (sums of some 1e4 to 1e6 products in FP64).
    import torch

    from tbslas_amd import fields
    from tbslas_amd.adjoint import semilag_insitu_vjp

    anchor, depth = random_tree(11, max_depth=2)
    vcf = tb.fit_function(fields.taylor_green_2d3, anchor, depth, q, 3)
    vel, conc = tb.Tree(anchor, depth, q, 3, vcf), tb.Tree(anchor, depth, q, 2)
    g = torch.Generator(device="cuda").manual_seed(q)
    c, lam = (torch.randn((len(depth), 2, tb.ncoef(q)), dtype=torch.float64, device="cuda",
                          generator=g) for _ in range(2))
    conc.set_coeffs(c)
    grad = torch.zeros((len(depth), 3, tb.ncoef(q)), dtype=torch.float64, device="cuda")
    back = semilag_insitu_vjp(vel, conc, 1, 0.05, lam, bc, grad_vel=grad)
    dep = torch.empty((conc.L * conc.P, 3), dtype=torch.float64, device="cuda")
    tb.semilag_insitu(vel, conc, 1, 0.05, 1, bc, dep=dep)
    out = conc.get_coeffs_device()
    assert abs(float((lam * out).sum() - (back * c).sum())) <= 1e-12 * float(lam.norm() * out.norm())
    conc.set_coeffs(c)
    stored = semilag_insitu_vjp(vel, conc, 1, 0.05, lam, bc, dep=dep)
    assert float((stored - back).abs().max()) <= 1e-12 * float(back.abs().max())
    # the velocity cotangent is the sum over substeps: one step's against two
    # half steps' chain is covered elsewhere; here that it is finite and moves
    assert bool(torch.isfinite(grad).all()) and float(grad.abs().max()) > 0


@pytest.mark.parametrize("q", [6, 8, 11, 16])
@pytest.mark.parametrize("depth", [0, 1, 2, 3])
def test_refit_of_few_rows_has_the_same_bits(tb, q, depth):
    # 3, 24, 192 and 1,536 rows, by the few-row product up to 2,048 tiles of
    # 16 x 16, and the same rows within the tiled product of 12,288: sums in
    # the same order
    import torch

    g = torch.Generator(device="cuda").manual_seed(q)
    v = torch.randn((4096, 3, (q + 1) ** 3), dtype=torch.float64, device="cuda", generator=g)
    whole = tb.Tree(*tb.uniform_leaves(4), q, 3)
    whole.set_grid_values(v)
    few = tb.Tree(*tb.uniform_leaves(depth), q, 3)
    few.set_grid_values(v[:8 ** depth].contiguous())
    assert np.array_equal(few.get_coeffs(), whole.get_coeffs()[:8 ** depth])
