"""Coefficients that are not finite, at points outside their leaf's box, where
the basis is zero: zero times a NaN or an infinity is a NaN, in every mode as
in TBX_EXACT, by every route of an evaluation and through a step."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MODES = ["fp64", "fp32", "fp32h"]


def _tree(tb, depth, q, dof, bad=()):
    leaves = tb.uniform_leaves(depth)
    c = np.random.default_rng(q).standard_normal((len(leaves[1]), dof, tb.ncoef(q)))
    for leaf, comp, k, v in bad:
        c[leaf, comp, k] = v
    return tb.Tree(*leaves, q, dof, c)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("q", [1, 4, 9, 14])
@pytest.mark.parametrize("n,kind", [(300, "scattered"), (70001, "scattered"), (70001, "runs"),
                                    (400000, "scattered")])
def test_values_outside_the_box(tb, q, n, kind, mode):
    import torch

    last = tb.ncoef(q) - 1
    t = _tree(tb, 2, q, 2, [(0, 0, last, np.nan), (21, 1, 1, np.inf), (63, 1, 0, -np.inf), (42, 0, 2, np.nan)])
    g = torch.Generator(device="cuda").manual_seed(q)
    x = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=g) * 2.0 - 0.5
    if kind == "runs":
        x = x[t.locate(x).argsort(stable=True)].contiguous()
    x[0] = float("nan")
    x[1, 0], x[2, 1] = float("inf"), -float("inf")
    want, got = t.eval(x, 0, "exact"), t.eval(x, 0, mode)
    assert bool(torch.equal(torch.isfinite(got), torch.isfinite(want)))
    out = ((x < 0) | (x > 1) | x.isnan()).any(1)
    assert bool((~torch.isfinite(want[out])).any()) and bool(torch.isfinite(want[out]).any())
    assert float(got[out][torch.isfinite(got[out])].abs().max()) == 0.0


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("depth", [0, 1, 2])
def test_step_through_a_velocity_that_is_not_finite(tb, depth, mode):
    import torch

    vel = _tree(tb, depth, 5, 3, [(0, 0, 1, np.nan), (8 ** depth - 1, 2, 0, np.inf)])
    conc = _tree(tb, depth, 5, 1)
    want = tb.semilag_values(vel, conc, 1, 1e-3, 2, 1, "exact")
    got = tb.semilag_values(vel, conc, 1, 1e-3, 2, 1, mode)
    # a departure point that is no number has the value 0
    assert bool(torch.equal(got == 0, want == 0)) and bool((want == 0).any())
