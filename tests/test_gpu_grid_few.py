"""A grid step's two forms, every gather issued up front (up to 65,536 sample
points) and a plane at a time, against the step written out with evaluations
(a plane at a time at every size): the same bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["fp64", "exact", "fp32"])
@pytest.mark.parametrize("depth,n,dof", [(0, 4, 1), (1, 8, 3), (2, 9, 1), (3, 5, 2), (2, 10, 1),
                                         (2, 11, 1), (3, 8, 1), (2, 16, 3)])
def test_step_is_its_evaluations(tb, depth, n, dof, mode):
    import torch

    from tbslas_amd import _lib
    from tbslas_amd.grid import grid_points

    leaves = tb.uniform_leaves(depth)
    L = len(leaves[1])
    rng = np.random.default_rng(n)
    vel, conc = tb.Grid(*leaves, n, 3), tb.Grid(*leaves, n, dof)
    vel.set_samples(rng.standard_normal((L, 3, n ** 3)))
    conc.set_samples(rng.standard_normal((L, dof, n ** 3)))
    x = torch.from_numpy(np.ascontiguousarray(grid_points(*leaves, n))).cuda()
    old = [_lib.get_option(k) for k in (_lib.OPT_GRID_LDS, _lib.OPT_NODE_VELOCITY)]
    _lib.set_option(_lib.OPT_GRID_LDS, 0)
    _lib.set_option(_lib.OPT_NODE_VELOCITY, 0)  # the first stage too is evaluated
    try:
        dt = 0.0625 * 0.5 ** depth
        half = x + (-0.5 * dt) * vel.eval(x, 0, mode)
        want = x + (-dt) * vel.eval(half, 0, mode)
        vals = conc.eval(want, 0, mode).reshape(L, n ** 3, dof).transpose(1, 2)
        dep = torch.empty_like(x)
        tb.grid_semilag_insitu(vel, conc, 1, dt, 1, 0, mode, dep=dep)
    finally:
        _lib.set_option(_lib.OPT_GRID_LDS, old[0])
        _lib.set_option(_lib.OPT_NODE_VELOCITY, old[1])
    assert torch.equal(dep, want)
    assert np.array_equal(conc.get_samples().reshape(L, dof, -1), vals.cpu().numpy())
