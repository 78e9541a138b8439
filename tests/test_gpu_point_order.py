"""The routes of tbx_eval and tbx_traj_rk2 by the order in which points come:
in runs of a leaf (contracted in place), scattered (ordered by leaf first),
partly both; their scratch between calls, streams and threads.  A point's
value does not depend on the route (bit-identical with calls of 3,000 points,
which neither route takes)."""
import threading

import numpy as np
import pytest

from conftest import random_tree

pytestmark = pytest.mark.gpu


def _tree(tb, leaves, q, dof, seed=0):
    deg = np.array([i + j + k for i in range(q + 1) for j in range(q + 1 - i)
                    for k in range(q + 1 - i - j)])
    rng = np.random.default_rng(seed)
    return tb.Tree(*leaves, q, dof,
                   rng.standard_normal((len(leaves[1]), dof, tb.ncoef(q))) * 0.5 ** deg)


def _points(tree, n, kind, seed, size=1.0):
    import torch

    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.rand((n, 3), dtype=torch.float64, device="cuda", generator=g) * size - (size - 1) / 2
    s = x[tree.locate(x, int(size > 1)).argsort(stable=True)].contiguous()
    if kind == "runs":
        return s
    if kind == "grid":  # faces belong to the neighbours: many changes of leaf, few leaves
        g = tree.grid_points()
        return g.repeat(1 + n // len(g), 1)[:n].contiguous()
    if kind == "half":  # the last half scattered
        return torch.cat([s[:n // 2], x[:n - n // 2]]).contiguous()
    if kind == "runs of 20":  # more leaves in a wavefront, at most two in some rows
        m = n // 20 * 20
        return torch.cat([s[:m].reshape(-1, 20, 3)[torch.randperm(m // 20, device="cuda",
                                                                  generator=g)].reshape(-1, 3), s[m:]]).contiguous()
    return x


def _parts(f, x):
    import torch

    return torch.cat([f(x[a:a + 3000].contiguous()) for a in range(0, len(x), 3000)])


@pytest.mark.parametrize("mode", ["fp64", "fp32", "fp32h"])
@pytest.mark.parametrize("kind", ["runs", "half", "runs of 20", "grid", "scattered"])
@pytest.mark.parametrize("q,dof", [(1, 1), (2, 3), (5, 2), (8, 1), (8, 4), (13, 1), (16, 3)])
def test_route_keeps_values(tb, q, dof, kind, mode):
    import torch

    t = _tree(tb, random_tree(q, max_depth=4, p_split=0.5, min_depth=2), q, dof)
    for n, bc, size in ((65537, 0, 1.0), (150001, 1, 1.3)):
        x = _points(t, n, kind, q, size)
        assert torch.equal(t.eval(x, bc, mode), _parts(lambda p: t.eval(p, bc, mode), x)), (n, bc)


@pytest.mark.parametrize("kind", ["runs", "half", "scattered"])
def test_trajectory_route_keeps_values(tb, kind):
    import torch

    v = _tree(tb, tb.uniform_leaves(3), 7, 3)
    x = _points(v, 120001, kind, 4)
    run = lambda p: tb.traj_rk2(v, p, 0.05, 0.0, 3, 1)
    assert torch.equal(run(x), _parts(run, x))


def test_scratch_between_streams_and_sizes(tb):
    # blocks go back and forth between calls of several sizes on more streams
    # than are kept, with nothing waited for in between
    import torch

    t = _tree(tb, tb.uniform_leaves(3), 8, 3)
    xs = [_points(t, n, "scattered", n) for n in (70001, 300000, 65537, 150003)]
    want = [_parts(t.eval, x) for x in xs]
    torch.cuda.synchronize()
    for rep in range(2):
        streams = [torch.cuda.Stream() for _ in range(12)]
        out = []
        for k in range(48):
            with torch.cuda.stream(streams[k % 12]):
                out.append((k % 4, t.eval(xs[k % 4])))
        torch.cuda.synchronize()
        assert all(torch.equal(o, want[k]) for k, o in out)


def test_scratch_between_threads(tb):
    import torch

    t = _tree(tb, tb.uniform_leaves(3), 8, 3)
    xs = [_points(t, 100000 + 20000 * k, "scattered", k) for k in range(4)]
    want = [_parts(t.eval, x) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(k):
        with torch.cuda.stream(torch.cuda.Stream()):
            got = [t.eval(xs[k]) for _ in range(20)]
            torch.cuda.current_stream().synchronize()
            if not all(torch.equal(o, want[k]) for o in got):
                bad.append(k)

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for w in th:
        w.start()
    for w in th:
        w.join()
    assert not bad
