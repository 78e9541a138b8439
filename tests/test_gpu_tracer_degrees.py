"""Many components on the matrix cores against the vector contraction of the
same step, at the degrees about which the chunk of terms is cut: 4 terms, one
to a lane group, and 10, several.  1e-12 of the largest value in FP64 and
2e-6 in FP32, as the other parity bars: sums of at most 10 products of four
factors, 60 roundings of 1.2e-7 / 2 in FP32 if all pointed one way, 3.6e-6,
and no ten values do."""
import numpy as np
import pytest

from conftest import random_tree

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,tol", [("fp64", 1e-12), ("fp32", 2e-6)])
@pytest.mark.parametrize("q,dof", [(1, 16), (1, 80), (2, 48)])
def test_matrix_cores_match_vector_units(tb, q, dof, mode, tol):
    from tbslas_amd import _lib, fields

    leaves = random_tree(3, max_depth=3)
    rng = np.random.default_rng(q)
    deg = np.array([i + j + k for i in range(q + 1) for j in range(q + 1 - i)
                    for k in range(q + 1 - i - j)])
    vel = tb.Tree(*leaves, q, 3, tb.fit_function(fields.taylor_green_2d3, *leaves, q, 3))
    conc = tb.Tree(*leaves, q, dof, rng.standard_normal((len(leaves[1]), dof, tb.ncoef(q))) * 0.5 ** deg)
    out = []
    try:
        for on in (1, 0):
            _lib.set_option(_lib.OPT_TRACER_MFMA, on)
            out.append(tb.semilag_values(vel, conc, 1, 0.02, 1, 1, mode))
    finally:
        _lib.set_option(_lib.OPT_TRACER_MFMA, 1)
    assert float((out[0] - out[1]).abs().max()) <= tol * float(out[1].abs().max())
