"""Launch and kernel variants chosen by size: each against the oracle or the general path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def ctx1(nyx, n, lo=(0, 0, 0), hi=(1, 1, 1), **kw):
    return nyx.PMContext(nyx.BoxGeom(tuple(int(v) for v in n), tuple(lo), tuple(hi)), **kw)


def mean_free(n, seed):
    f = np.random.default_rng(seed).standard_normal((n[2], n[1], n[0]))
    return f - f.mean()


@pytest.mark.parametrize("n", [(32, 32, 32), (66, 18, 10), (130, 34, 6), (40, 24, 18)])
def test_residual_chunks_bitwise(nyx, orc, n):
    # the level-0 residual in short z-chunks (small boxes), chunks that do not
    # divide the box and columns that pass its edge: iterates and norms of two
    # V-cycles from a non-zero guess, bit for bit
    f = mean_free(n, 31)
    guess = mean_free(n, 32)
    dx = [1.0 / 32] * 3
    hi = [v / 32 for v in n]
    with ctx1(nyx, n, hi=hi) as c:
        phi, it, norms = c.solve_poisson(f, guess, fixed_iters=2)
    ref, it2, st, _ = orc.mg_solve(n, dx, f, guess, fixed_iters=2)
    assert it == it2 == 2
    assert np.array_equal(phi, ref)
    assert np.array_equal(norms[:3], st[:3])
