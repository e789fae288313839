"""Values at the edge of the number range and calls at the edge of what the
engine takes: infinities, zeros and NaN in networks, captured streams, several
streams and contexts, networks with very many vertices."""
import math

import numpy as np
import pytest

from helpers import oracle_eval, rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-12


@pytest.fixture(scope="module")
def eng(q):
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return q.engine_context()


def _chain(q, L, bond, dims=1):
    return q.continuous_siteinds(q.named_grid((L * dims, 1)), map_dimension=dims)


def _comb(q, teeth, digits):
    return q.continuous_siteinds(q.named_comb_tree((teeth, digits)),
                                 [[(i, j) for j in range(1, digits + 1)] for i in range(1, teeth + 1)])


def _overflowing(q, s, bond, rng, scale):
    """Positive cores whose digit-1 slices are `scale` times larger, the root
    negative: points with many 1 digits have the value -inf."""
    f = q.random_itn(s, link_space=bond, rng=rng)
    cores = [rng.uniform(0.5, 1.5, c.shape) / math.sqrt(c[0].size) for c in f.cores]
    for c in cores:
        if c.shape[1] == 2:
            c[:, 1] *= scale
    cores[0] = -cores[0]
    f.set_cores(cores)
    return f


def _same_with_infinities(y, ref):
    # sums of numbers of one sign: relative per value; infinite where the reference is
    inf = np.isinf(ref)
    assert inf.any() and not inf.all()
    assert np.array_equal(y[inf], ref[inf])
    assert np.max(np.abs(y[~inf] / ref[~inf] - 1.0)) < TOL


# ------------------------------------------------------------------ infinite values
@pytest.mark.parametrize("bond,npts", [(1, 7), (2, 1000), (3, 1000), (4, 64), (5, 100), (8, 16384), (9, 1000),
                                       (12, 500), (15, 12288), (16, 1000), (17, 100), (31, 1000), (32, 1000)])
def test_few_points_infinite(q, po, eng, rng, bond, npts):
    # a value that overflows is infinite, not NaN: the lanes past the bond stay zero
    f = _overflowing(q, _chain(q, 13, bond), bond, rng, 1e40)
    xs = rng.uniform(0, 1, (npts, 1))
    xs[:4, 0] = [0.0, 0.25, 0.5, 1.0]
    _same_with_infinities(q.evaluate(f, xs), oracle_eval(po, f, xs))
