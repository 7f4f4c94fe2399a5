"""Transforms above 2^22: the pass layouts 2^8 2^8 2^7, 2^8 2^8 2^8 and the
four-pass 2^6 2^6 2^6 2^7, all four kinds. Uniform data at rows against direct
evaluation of the polynomial by the oracle, and the largest canonical value
everywhere, whose transform is known in every row."""
import numpy as np
import pytest

import oracle as O
import zyklop_amd as zk
from tests import pyref
from tests.test_gpu_configs import uniform_fr

pytestmark = pytest.mark.gpu
RR = pyref.R


@pytest.fixture(scope="module")
def ctx():
    c = zk.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("log_n", [23, 24, 25])
def test_rows_by_definition(ctx, log_n):
    n = 1 << log_n
    rng = np.random.default_rng(9000 + log_n)
    x = uniform_fr(rng, n)
    rows = [0, 1, n // 2, n - 1] + [int(v) for v in rng.integers(2, n - 1, size=4)]
    w, g = pyref.root(log_n), pyref.root(log_n + 1)
    winv, ginv, ninv = pow(w, RR - 2, RR), pow(g, RR - 2, RR), pow(n, RR - 2, RR)
    points = [pow(w, k, RR) for k in rows] + [pow(g, 2 * k + 1, RR) for k in rows] + [pow(winv, k, RR) for k in rows]
    ev = O.poly_eval(x, points)
    fwd, coset, inv = ev[:8], ev[8:16], ev[16:]
    expect = [fwd, [v * ninv % RR for v in inv], coset,
              [v * ninv * pow(ginv, k, RR) % RR for k, v in zip(rows, inv)]]
    for kind in range(4):
        y = ctx.ntt(x, log_n, kind)
        assert [O.from_limbs(y[k]) for k in rows] == expect[kind], kind


@pytest.mark.parametrize("log_n", [23, 24, 25])
@pytest.mark.parametrize("kind", [0, 1])
def test_largest_value_everywhere(ctx, log_n, kind):
    n = 1 << log_n
    x = np.empty((n, 4), np.uint64)
    x[:] = O.to_limbs(RR - 1)
    y = ctx.ntt(x, log_n, kind)
    assert O.from_limbs(y[0]) == ((RR - 1) * n % RR if kind == 0 else RR - 1)
    assert not y[1:].any()
