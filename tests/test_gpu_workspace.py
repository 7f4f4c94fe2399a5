"""The MSM workspace a context keeps between calls: results do not depend on
what ran before (other curve, size, window, skew), on another thread taking
idle workspaces back, or on a second context at work."""
import threading

import numpy as np
import pytest

import zyklop_amd as zk
from tests.test_gpu_parity import mont_pts_g1, mont_pts_g2, oracle_msm_g1, oracle_msm_g2

pytestmark = pytest.mark.gpu


def problem(n, g2, small, seed):
    ks = [1 + (i * 7 + seed) % 11 for i in range(n)]
    pts = (mont_pts_g2 if g2 else mont_pts_g1)(ks)
    sc = zk.synth_uniform(seed, n)
    if small:
        sc[:, 1:] = 0
        sc[:, 0] %= 3
    expect, inf = (oracle_msm_g2 if g2 else oracle_msm_g1)(pts, sc)
    return pts, sc, expect, inf


def check(ctx, p, g2, window):
    pts, sc, expect, inf = p
    got, got_inf = (ctx.msm_g2 if g2 else ctx.msm_g1)(pts, sc, window)
    assert got_inf == inf and (inf or np.array_equal(got, expect))


SHAPES = [(700, False, False, 0), (40, True, False, 8), (3, False, False, 13), (2500, False, True, 0),
          (90, True, True, 4), (700, False, False, 19), (0, False, False, 0), (701, False, False, 5)]


def test_results_do_not_depend_on_earlier_calls():
    probs = [problem(n, g2, small, 50 + i) for i, (n, g2, small, _) in enumerate(SHAPES)]
    ctx = zk.Context(0)
    for _ in range(2):
        for p, (_, g2, _, window) in zip(probs, SHAPES):
            check(ctx, p, g2, window)
    ctx.close()


def test_workspaces_taken_back_by_another_thread():
    """A circuit load asks for free memory, which takes idle workspaces back,
    while two contexts run MSMs on threads of their own."""
    probs = [problem(n, g2, small, 80 + i) for i, (n, g2, small, _) in enumerate(SHAPES[:4])]
    errors = []

    def work():
        try:
            ctx = zk.Context(0)
            for _ in range(4):
                for p, (_, g2, _, window) in zip(probs, SHAPES):
                    check(ctx, p, g2, window)
            ctx.close()
        except Exception as e:   # reported below, on the main thread
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    ctx = zk.Context(0)
    for i in range(4):
        ctx.synth_circuit(3 + i, 200, 2).free()
    for t in threads:
        t.join()
    ctx.close()
    assert not errors, errors
