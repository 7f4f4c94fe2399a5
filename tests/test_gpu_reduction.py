"""The bucket reduction (tree of joins by lane groups) at the edges of its
shapes, through the MSM entry points, bit for bit against the oracle: windows
whose bucket sets take one, two or three tree launches, sets of exactly one
tile, and sets large enough for the level-1 segments. Equal and opposite points
in neighbouring buckets make the joins meet equal operands (doubling), opposite
ones (infinity) and infinity on either side."""
import numpy as np
import pytest

import oracle as O
import zyklop_amd as zk
from tests import pyref
from tests.test_gpu_parity import mont_pts_g1, mont_pts_g2, oracle_msm_g1, oracle_msm_g2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = zk.Context(0)
    yield c
    c.close()


def scalars(vals):
    return np.array([[(v >> (64 * i)) & (2**64 - 1) for i in range(4)] for v in vals], dtype=np.uint64)


def cases(n):
    """(point multiples, scalars): one point in n neighbouring buckets; the
    same with alternating signs; full-size scalars over few points."""
    rng = np.random.default_rng(7)
    full = [int.from_bytes(rng.bytes(32), "little") % pyref.R for _ in range(n)]
    yield [1] * n, list(range(1, n + 1))
    yield [1 if i % 4 < 2 else pyref.R - 1 for i in range(n)], list(range(1, n + 1))
    yield [1 + i % 3 for i in range(n)], full


@pytest.mark.parametrize("window", [4, 8, 9, 15, 16, 19])
def test_reduction_g1(ctx, window):
    for ks, vals in cases(300):
        pts, sc = mont_pts_g1(ks), scalars(vals)
        expect, expect_inf = oracle_msm_g1(pts, sc)
        got, inf = ctx.msm_g1(pts, sc, window)
        assert inf == expect_inf and (inf or np.array_equal(got, expect))


@pytest.mark.parametrize("window", [4, 7, 8, 13, 16, 19])
def test_reduction_g2(ctx, window):
    for ks, vals in cases(150):
        pts, sc = mont_pts_g2(ks), scalars(vals)
        expect, expect_inf = oracle_msm_g2(pts, sc)
        got, inf = ctx.msm_g2(pts, sc, window)
        assert inf == expect_inf and (inf or np.array_equal(got, expect))


@pytest.mark.parametrize("g2,n", [(False, 40), (False, 1500), (True, 40), (True, 600)])
def test_many_parts_per_bucket(ctx, g2, n):
    """Few buckets, so that each is accumulated in 2 to 64 parts (joined before
    any bit of the bucket index): the smallest window, all scalars full size."""
    three = (mont_pts_g2 if g2 else mont_pts_g1)([1, 2, pyref.R - 3])
    pts, sc = np.ascontiguousarray(three[np.arange(n) % 3]), zk.synth_uniform(5, n)
    expect, expect_inf = (oracle_msm_g2 if g2 else oracle_msm_g1)(pts, sc)
    for window in (4, 5):
        got, inf = (ctx.msm_g2 if g2 else ctx.msm_g1)(pts, sc, window)
        assert inf == expect_inf and np.array_equal(got, expect)


@pytest.mark.parametrize("g2,n", [(False, 65), (False, 512), (False, 513), (False, 1100), (True, 65), (True, 513)])
def test_oversized_bucket_chunks(ctx, g2, n):
    """One bucket far above the mean load, at the edges of its chunks: equal,
    opposite and infinite bases in every lane's sum, and bases that cancel."""
    four = (mont_pts_g2 if g2 else mont_pts_g1)([1, pyref.R - 1, 0, 5])
    for pattern in ([0], [0, 1], [3, 2, 0, 1, 0]):
        pts = np.ascontiguousarray(four[np.resize(pattern, n)])
        sc = scalars([1] * (n - 1) + [pyref.R - 1])
        expect, expect_inf = (oracle_msm_g2 if g2 else oracle_msm_g1)(pts, sc)
        got, inf = (ctx.msm_g2 if g2 else ctx.msm_g1)(pts, sc)
        assert inf == expect_inf and (inf or np.array_equal(got, expect))


def test_oversized_bucket_most_chunks(ctx):
    """A bucket whose chunks grow because their number is bounded (above 2^19
    entries), beside two light ones; sums of known multiples of the generator."""
    n = 600001
    three = mont_pts_g1([1, 2, 7])
    pts = np.ascontiguousarray(three[np.arange(n) % 3])
    vals = np.zeros((n, 4), np.uint64)
    vals[:, 0] = 1
    vals[:5, 0] = [9, 12, 0, 9, 3]
    total = sum(int(v) * [1, 2, 7][i % 3] for i, v in enumerate(vals[:, 0]))
    expect = mont_pts_g1([total])[0]
    got, inf = ctx.msm_g1(pts, vals)
    assert not inf and np.array_equal(got, expect)


@pytest.mark.parametrize("m", [300, 2500, 8200, 17000])
def test_parts_of_few_buckets_in_proofs(tmp_path, m):
    """A proof over few buckets takes more parts per bucket than a tuning table
    can name: the same proof as with one part and the trapdoor closed form's."""
    c = zk.Context(0)
    circ = c.synth_circuit(91, m, 8)
    w = circ.witness(5)
    r, s = zk.synth_blinding(6)
    base = c.prove(circ, w, r, s).words()
    counted, held, left = c.slot_bytes_check(circ)
    assert counted == held and left == 0
    c.autotune(circ)
    path = tmp_path / "t.txt"
    c.tune_save(path)
    rows = [ln.split() for ln in path.read_text().splitlines() if not ln.startswith("#")]
    path.write_text("".join(" ".join(row[:4]) + " 1 1\n" for row in rows))
    one = zk.Context(0)
    one.tune_load(path)
    assert np.array_equal(one.prove(circ, w, r, s).words(), base)
    one.close()
    ref = O.Circuit(91, m, 8, with_crs=False)
    assert np.array_equal(base, ref.prove_trapdoor(r, s, w=w))
    circ.free()
    c.close()
