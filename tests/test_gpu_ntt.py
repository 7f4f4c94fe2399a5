"""Fr transforms at every pass shape, bit for bit against the oracle: each size
with two points per lane (radices 2^1..2^7, one to three passes) and the sizes
with four points per lane (radices 2^6, 2^7, 2^8), batches with arrays of their
own, all four kinds."""
import ctypes

import numpy as np
import pytest

import oracle as O
import zyklop_amd as zk

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = zk.Context(0)
    yield c
    c.close()


def run(ctx, arrays, log_n, kind):
    nbytes = 32 << log_n
    d_in = [ctx.dev_alloc(nbytes) for _ in arrays]
    d_out = [ctx.dev_alloc(nbytes) for _ in arrays]
    try:
        for p, a in zip(d_in, arrays):
            ctx.upload(p, a)
        ctx.ntt_device(d_in, d_out, log_n, kind)
        return [ctx.download(p, nbytes).reshape(-1, 4) for p in d_out]
    finally:
        for p in d_in + d_out:
            ctx.dev_free(p)


@pytest.mark.parametrize("log_n", [1, 2, 4, 6, 7, 8, 10, 14, 15, 17])
@pytest.mark.parametrize("kind", [0, 1, 2, 3])
def test_two_points_per_lane(ctx, log_n, kind):
    arrays = [zk.synth_uniform(300 + i, 1 << log_n) for i in range(2)]
    arrays[0][0] = 0
    arrays[0][-1] = [0x43E1F593F0000000, 0x2833E84879B97091, 0xB85045B68181585D, 0x30644E72E131A029]   # r - 1
    for a, got in zip(arrays, run(ctx, arrays, log_n, kind)):
        assert np.array_equal(got, O.ntt(a, log_n, kind))


# passes 2^6 2^6 2^6; 2^6 2^6 2^7; 2^8 2^6 2^6; 2^8 2^6 2^7
@pytest.mark.parametrize("log_n,batch,kind", [(18, 1, 1), (18, 4, 0), (18, 4, 3), (19, 1, 2), (19, 2, 1), (19, 2, 2),
                                              (20, 1, 0), (20, 1, 3), (21, 1, 1), (21, 1, 2)])
def test_four_points_per_lane(ctx, log_n, batch, kind):
    arrays = [zk.synth_uniform(400 + i, 1 << log_n) for i in range(batch)]
    got = run(ctx, arrays, log_n, kind)
    for i in {0, batch - 1}:
        assert np.array_equal(got[i], O.ntt(arrays[i], log_n, kind))


def test_in_place_stays_refused_above_16_points(ctx):
    for log_n in (1, 4, 5, 8):
        a = zk.synth_uniform(9, 1 << log_n)
        p = ctx.dev_alloc(a.nbytes)
        ctx.upload(p, a)
        if log_n > 4:
            with pytest.raises(zk.ZkError):
                ctx.ntt_device([p], [ctypes.c_void_p(p.value)], log_n, 0)
        else:
            ctx.ntt_device([p], [ctypes.c_void_p(p.value)], log_n, 0)
            assert np.array_equal(ctx.download(p, a.nbytes).reshape(-1, 4), O.ntt(a, log_n, 0))
        ctx.dev_free(p)
