"""What becomes of the device memory of the workspace that a context keeps
between MSM calls, seen from outside (free device bytes) and by results."""
import ctypes
import threading

import numpy as np
import pytest

import zyklop_amd as zk

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def free_bytes():
    f, t = ctypes.c_size_t(0), ctypes.c_size_t(0)
    assert zk.lib().hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


class Setup:
    """A context with a resident circuit, and an MSM over its H bases whose
    workspace the context keeps: `held` bytes."""

    def __init__(self, m=300000):
        self.ctx = zk.Context(0)
        self.ctx.set_window_tables(0)
        self.circ = self.ctx.synth_circuit(31, m, 4)
        self.ctx.set_window_tables(-1)
        self.pts, self.n = self.circ.bases(4)
        sc = zk.synth_uniform(3, self.n)
        self.sc = self.ctx.dev_alloc(sc.nbytes)
        self.ctx.upload(self.sc, sc)
        self.small = self.ctx.synth_circuit(32, 400, 4)
        self.ctx.prove(self.small, self.small.witness(1))
        before = free_bytes()
        self.out = self.msm()
        self.held = before - free_bytes()

    def msm(self):
        return self.ctx.msm_g1_device(self.pts, self.sc, self.n)

    def allocated_by_msm(self):
        """Device bytes that the same MSM takes beyond what is kept."""
        before = free_bytes()
        got = self.msm()
        assert got[1] == self.out[1] and np.array_equal(got[0], self.out[0])
        return before - free_bytes()

    def close(self):
        self.ctx.dev_free(self.sc)
        self.circ.free()
        self.small.free()
        self.ctx.close()


@pytest.fixture
def kept():
    s = Setup()
    assert s.held > 64 * MIB
    yield s
    s.close()


def test_submit_leaves_the_workspace(kept):
    """A proof served while memory is plentiful frees nothing: freeing would
    wait for the proofs in flight and the next MSM would allocate again."""
    srv = zk.Server(kept.ctx, max_slots=2, reserve_bytes=1 << 30)
    w = kept.small.witness(2)
    for t in [srv.submit(kept.small, w) for _ in range(6)]:
        srv.wait(t)
    assert kept.allocated_by_msm() < kept.held // 4
    assert srv.prepare([kept.small]) == 2
    assert kept.allocated_by_msm() < kept.held // 4
    srv.close()
    circ = kept.ctx.synth_circuit(33, 500, 4)   # looks at the free memory for its window tables
    assert kept.allocated_by_msm() < kept.held // 4
    circ.free()


def test_admission_takes_the_workspace_where_it_makes_room(kept):
    """A server whose reserve is only met once the idle workspace is given back
    admits the request, as it would if nothing were kept."""
    need = kept.ctx.slot_bytes_check(kept.small)[0]
    free = free_bytes()
    w = kept.small.witness(2)
    srv = zk.Server(kept.ctx, max_slots=1, reserve_bytes=free + kept.held // 2 - need)
    pr, _ = srv.wait(srv.submit(kept.small, w))
    assert free_bytes() - free > kept.held // 4
    srv.close()
    assert np.array_equal(pr.words(), kept.ctx.prove(kept.small, w).words())
    assert kept.allocated_by_msm() > kept.held // 4


def test_workspace_given_back_under_a_running_thread(kept):
    """zk_msm_free_workspace gives the memory back; called over and over while
    another thread runs MSMs on the same context it changes no result."""
    before = free_bytes()
    kept.ctx.free_msm_workspace()
    assert free_bytes() - before > kept.held // 2
    bad = []

    def work():
        for _ in range(20):
            got = kept.msm()
            if got[1] != kept.out[1] or not np.array_equal(got[0], kept.out[0]):
                bad.append(got)

    t = threading.Thread(target=work)
    t.start()
    while t.is_alive():
        kept.ctx.free_msm_workspace()
    t.join()
    assert not bad
