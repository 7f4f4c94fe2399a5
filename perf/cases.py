"""The work that this prover is given in use, as cases that can be timed.

Every case goes through the public entry points of zyklop_amd on one GPU:

  prove  one Groth16 proof of a resident circuit, the witness in host memory
         (Context.prove) or already on the device (Context.prove_device)
  batch  several proofs of one resident circuit in one call
         (Context.prove_batch_device)
  ntt    Fr transforms of resident arrays (Context.ntt_device), one array or
         three at once, as the H polynomial's A, B and C are
  msm1   a G1 multi-scalar multiplication of resident points and scalars
         (Context.msm_g1_device)
  msm2   the same over G2 (Context.msm_g2_device)

Circuits, witnesses and blinding come from the package's seeded synthetic
workload. All outputs are field elements, points and proofs as 64-bit words,
so they are the same words on every run.
"""
import ctypes
import math

import numpy as np
import torch

import zyklop_amd as zk

P_WORDS_G1, P_WORDS_G2 = 8, 16
# top 64-bit word of the group order; words below it with any lower words are canonical scalars
R_TOP = zk.R >> 192
_ctx = None


def _context():
    """The one context that a program keeps per GPU."""
    global _ctx
    if _ctx is None:
        _ctx = zk.Context(0)
    return _ctx


def listed():
    return [
        # kernel level: the smallest transform (latency of one call), the H
        # polynomial's three arrays of a 2^16-constraint circuit (odd log),
        # and the 2^22 transform of the kernel benchmark
        {"name": "ntt_2p12_coset", "kind": "ntt", "log_n": 12, "batch": 1, "dir": 2},
        {"name": "ntt_2p17_inverse_x3", "kind": "ntt", "log_n": 17, "batch": 3, "dir": 1},
        {"name": "ntt_2p22_forward", "kind": "ntt", "log_n": 22, "batch": 1, "dir": 0},
        # MSMs: a commitment of a thousand points; 2^22 points with uniform
        # scalars (an H-like MSM); a bit-heavy witness vector as circom
        # circuits make it (most wires are 0 or 1)
        {"name": "msm_g1_1000", "kind": "msm1", "n": 1000, "scalars": "uniform"},
        {"name": "msm_g1_2p22", "kind": "msm1", "n": 1 << 22, "scalars": "uniform"},
        {"name": "msm_g1_700001_witness", "kind": "msm1", "n": 700001, "scalars": "witness"},
        {"name": "msm_g2_200003", "kind": "msm2", "n": 200003, "scalars": "uniform"},
        # whole proofs: a small circuit with the witness in host memory, a
        # mid-size one that fills no power of two, and the 2^20-constraint
        # circuit with 4096 public inputs that the benchmark quotes
        {"name": "prove_2p14_host", "kind": "prove", "m": 1 << 14, "n_pub": 1024, "witness": "host"},
        {"name": "prove_200003", "kind": "prove", "m": 200003, "n_pub": 1024, "witness": "device"},
        {"name": "prove_2p20", "kind": "prove", "m": 1 << 20, "n_pub": 4096, "witness": "device"},
        # batched proving: many small proofs, and the quoted circuit
        {"name": "batch_8x50021", "kind": "batch", "m": 50021, "n_pub": 1024, "count": 8},
        {"name": "batch_4x2p20", "kind": "batch", "m": 1 << 20, "n_pub": 4096, "count": 4},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["prove", "prove", "batch", "ntt", "msm1", "msm1", "msm2"])
    if kind == "ntt":
        batch = rng.choice([1, 3])
        return {"kind": kind, "log_n": rng.randint(10, 22 if batch == 1 else 20), "batch": batch,
                "dir": rng.randint(0, 3)}
    if kind == "msm1":
        return {"kind": kind, "n": _log_uniform(rng, 500, 1 << 22), "scalars": rng.choice(["uniform", "witness"])}
    if kind == "msm2":
        return {"kind": kind, "n": _log_uniform(rng, 500, 1 << 20), "scalars": rng.choice(["uniform", "witness"])}
    n_pub = _log_uniform(rng, 1, 4096)
    if kind == "prove":
        return {"kind": kind, "m": _log_uniform(rng, 1 << 13, 1 << 20), "n_pub": n_pub,
                "witness": rng.choice(["host", "device"])}
    m = _log_uniform(rng, 1 << 13, 1 << 19)
    return {"kind": kind, "m": m, "n_pub": n_pub, "count": rng.randint(2, 4 if m > 1 << 17 else 12)}


# ------------------------------------------------------------------ inputs
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform_fr(shape, g):
    """Canonical field elements (4 words each, below the group order)."""
    w = torch.empty(shape + (4,), dtype=torch.int64, device="cuda")
    w[..., :3].random_(-(1 << 63), (1 << 63) - 1, generator=g)
    w[..., 3].random_(0, R_TOP, generator=g)
    return w


def _witness_fr(n, g):
    """A bit-heavy witness: 70 % bits, 10 % 32-bit words, the rest uniform."""
    w = _uniform_fr((n,), g)
    u = torch.rand(n, device="cuda", generator=g)
    small = torch.zeros_like(w)
    small[:, 0] = torch.randint(0, 2, (n,), device="cuda", generator=g)
    words = torch.zeros_like(w)
    words[:, 0] = torch.randint(0, 1 << 32, (n,), device="cuda", generator=g)
    w = torch.where((u < 0.8)[:, None], words, w)
    return torch.where((u < 0.7)[:, None], small, w)


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def _circuit(seed, m, n_pub):
    return _context().synth_circuit(1 + seed, m, n_pub)


def _points(n, g2, seed):
    """n resident CRS points, affine Montgomery: a circuit's H bases, then its
    A' and B1' bases (G1), or its B2' bases (G2)."""
    ctx = _context()
    words = P_WORDS_G2 if g2 else P_WORDS_G1
    m = 1 << 10
    while (m if g2 else 4 * m) < n:
        m *= 2
    ctx.set_window_tables(0)    # the circuit only lends its points
    circ = _circuit(seed, m, 1)
    ctx.set_window_tables(-1)
    pts = torch.empty((n, words), dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    done = 0
    for which in ([2] if g2 else [4, 0, 1]):
        src, count = circ.bases(which)
        k = min(count, n - done)
        if k > 0:
            ctx.dev_copy(ctypes.c_void_p(pts.data_ptr() + done * words * 8), src, k * words * 8)
            done += k
    assert done == n
    circ.free()
    return pts


def _blinding(seed, count):
    rs = [zk.synth_blinding(1000 * seed + i + 1) for i in range(count)]
    return np.stack([r for r, _ in rs]), np.stack([s for _, s in rs])


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    st = {"case": case, "ctx": ctx}
    if kind == "ntt":
        n, b = 1 << case["log_n"], case["batch"]
        st["data"] = _uniform_fr((b, n), _generator(seed))
        st["work"] = torch.empty_like(st["data"])
        st["out"] = torch.empty_like(st["data"])
    elif kind in ("msm1", "msm2"):
        n = case["n"]
        st["points"] = _points(n, kind == "msm2", seed)
        g = _generator(seed)
        st["scalars"] = _witness_fr(n, g) if case["scalars"] == "witness" else _uniform_fr((n,), g)
    else:
        count = case.get("count", 1)
        circ = _circuit(seed, case["m"], case["n_pub"])
        st["circuit"] = circ
        st["r"], st["s"] = _blinding(seed, count)
        if case.get("witness") == "host":
            st["w"] = circ.witness(seed + 7)
        else:
            st["w"] = [torch.empty((circ.n_vars, 4), dtype=torch.int64, device="cuda") for _ in range(count)]
            for i, w in enumerate(st["w"]):
                circ.witness_device(1000 * seed + i, _ptr(w))
    torch.cuda.synchronize()
    return st


def run(st):
    case, ctx = st["case"], st["ctx"]
    kind = case["kind"]
    if kind == "ntt":
        # the transform uses up its input, so a caller that keeps it works on a copy
        data, work, out = st["data"], st["work"], st["out"]
        ctx.dev_copy(_ptr(work), _ptr(data), data.numel() * 8)
        ctx.ntt_device([_ptr(x) for x in work], [_ptr(x) for x in out], case["log_n"], case["dir"])
        return out
    if kind == "msm1":
        point, inf = ctx.msm_g1_device(_ptr(st["points"]), _ptr(st["scalars"]), case["n"])
        return {"point": point, "inf": inf}
    if kind == "msm2":
        point, inf = ctx.msm_g2_device(_ptr(st["points"]), _ptr(st["scalars"]), case["n"])
        return {"point": point, "inf": inf}
    if kind == "prove":
        if case["witness"] == "host":
            return ctx.prove(st["circuit"], st["w"], st["r"][0], st["s"][0]).words()
        return ctx.prove_device(st["circuit"], _ptr(st["w"][0]), st["r"][0], st["s"][0]).words()
    proofs = ctx.prove_batch_device([st["circuit"]] * case["count"], [_ptr(w) for w in st["w"]], st["r"], st["s"])
    return np.stack([p.words() for p in proofs])


# ------------------------------------------------------------------ work
MACS = 136          # 32 x 32-bit multiply-adds of one 254-bit modular product


def _msm_products(n, g2):
    """Field products of a bucket MSM of n points at its best window."""
    add, red = (29, 43) if g2 else (11, 16)
    return min(math.ceil(254 / c) * (add * n + red * 2 ** c) for c in range(6, 23))


def _ntt_products(n):
    return n // 2 * int(math.log2(n))


def work(case):
    kind = case["kind"]
    if kind == "ntt":
        n, b = 1 << case["log_n"], case["batch"]
        return {"bytes": 64 * n * b, "flops": 2 * MACS * _ntt_products(n) * b}
    if kind in ("msm1", "msm2"):
        g2 = kind == "msm2"
        n = case["n"]
        return {"bytes": n * (32 + (128 if g2 else 64)), "flops": 2 * MACS * _msm_products(n, g2)}
    m, n_pub, count = case["m"], case["n_pub"], case.get("count", 1)
    n_vars = m + n_pub + 1
    n = 1 << (m + n_pub).bit_length()
    nnz = 6 * m + n_pub + 1
    # CSR of A and B, bases of A, B1 and C (G1), B2 (G2) and H (G1), the witness
    nbytes = 36 * nnz + n_vars * (3 * 64 + 128) + 64 * n + 32 * n_vars
    products = (3 * _msm_products(n_vars, False) + _msm_products(n_vars, True) + _msm_products(n, False) +
                6 * _ntt_products(n) + nnz + 2 * n)
    return {"bytes": count * nbytes, "flops": count * 2 * MACS * products}
