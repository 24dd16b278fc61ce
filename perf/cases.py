"""Performance cases of the framework's public entry points.

Every case is work that a program proving with this package has it do: the
multi-exponentiations over a key's points (one call, a batch of uneven ones,
from a fixed-base table), the transforms and the H step, and a whole proof.
All data are on the GPU before the call except a proof's witness, which a
prover hands over in host memory.  Outputs are field elements and points as
32-bit words (int32 here), so they are exact.

Keys of a case:
  op       msm | table | batch | ntt | hstep | prove
  g2       the curve (msm, table)
  n        points (msm, table); the members' sizes are drawn for a batch
  scalars  uniform: field elements as a proof's H coefficients are;
           witness: half of them 0 or 1, a quarter below 2^32, the rest
           uniform, as the wires of a circuit with many bit signals are
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

Q = 21888242871839275222246405745257275088696311157297823662689037894645226208583
R = 21888242871839275222246405745257275088548364400416034343698204186575808495617
TOP = R >> 224  # the scalar field's top word: below it every value is < R


def listed():
    return [
        # one small circuit's public-input or test multiexp: launches and latency
        {"name": "g1_1000", "op": "msm", "g2": False, "n": 1000, "scalars": "uniform"},
        # a small circuit's key, an odd size
        {"name": "g1_20011", "op": "msm", "g2": False, "n": 20011, "scalars": "uniform"},
        # A, B1 and C of a proof: the scalars are wire values, many of them bits
        {"name": "g1_witness_300007", "op": "msm", "g2": False, "n": 300007, "scalars": "witness"},
        # a 2^20-point multiexp, the size of a mid-sized circuit's key
        {"name": "g1_2e20", "op": "msm", "g2": False, "n": 1 << 20, "scalars": "uniform"},
        # the benchmark's multiexp
        {"name": "g1_2e24", "op": "msm", "g2": False, "n": 1 << 24, "scalars": "uniform"},
        # B2 of a small circuit
        {"name": "g2_5003", "op": "msm", "g2": True, "n": 5003, "scalars": "uniform"},
        # B2 of a mid-sized circuit
        {"name": "g2_2e18", "op": "msm", "g2": True, "n": 1 << 18, "scalars": "uniform"},
        # a resident proving key's points, tabulated once and used for every proof
        {"name": "table_g1_100003", "op": "table", "g2": False, "n": 100003, "scalars": "uniform"},
        # many uneven multiexps planned into one pipeline (a server's cohort)
        {"name": "batch_64", "op": "batch", "count": 64, "lg_lo": 10, "lg_hi": 22, "sizes_seed": 7},
        # one transform, natural order in and out
        {"name": "ntt_2e20", "op": "ntt", "log2n": 20, "inverse": False, "fmt": 1},
        # the H polynomial of a 2^20-constraint circuit
        {"name": "hstep_2e21", "op": "hstep", "log2m": 21},
        # a whole proof: witness in host memory in, three points out
        {"name": "prove_50000", "op": "prove", "constraints": 50000, "overlapped": False},
    ]


def _between(rng, lo, hi):
    """A size spread evenly over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng: random.Random):
    op = rng.choice(["msm", "msm", "msm", "table", "batch", "ntt", "hstep", "prove"])
    if op in ("msm", "table"):
        g2 = rng.random() < 0.35
        return {"op": op, "g2": g2, "n": _between(rng, 100, 1 << 18 if g2 else 1 << (22 if op == "msm" else 20)),
                "scalars": rng.choice(["uniform", "witness"])}
    if op == "batch":
        return {"op": op, "count": rng.randint(3, 64), "lg_lo": rng.randint(6, 10), "lg_hi": rng.randint(12, 18),
                "sizes_seed": rng.randrange(1 << 20)}
    if op == "ntt":
        return {"op": op, "log2n": rng.randint(6, 22), "inverse": rng.random() < 0.5, "fmt": rng.randint(0, 1)}
    if op == "hstep":
        return {"op": op, "log2m": rng.randint(8, 21)}
    return {"op": op, "constraints": _between(rng, 1000, 60000) | 1, "overlapped": rng.random() < 0.5}


# ------------------------------------------------------------------ inputs
def _gen(seed, part):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed * 16 + part)
    return g


def _elements(n, seed, part, kind="uniform"):
    """(n, 8) int32: little-endian words of values below R."""
    g = _gen(seed, part)
    a = torch.randint(-(1 << 31), 1 << 31, (n, 8), dtype=torch.int32, device="cuda", generator=g)
    a[:, 7] = torch.randint(0, TOP, (n,), dtype=torch.int32, device="cuda", generator=g)
    if kind == "witness":
        u = torch.rand(n, device="cuda", generator=g)
        a[:, 1:] *= (u >= 0.75).to(torch.int32)[:, None]
        a[:, 0] = torch.where(u < 0.5, a[:, 0] & 1, a[:, 0])
    return a


def _sizes(case):
    r = random.Random(case["sizes_seed"])
    return [int(round(2.0 ** r.uniform(case["lg_lo"], case["lg_hi"]))) for _ in range(case["count"])]


def _points(k, g2):
    """The multiples k_i of the generator, the points of a synthetic key."""
    from cusnarks_amd.msm import fixed_base
    out = torch.empty((k.shape[0], 32 if g2 else 16), dtype=torch.int32, device="cuda")
    fixed_base(k, k.shape[0], out, g2=g2)
    return out


def prepare(case, seed):
    op = case["op"]
    if op in ("msm", "table"):
        n, g2 = case["n"], case["g2"]
        pts = _points(_elements(n, seed, 1), g2)
        st = {"op": op, "n": n, "g2": g2, "scalars": _elements(n, seed, 2, case["scalars"]),
              "out": torch.empty(32 if g2 else 16, dtype=torch.int32, device="cuda")}
        if op == "table":
            from cusnarks_amd.msm import MsmTable
            st["table"] = MsmTable(pts, n, g2=g2)
        else:
            st["points"] = pts
        return st
    if op == "batch":
        from cusnarks_amd.batch import MsmBatch
        sizes = _sizes(case)
        pts = _points(_elements(sum(sizes), seed, 1), False)
        sc = _elements(sum(sizes), seed, 2)
        out = torch.empty((len(sizes), 16), dtype=torch.int32, device="cuda")
        return {"op": op, "batch": MsmBatch(sizes), "scalars": list(sc.split(sizes)),
                "points": list(pts.split(sizes)), "outs": list(out), "out": out}
    if op == "ntt":
        a = _elements(1 << case["log2n"], seed, 1)
        return dict(case, a=a, out=torch.empty_like(a))
    if op == "hstep":
        m = 1 << case["log2m"]
        return dict(case, a=_elements(m, seed, 1), b=_elements(m, seed, 2),
                    out=torch.empty((2 * m, 8), dtype=torch.int32, device="cuda"))
    from cusnarks_amd.prover import GrothProver, OverlappedProver, ProvingKey
    from cusnarks_amd.synth import Circuit, KeyScalars
    nc = case["constraints"]
    circuit = Circuit(nc, nc, n_public=1, seed=seed % (1 << 40))
    pk = ProvingKey(circuit, KeyScalars(circuit, seed=seed % (1 << 40)))
    r = random.Random(seed)
    return {"op": op, "prover": OverlappedProver(pk) if case["overlapped"] else GrothProver(pk),
            "witness": circuit.witness, "r": r.randrange(1, R), "s": r.randrange(1, R)}


def run(st):
    op = st["op"]
    if op == "msm":
        from cusnarks_amd.msm import msm_device
        msm_device(st["scalars"], st["points"], st["n"], st["out"], g2=st["g2"])
        return st["out"]
    if op == "table":
        st["table"].run(st["scalars"], st["out"])
        return st["out"]
    if op == "batch":
        st["batch"].run(st["scalars"], st["points"], st["outs"])
        return st["out"]
    if op == "ntt":
        from cusnarks_amd.poly import ntt_device
        ntt_device(st["a"], st["out"], st["log2n"], inverse=st["inverse"], fmt=st["fmt"])
        return st["out"]
    if op == "hstep":
        from cusnarks_amd.poly import interpolandmul_device
        interpolandmul_device(st["a"], st["b"], st["log2m"], st["out"])
        return st["out"]
    return tuple(p.view(np.int32) for p in st["prover"].prove(st["witness"], st["r"], st["s"]))


# ------------------------------------------------------------------ work
_MUL = 2 * 128  # one 256-bit Montgomery product: 128 32-bit multiply-adds


def _msm_flops(n, g2):
    """Mixed additions (10 products, 3 base-field products each on G2) of the
    bucket method at its best window width: every point once per window and
    each bucket reduced with two additions."""
    adds = min((254 // c + 1) * (n + 2 ** c) for c in range(4, 21))
    return adds * 10 * (3 if g2 else 1) * _MUL


def work(case):
    op = case["op"]
    if op in ("msm", "table"):
        return {"bytes": case["n"] * (160 if case["g2"] else 96), "flops": _msm_flops(case["n"], case["g2"])}
    if op == "batch":
        s = _sizes(case)
        return {"bytes": 96 * sum(s), "flops": sum(_msm_flops(n, False) for n in s)}
    if op == "ntt":
        n = 1 << case["log2n"]
        return {"bytes": 64 * n, "flops": n // 2 * case["log2n"] * _MUL}
    if op == "hstep":
        m, lg = 1 << case["log2m"], case["log2m"]
        return {"bytes": 128 * m, "flops": (4 * (m // 2) * lg + m * (lg + 1)) * _MUL}
    nc = case["constraints"]
    m = 1 << nc.bit_length()
    return {"bytes": nc * (32 + 3 * 64 + 128 + 2 * 3 * 36) + m * 64,
            "flops": 3 * _msm_flops(nc, False) + _msm_flops(m, False) + _msm_flops(nc, True)
            + (2 * m * nc.bit_length() + m * (nc.bit_length() + 1) + 6 * nc) * _MUL}


# ------------------------------------------------------------------ exact results
def _dot(a, b):
    """sum_i a_i b_i mod R over 16-bit limbs: float64 products of 2^20 terms
    stay below 2^53, so every partial sum is exact."""
    total = 0
    for lo in range(0, a.shape[0], 1 << 20):
        x, y = (v[lo:lo + (1 << 20)].contiguous().view(torch.uint16).to(torch.float64) for v in (a, b))
        p = (x.t().contiguous() @ y).cpu().tolist()
        total += sum(int(p[i][j]) << (16 * (i + j)) for i in range(16) for j in range(16))
    return total % R


# Fq2 = Fq[u]/(u^2 + 1) as pairs; G1 coordinates have a zero second component
def _mul(a, b):
    return ((a[0] * b[0] - a[1] * b[1]) % Q, (a[0] * b[1] + a[1] * b[0]) % Q)


def _sub(a, b):
    return ((a[0] - b[0]) % Q, (a[1] - b[1]) % Q)


def _inv(a):
    d = pow(a[0] * a[0] + a[1] * a[1], -1, Q)
    return (a[0] * d % Q, -a[1] * d % Q)


def _add(p, q):
    if p is None or q is None:
        return p or q
    (x1, y1), (x2, y2) = p, q
    if x1 == x2:
        if y1 != y2:
            return None
        xx = _mul(x1, x1)
        lam = _mul((3 * xx[0], 3 * xx[1]), _inv((2 * y1[0] % Q, 2 * y1[1] % Q)))
    else:
        lam = _mul(_sub(y2, y1), _inv(_sub(x2, x1)))
    x3 = _sub(_sub(_mul(lam, lam), x1), x2)
    return x3, _sub(_mul(lam, _sub(x1, x3)), y1)


_G1 = ((1, 0), (2, 0))
_G2 = ((10857046999023057135944570762232829481370756359578518086990519993285655852781,
        11559732032986387107991004021392285783925812861821192530917403151452391805634),
       (8495653923123431417604973247489272438418190587263600148770280649306958101930,
        4082367875863433681332203403145435568316851327593401208105741076214120093531))


def _words(v):
    return np.frombuffer(int(v).to_bytes(32, "little"), dtype=np.int32)


def _multiple(k, g2):
    """k times the generator as the package encodes it (Montgomery, affine)."""
    acc, p = None, _G2 if g2 else _G1
    while k:
        if k & 1:
            acc = _add(acc, p)
        p, k = _add(p, p), k >> 1
    x, y = acc or ((0, 0), (1, 0))
    return np.concatenate([_words((c << 256) % Q) for c in ((*x, *y) if g2 else (x[0], y[0]))])


def _ints(a):
    b = a.cpu().numpy().tobytes()
    return np.array([int.from_bytes(b[i:i + 32], "little") for i in range(0, len(b), 32)], dtype=object)


def _rows(v):
    return np.frombuffer(b"".join(int(x).to_bytes(32, "little") for x in v), dtype=np.int32).reshape(-1, 8)


def _dft(a, inverse):
    """sum_i a_i w^(ik) for the 2^L-th root w = 5^((R-1)/2^L); decimation in
    frequency, then the bit reversal.  The inverse is scaled by 1/N."""
    n = len(a)
    w = pow(5, (R - 1) // n, R)
    w = pow(w, -1, R) if inverse else w
    tw = [1]
    for _ in range(n // 2 - 1):
        tw.append(tw[-1] * w % R)
    tw = np.array(tw, dtype=object)
    x = a.reshape(1, n)
    while x.shape[1] > 1:
        h = x.shape[1] // 2
        u, v = x[:, :h], x[:, h:]
        x = np.stack([(u + v) % R, (u - v) * tw[:: n // (2 * h)][:h] % R], axis=1).reshape(-1, h)
    bits = n.bit_length() - 1
    rev = np.zeros(n, dtype=np.int64)
    for b in range(bits):
        rev |= ((np.arange(n) >> b) & 1) << (bits - 1 - b)
    x = x.reshape(-1)[rev]
    return x * pow(n, -1, R) % R if inverse else x


def exact(case, seed):
    op = case["op"]
    if op in ("msm", "table"):
        return _multiple(_dot(_elements(case["n"], seed, 1), _elements(case["n"], seed, 2, case["scalars"])),
                         case["g2"])
    if op == "batch":
        s = _sizes(case)
        k, c = _elements(sum(s), seed, 1).split(s), _elements(sum(s), seed, 2).split(s)
        return np.stack([_multiple(_dot(a, b), False) for a, b in zip(k, c)])
    unmont = pow(1 << 256, -1, R)
    if op == "ntt" and case["log2n"] <= 20:
        x = _dft(_ints(_elements(1 << case["log2n"], seed, 1)), case["inverse"])
        return _rows(x if case["fmt"] or not case["inverse"] else x * unmont % R)
    if op == "hstep" and case["log2m"] <= 16:
        m = 1 << case["log2m"]
        zero = np.zeros(m, dtype=object)
        a, b = (_dft(np.concatenate([_dft(_ints(_elements(m, seed, p)), True), zero]), False) for p in (1, 2))
        # two Montgomery factors, normal form out
        return _rows(_dft(a * b % R * unmont % R * unmont % R, True))
    return None  # large transforms and whole proofs: over 20 seconds in Python integers
