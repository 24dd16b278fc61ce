"""Headers of device code that hold plain integer arithmetic, compiled for the
host and compared with Python integers."""
import ctypes
import os
import random
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "cusnarks_amd", "csrc")
Q = 21888242871839275222246405745257275088696311157297823662689037894645226208583
R = 21888242871839275222246405745257275088548364400416034343698204186575808495617
W8 = ctypes.c_uint32 * 8


def words(v):
    return W8(*[(v >> (32 * i)) & 0xFFFFFFFF for i in range(8)])


def value(w):
    return sum(int(x) << (32 * i) for i, x in enumerate(w))


def compiled(tmp_path, header, body):
    src = tmp_path / "h.cpp"
    src.write_text('#define __device__\n#define __constant__\n#define __forceinline__ inline\n#include <stdint.h>\n'
                   '#include "%s"\nextern "C" %s\n' % (os.path.join(CSRC, header), body))
    so = str(tmp_path / "h.so")
    subprocess.run(["g++", "-O2", "-shared", "-fPIC", "-o", so, str(src)], check=True)
    return ctypes.CDLL(so)


@pytest.mark.parametrize("p", [Q, R])
def test_division_step_inverse(tmp_path, p):
    L = compiled(tmp_path, "inv30.h", "void inv(const uint32_t *a, const uint32_t *p, uint32_t np, uint32_t *o) "
                                      "{ csk::i30_inverse<false>(a, p, np, o); }")
    rng = random.Random(5)
    np_ = -pow(p, -1, 1 << 32) % (1 << 32)
    xs = [1, 2, 3, p - 1, p - 2, (p + 1) // 2, p // 2, 1 << 253, p + 5, 2**256 - 1]
    xs += [rng.randrange(1, p) for _ in range(3000)] + [rng.randrange(1, 1 << rng.randrange(1, 254)) for _ in range(500)]
    for x in xs:
        o = W8()
        L.inv(words(x), words(p), np_, o)
        assert value(o) < p and value(o) * x % p == 1, hex(x)


LAMBDA = 4407920970296243842393367215006156084916469457145843978461


def test_scalar_split(tmp_path):
    L = compiled(tmp_path, "glv.h", "uint32_t split(const uint32_t *k, uint32_t *a, uint32_t *b) "
                                    "{ return csk::glv_split(k, a, b); }")
    assert pow(LAMBDA, 3, R) == 1 and LAMBDA != 1
    rng = random.Random(6)
    ks = [0, 1, 2, R - 1, R - 2, R // 2, R // 2 + 1, R // 3, LAMBDA, LAMBDA - 1, LAMBDA + 1, R - LAMBDA, (1 << 253)]
    ks += [rng.randrange(R) for _ in range(5000)] + [rng.randrange(1 << rng.randrange(1, 253)) for _ in range(500)]
    # where c1 or c2 is half way between two whole numbers
    for n in (9931322734385697763, 147946756881789319000765030803803410728):
        ks += [x for c in (0, 1, 12345, n - 1) for d in range(-2, 3) for x in [(2 * c + 1) * R // (2 * n) + d] if 0 <= x < R]
    for k in ks:
        a, b = W8(), W8()
        neg = L.split(words(k), a, b)
        k1 = -value(a) if neg & 1 else value(a)
        k2 = -value(b) if neg & 2 else value(b)
        assert (k1 + k2 * LAMBDA - k) % R == 0 and abs(k1) < 1 << 126 and abs(k2) < 1 << 126, hex(k)
        if k < 1 << 100:
            assert (k1, k2) == (k, 0)  # small scalars (most wire values) stay small


@pytest.mark.parametrize("least", [4, 8])
@pytest.mark.parametrize("buckets", [2, 128, 2048, 40960, (1 << 17) - 1, 1 << 17, 1 << 18, 3 << 20])
def test_chunk_length(tmp_path, buckets, least):
    # however many of a plan's entries there are, the chunks fit the slots it has
    L = compiled(tmp_path, "chunk.h", "uint32_t len(uint32_t f, uint32_t l, uint32_t e, uint32_t k) "
                                      "{ return csk::ChunkLen{f, l}(e, k); }\n"
                                      'extern "C" uint64_t most(uint32_t f, uint32_t l, uint32_t e) '
                                      "{ return csk::ChunkLen{f, l}.most(e); }")
    L.len.restype, L.most.restype = ctypes.c_uint32, ctypes.c_uint64
    rng = random.Random(buckets)
    es = {0, 1, 2, 2**31 - 1}
    for k in range(3, 32):
        es |= {min(max(0, (m << k >> 1) + d), 2**31 - 1) for m in (2, 3) for d in (-2, -1, 0, 1, 2)}
    es |= {rng.randrange(1 << rng.randrange(1, 32)) % 2**31 for _ in range(300)}
    for fixed in (0, 1, 5, 300):
        peak = 0
        for e in sorted(es):
            n = L.len(fixed, least, e, buckets)
            assert n >= (fixed or least)
            peak = max(peak, -(-e // n))
            assert peak <= L.most(fixed, least, e), (e, n)
def test_quarter_scalars(tmp_path):
    L = compiled(tmp_path, "glv.h", "uint32_t split(const uint32_t *k, uint32_t *o) "
                                    "{ return csk::gls_split(k, (uint32_t(*)[2])o); }")
    x = 4965661367192848881
    mu = Q % R
    assert mu == 6 * x * x and pow(mu, 2, R) == R - LAMBDA
    rng = random.Random(7)
    ks = [0, 1, 2, R - 1, R - 2, R // 2, R // 2 + 1, R // 3, mu, mu - 1, mu + 1, R - mu, pow(mu, 3, R), (1 << 253)]
    ks += [rng.randrange(R) for _ in range(5000)] + [rng.randrange(1 << rng.randrange(1, 253)) for _ in range(500)]
    # where a multiple of a basis vector is half way between two whole numbers
    for a in (6 * x**3 - x, 6 * x**3 + 6 * x**2 + 2 * x, 6 * x**3 + 6 * x**2 + 4 * x + 1, 6 * x**3 + 6 * x**2 + x):
        ks += [v for c in (0, 1, 12345, a // 2, a - 1) for d in range(-2, 3) for v in [(2 * c + 1) * R // (2 * a) + d]
               if 0 <= v < R]
    for k in ks:
        o = W8()
        neg = L.split(words(k), o)
        v = [int(o[2 * i]) | int(o[2 * i + 1]) << 32 for i in range(4)]
        v = [-t if neg >> i & 1 else t for i, t in enumerate(v)]
        assert (sum(t * pow(mu, i, R) for i, t in enumerate(v)) - k) % R == 0, hex(k)
        if k < 1 << 63:
            assert v == [k, 0, 0, 0]


@pytest.mark.parametrize("least", [4, 8])
def test_chunk_length_keeps_threads(tmp_path, least):
    # a chunk is longer than full rounds of 2^17 threads need only while it is
    # short and 2^14 threads are left, and no number of entries and buckets asks
    # for more than a plan takes (2^20 entries a chunk)
    L = compiled(tmp_path, "chunk.h", "uint32_t len(uint32_t l, uint32_t e, uint32_t k) "
                                      "{ return csk::ChunkLen{0, l}(e, k); }")
    L.len.restype = ctypes.c_uint32
    rng = random.Random(3)
    es = [1 << k for k in range(31)] + [2**31 - 1] + [rng.randrange(1 << rng.randrange(1, 32)) % 2**31 for _ in range(400)]
    for k in [1 << c for c in range(1, 20)] + [3 << c for c in range(1, 16)]:
        for e in es:
            n = L.len(least, e, k)
            assert n <= 1 << 14, (e, k)
            if n > max(least, -(-e // (1 << 17))):
                assert n <= 48 and e // n >= 1 << 14, (e, k, n)
    for n in range(1000, 4096):  # a table's 32 windows of 8 bits, sorted together
        assert L.len(8, 32 * n, 128) == 8


def test_table_windows_sorted_together(tmp_path):
    # a top window that would sit in one bin of a large joint sort keeps the windows apart
    L = compiled(tmp_path, "chunk.h", "int joint(uint64_t n, uint32_t c, uint32_t w, int g2) "
                                      "{ return csk::table_joint(n, c, w, g2 != 0); }")
    L.joint.argtypes = [ctypes.c_uint64, ctypes.c_uint32, ctypes.c_uint32, ctypes.c_int]
    joint = lambda n, c, g2=False: bool(L.joint(n, c, 254 // c + 1, int(g2)))
    for c in range(2, 21):
        w = 254 // c + 1
        for g2 in (False, True):
            assert joint(4096, c, g2)
            assert not joint((1 << 25) // w // 4096 * 4096 + 4096, c, g2)
            assert joint(min(1 << 18, (1 << 25) // w // 4096 * 4096), c, g2)
    for c in (12, 14, 18):
        assert not joint(1 << 20, c)
    for c in (10, 13, 16, 17):
        assert joint(1 << 20, c)


@pytest.mark.parametrize("p", [Q, R])
def test_inverse_with_a_scale(tmp_path, p):
    L = compiled(tmp_path, "inv30.h", "void inv(const uint32_t *a, const uint32_t *p, uint32_t np, uint32_t *o, "
                                      "const uint32_t *s) { csk::i30_inverse<false>(a, p, np, o, s); }")
    rng = random.Random(8)
    np_ = -pow(p, -1, 1 << 32) % (1 << 32)
    xs = [1, 2, p - 1, p - 2, (p + 1) // 2, p + 1, 2**256 - 1, 2**255, 3 << 200] + [rng.randrange(1, p) for _ in range(3000)]
    for i, x in enumerate(xs):
        s = (0, 1, p - 1, 1 << 253)[i % 8] if i % 8 < 4 else rng.randrange(p)
        o = W8()
        L.inv(words(x), words(p), np_, o, words(s))
        assert value(o) == s * pow(x, -1, p) % p, (hex(x), hex(s))
