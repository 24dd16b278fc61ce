"""The window combination's exceptional additions: a window sum equal to the
running sum (a doubling) or to its negative (infinity, with windows still to
come), windows that sum to infinity, and a chain that starts at infinity."""
import numpy as np
import pytest

import oracle as O
from cusnarks_amd import inputs
from cusnarks_amd import _capi
from cusnarks_amd.device import DeviceBuffer
from cusnarks_amd.msm import fixed_base, msm_device, msm_host
from oracle import pyoracle as P
from tests.gpu_util import dot_mod_r, gen_mul

pytestmark = pytest.mark.gpu


def _case(c, g2, base, plus):
    """Scalars and multiples of the generator: base 2^c under 1, and base
    under 2^c as the second window's only entry, so the running sum meets the
    first window's sum base 2^c (plus) or its negative."""
    k = [1, 1 << c]
    s = [base << c if plus else -base << c, base]
    return k, s


@pytest.mark.parametrize("g2", [False, True])
@pytest.mark.parametrize("c", [3, 8])
@pytest.mark.parametrize("plus", [True, False])
def test_equal_and_opposite_window_sums(g2, c, plus):
    k, s = _case(c, g2, 5, plus)
    # the same one window pair higher, with more windows below it
    k2 = [x << (2 * c) for x in k] + [1, 3]
    s2 = s + [7, 11]
    for ks, ss in ((k, s), (k2, s2)):
        pts = np.stack([gen_mul(x, g2) for x in ss])
        want = gen_mul(sum(a * b for a, b in zip(ks, ss)), g2)
        got = msm_host(inputs.from_ints(ks), pts, g2=g2, window_bits=c)
        if sum(a * b for a, b in zip(ks, ss)) % P.RR == 0:
            want = np.array(P.g2_to_words(None) if g2 else P.g1_to_words(None), np.uint32)
        assert np.array_equal(got, want)
        exp, _ = O.ec_jacreduce(inputs.from_ints(ks), pts, ec2=g2)
        assert np.array_equal(got, exp)


@pytest.mark.parametrize("g2", [False, True])
def test_sparse_windows(g2):
    # one entry each in a few far-apart windows: the windows between are infinity
    ks = [1 << 250, (1 << 131) + 1, 1 << 64]
    ss = [3, 1 << 40, P.RR - 9]
    pts = np.stack([gen_mul(x, g2) for x in ss])
    got = msm_host(inputs.from_ints(ks), pts, g2=g2, window_bits=7)
    assert np.array_equal(got, gen_mul(sum(a * b for a, b in zip(ks, ss)) % P.RR, g2))


@pytest.mark.parametrize("g2", [False, True])
@pytest.mark.parametrize("c", [2, 3, 6, 10, 13, 17])
@pytest.mark.parametrize("reduce_seg", [0, 1, 2, 32])
def test_reduction_shapes(g2, c, reduce_seg):
    # one to three joining passes, windows down to two buckets, segments that
    # are most of a window; equal points put equal sums in neighbouring nodes
    n = 90
    ks = inputs.field_elements(40, n)
    ks[:30] = ks[0]
    exps = [1 + (i % 7) for i in range(n)]
    base = {e: gen_mul(e, g2) for e in set(exps)}
    pts = np.stack([base[e] for e in exps])
    want = gen_mul(sum(k * e for k, e in zip(inputs.to_ints(ks), exps)) % P.RR, g2)
    assert np.array_equal(msm_host(ks, pts, g2=g2, window_bits=c, reduce_seg=min(reduce_seg, 1 << (c - 1))), want)


@pytest.mark.parametrize("n,g2", [(9000, False), (33000, False), (150001, False), (40001, True)])
def test_wire_value_scalars(n, g2):
    # one bucket holds most of the entries: long first-pass bins (a launch of
    # their own above 4 tiles) and carry chains of more than 64 chunks
    ctx = _capi.default_context()
    rng = np.random.default_rng(n)
    k = inputs.field_elements(50, n, nonzero=True)
    sc = inputs.field_elements(51, n)
    u = rng.random(n)
    sc[u < 0.9, 1:] = 0
    sc[u < 0.7, 0] = 1
    d_k, d_s = DeviceBuffer.from_array(ctx, k), DeviceBuffer.from_array(ctx, sc)
    pts, out = DeviceBuffer(ctx, n * (128 if g2 else 64)), DeviceBuffer(ctx, 128)
    fixed_base(d_k, n, pts, g2=g2)
    want = gen_mul(dot_mod_r(k, sc), g2)
    for c in (0, 9):
        msm_device(d_s, pts, n, out, g2=g2, window_bits=c)
        assert np.array_equal(out.download((32 if g2 else 16,)), want)


@pytest.mark.parametrize("g2,n", [(False, 127 * 2048), (False, 127 * 2048 + 1), (True, 127 * 1024), (True, 127 * 1024 + 1)])
def test_points_converted_apart(g2, n):
    # 127 sort tiles: other workgroups write the points; 128: the digits' own
    ctx = _capi.default_context()
    k, sc = inputs.field_elements(52, n, nonzero=True), inputs.field_elements(53, n)
    d_k, d_s = DeviceBuffer.from_array(ctx, k), DeviceBuffer.from_array(ctx, sc)
    pts, out = DeviceBuffer(ctx, n * (128 if g2 else 64)), DeviceBuffer(ctx, 128)
    fixed_base(d_k, n, pts, g2=g2)
    msm_device(d_s, pts, n, out, g2=g2, window_bits=13)
    assert np.array_equal(out.download((32 if g2 else 16,)), gen_mul(dot_mod_r(k, sc), g2))
