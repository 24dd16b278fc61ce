"""Which plan a multiexp runs by: whole scalars or split ones, and what is taken
when a width or a workspace cannot be had.  The sum is the same by every plan."""
import ctypes

import numpy as np
import pytest

from cusnarks_amd import _capi, inputs
from cusnarks_amd.device import DeviceBuffer
from cusnarks_amd.msm import fixed_base, msm_device

pytestmark = pytest.mark.gpu


def last_plan(ctx):
    """(window bits, windows, points) of the context's last multiexp"""
    plan = (ctypes.c_uint32 * 8)()
    _capi.check(_capi.lib().csk_last_msm_plan(ctx.ptr, plan, 8), "csk_last_msm_plan")
    return plan[0], plan[1], plan[6]


@pytest.mark.parametrize("n,windows", [(4194304, 9), (4500000, 17)])
def test_whole_scalars_of_large_multiexps(n, windows):
    # c = 15: 18 entries a point in halves, 17 whole, which 4.3 million points and
    # more take; the sum is the default width's
    ctx = _capi.default_context()
    pts, out, want = DeviceBuffer(ctx, n * 64), DeviceBuffer(ctx, 64), DeviceBuffer(ctx, 64)
    sc = DeviceBuffer.from_array(ctx, inputs.field_elements(921, n))
    fixed_base(sc, n, pts, ctx=ctx)
    msm_device(sc, pts, n, want, ctx=ctx)
    msm_device(sc, pts, n, out, ctx=ctx, window_bits=15)
    assert last_plan(ctx) == (15, windows, n)
    assert np.array_equal(out.download((16,)), want.download((16,)))


@pytest.mark.parametrize("lg,whole", [(18, 2531), (20, 1783), (22, 1483)])
def test_split_plans_workspace(lg, whole):
    # a proof's four G1 multiexps and the one on G2: points twice, on G2 up to four
    # times, but not much more workspace than whole scalars took, in bytes a point
    from cusnarks_amd.batch import MsmBatch
    from cusnarks_amd.tune import apply
    ctx, n = _capi.Context(0), 1 << lg
    apply(ctx)
    need = MsmBatch.workspace_bytes([n] * 4, ctx=ctx) + MsmBatch.workspace_bytes([n], g2=True, ctx=ctx)
    assert need < 1.04 * whole * n


@pytest.mark.parametrize("g2,n", [(False, 1), (False, 1 << 20), (True, 1 << 18), (True, 1 << 20)])
def test_workspace_limit(g2, n):
    # a context that the split plan does not fit in runs a plan that needs less;
    # below that the call is refused, the context stays usable and nothing lingers
    from cusnarks_amd.batch import MsmBatch
    from cusnarks_amd.tune import apply
    ctx, nw, L = _capi.Context(0), 32 if g2 else 16, _capi.lib()
    apply(ctx)
    limit = lambda b: _capi.check(L.csk_ctx_limit_workspace(ctx.ptr, int(b)), "limit")  # noqa: E731
    pts, out, want = DeviceBuffer(ctx, n * nw * 4), DeviceBuffer(ctx, nw * 4), DeviceBuffer(ctx, nw * 4)
    sc = DeviceBuffer.from_array(ctx, inputs.field_elements(922, n))
    fixed_base(sc, n, pts, g2=g2, ctx=ctx)
    msm_device(sc, pts, n, want, g2=g2, ctx=_capi.Context(0))
    expected = want.download((nw,))
    need = MsmBatch.workspace_bytes([n], g2=g2, ctx=ctx)
    least = MsmBatch.workspace_bytes([n], g2=g2, ctx=ctx, least_workspace=True)
    assert least <= need
    limit(least // 2)
    with pytest.raises(_capi.CskError):
        MsmBatch([n], g2=g2, ctx=ctx, shared_workspace=True)
    with pytest.raises(_capi.CskError):
        msm_device(sc, pts, n, out, g2=g2, ctx=ctx)
    limit(max(least, need - 1))
    b = MsmBatch([n], g2=g2, ctx=ctx, shared_workspace=True)
    assert least <= b.info()["bytes"] <= max(least, need - 1) + 4096
    b.run([sc], [pts], [out])
    assert np.array_equal(out.download((nw,)), expected)
    if g2 and n == 1 << 20:  # whole scalars need less at the tuned width
        msm_device(sc, pts, n, out, g2=g2, ctx=ctx)
        assert last_plan(ctx)[1] == 254 // last_plan(ctx)[0] + 1 and L.csk_last_error() == b""
        assert np.array_equal(out.download((nw,)), expected)
    limit(0)
    msm_device(sc, pts, n, out, g2=g2, ctx=ctx)
    assert np.array_equal(out.download((nw,)), expected)
    b2 = MsmBatch([n], g2=g2, ctx=ctx, least_workspace=True)
    b2.run([sc], [pts], [out], use_graph=False)
    assert np.array_equal(out.download((nw,)), expected)


def test_launches_after_an_allocation_that_failed():
    ctx = _capi.Context(0)
    sc = DeviceBuffer.from_array(ctx, inputs.field_elements(923, 100))
    pts, out = DeviceBuffer(ctx, 6400), DeviceBuffer(ctx, 64)
    fixed_base(sc, 100, pts, ctx=ctx)
    with pytest.raises(_capi.CskError):
        DeviceBuffer(ctx, 1 << 46)
    msm_device(sc, pts, 100, out, ctx=ctx)
    out.download((16,))


def test_batch_takes_the_sizes_of_single_calls():
    # two members of 2^27 points at a tuned width of 18: 15 windows fit the index
    # range, the 16 of the next narrower width do not
    from cusnarks_amd import tune
    from cusnarks_amd.batch import MsmBatch
    ctx = _capi.Context(0)
    tune.install(ctx, False, {"classes": {"27": {"window_bits": 18}}})
    one = MsmBatch.workspace_bytes([1 << 27], ctx=ctx)
    assert MsmBatch.workspace_bytes([1 << 27] * 2, ctx=ctx) == 2 * one


@pytest.mark.parametrize("g2,n,c", [(False, 50000, 7), (False, 50000, 9), (False, 70001, 14), (False, 300000, 18),
                                    (False, 30000, 17), (True, 30000, 8), (True, 30000, 14), (True, 5000, 2)])
def test_top_windows_whose_bins_are_buckets(g2, n, c):
    # the parts' bits leave the top window 0 to 7 bits: its entries, half of the
    # points' carries in one bucket for 0, are ordered by the sort's first pass
    ctx, nw = _capi.default_context(), 32 if g2 else 16
    pts, out, want = DeviceBuffer(ctx, n * nw * 4), DeviceBuffer(ctx, nw * 4), DeviceBuffer(ctx, nw * 4)
    k = inputs.field_elements(924, n)
    k[: n // 3, 2:] = 0
    sc = DeviceBuffer.from_array(ctx, k)
    fixed_base(DeviceBuffer.from_array(ctx, inputs.field_elements(925, n, nonzero=True)), n, pts, g2=g2, ctx=ctx)
    msm_device(sc, pts, n, want, g2=g2, ctx=ctx)
    msm_device(sc, pts, n, out, g2=g2, ctx=ctx, window_bits=c)
    assert np.array_equal(out.download((nw,)), want.download((nw,)))
