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


def test_launches_after_an_allocation_that_failed():
    ctx = _capi.Context(0)
    sc = DeviceBuffer.from_array(ctx, inputs.field_elements(923, 100))
    pts, out = DeviceBuffer(ctx, 6400), DeviceBuffer(ctx, 64)
    fixed_base(sc, 100, pts, ctx=ctx)
    with pytest.raises(_capi.CskError):
        DeviceBuffer(ctx, 1 << 46)
    msm_device(sc, pts, 100, out, ctx=ctx)
    out.download((16,))
