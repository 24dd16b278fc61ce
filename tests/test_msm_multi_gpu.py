"""csk_msm_multi: several multiexps in one call equal the single calls, bit for
bit: members of one width and of several, more than a group holds, empty ones
and members that overlap in scalars and points."""
import ctypes

import numpy as np
import pytest

from cusnarks_amd import _capi, inputs
from cusnarks_amd.device import DeviceBuffer, Stream
from cusnarks_amd.msm import fixed_base, msm_device, msm_multi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g2", [False, True])
@pytest.mark.parametrize("sizes", [
    [1], [4, 1], [0, 5, 0, 7], [300, 4096, 4097, 2048, 2047],  # several widths
    [50] * 17,                                                 # three groups
    [9000, 12000, 8192, 16383],                                # a prover's four of one width
])
def test_multi_equals_single_calls(g2, sizes):
    ctx = _capi.default_context()
    nw, n = 32 if g2 else 16, max(sizes) + 8
    pts = DeviceBuffer(ctx, n * nw * 4)
    fixed_base(DeviceBuffer.from_array(ctx, inputs.field_elements(71, n, nonzero=True)), n, pts, g2=g2)
    k = inputs.field_elements(72, n)
    k[: n // 2, 1:] = 0
    sc = DeviceBuffer.from_array(ctx, k)
    outs, want = (DeviceBuffer(ctx, len(sizes) * nw * 4) for _ in range(2))
    members = [(sc.ptr + (i % 8) * 32, pts.ptr + (i % 3) * nw * 4, m, outs.ptr + i * nw * 4) for i, m in enumerate(sizes)]
    msm_multi(members, g2=g2)
    for i, (s, p, m, _) in enumerate(members):
        msm_device(s, p, m, want.ptr + i * nw * 4, g2=g2)
    shape = (len(sizes), nw)
    assert np.array_equal(outs.download(shape), want.download(shape))


def test_refused():
    ctx, L = _capi.default_context(), _capi.lib()
    none = (ctypes.c_void_p * 65)()
    n = (ctypes.c_uint64 * 65)(*[1] * 65)
    p, q = ctypes.cast(none, _capi.P), ctypes.cast(n, _capi.P)
    for count in (0, 1, 65):  # no member, null members, too many
        assert L.csk_msm_multi(ctx.ptr, 0, count, p, p, q, p, None) != 0


def _members(ctx, g2, sizes):
    nw, n = 32 if g2 else 16, max(sizes)
    pts, outs = DeviceBuffer(ctx, n * nw * 4), DeviceBuffer(ctx, len(sizes) * nw * 4)
    sc = DeviceBuffer.from_array(ctx, inputs.field_elements(73, n, nonzero=True))
    fixed_base(sc, n, pts, g2=g2, ctx=ctx)
    keep = (sc, pts, outs)
    return keep, [(sc.ptr, pts.ptr, m, outs.ptr + i * nw * 4) for i, m in enumerate(sizes)]


@pytest.mark.parametrize("g2", [False, True])
def test_empty_members_do_not_wait(g2):
    # a call with empty members is enqueued like any other: it can be captured, and
    # every replay writes all outputs
    hip = ctypes.CDLL("libamdhip64.so")
    ctx, sizes = _capi.Context(0), [0, 300, 0, 5000, 200]
    keep, members = _members(ctx, g2, sizes)
    outs, shape = keep[2], (len(sizes), 32 if g2 else 16)
    msm_multi(members, g2=g2, ctx=ctx)  # grows the workspace
    want = outs.download(shape)
    zero = np.zeros(shape, np.uint32)
    st, graph, ex = Stream(ctx), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(st.ptr, 1) == 0
    msm_multi(members, g2=g2, ctx=ctx, stream=st.ptr)
    assert hip.hipStreamEndCapture(st.ptr, ctypes.byref(graph)) == 0
    assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, 0) == 0
    for _ in range(3):
        outs.upload(zero)
        assert hip.hipGraphLaunch(ex, st.ptr) == 0
        _capi.check(_capi.lib().csk_stream_sync(ctx.ptr, st.ptr), "sync")
        assert np.array_equal(outs.download(shape), want)
    hip.hipGraphExecDestroy(ex)
    hip.hipGraphDestroy(graph)


@pytest.mark.parametrize("bad", [0, 1, 3])
def test_refused_before_anything_is_enqueued(bad):
    ctx, sizes = _capi.Context(0), [300, 400, 30000]
    keep, members = _members(ctx, False, sizes)
    mark = np.full((3, 16), 7, np.uint32)
    keep[2].upload(mark)
    last = list(members[2])
    last[bad] = 0
    with pytest.raises(_capi.CskError):
        msm_multi(members[:2] + [tuple(last)], ctx=ctx)
    last = members[2][:2] + ((1 << 31),) + members[2][3:]  # more entries than an index holds
    with pytest.raises(_capi.CskError):
        msm_multi(members[:2] + [last], ctx=ctx)
    _capi.check(_capi.lib().csk_stream_sync(ctx.ptr, None), "sync")
    assert np.array_equal(keep[2].download((3, 16)), mark)


def test_group_that_does_not_fit_runs_member_by_member():
    ctx, sizes = _capi.Context(0), [40000] * 8
    keep, members = _members(ctx, False, sizes)
    msm_multi(members, ctx=_capi.Context(0))
    want = keep[2].download((8, 16))
    keep[2].upload(np.zeros((8, 16), np.uint32))
    L = _capi.lib()
    _capi.check(L.csk_ctx_limit_workspace(ctx.ptr, 60 << 20), "limit")
    msm_multi(members, ctx=ctx)
    assert L.csk_last_error() == b""
    assert np.array_equal(keep[2].download((8, 16)), want)
