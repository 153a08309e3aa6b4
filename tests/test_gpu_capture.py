"""Recorded decodes of a small code: replays that run beside each other and
beside the context's own decodes each decode all of their frames."""
import ctypes

import numpy as np
import pytest

from gf2_amd import _lib, codes
from gf2_amd.device import DeviceBuffer, generate_frames
from gf2_amd.ldpc import Context, LdpcCode

pytestmark = pytest.mark.gpu

RELAXED = 2  # hipStreamCaptureModeRelaxed
F, MAX_IT = 6000, 30  # more frames than workgroups, of different lengths


def test_overlapping_replays():
    ctx, lib = Context(0), _lib.load()
    vp = ctypes.c_void_p

    def hip(name, *args):
        assert getattr(lib, name)(*args) == 0, name

    code = LdpcCode(codes.n2304_r12().qc(), ctx)
    kw = (code.k() + 63) // 64
    shapes = [(np.uint64, (F, kw)), (np.uint32, F), (np.uint8, F), (np.uint8, F)]
    llr, want, outs = [], [], []

    def decode(j):
        _lib.check(ctx.handle, lib.gf2l_decode_batch_device(ctx.handle, code.handle, llr[j].ptr, F, MAX_IT,
                                                            *[b.ptr for b in outs[j]]))

    for j in range(3):
        llr.append(generate_frames(code, 70 + j, 0, F, 1.4, 2.4, with_codewords=False)[0])
        outs.append([DeviceBuffer.from_array(ctx, np.zeros(shape, dtype)) for dtype, shape in shapes])
        decode(j)
        ctx.synchronize()
        want.append([b.download(*s) for b, s in zip(outs[j], shapes)])
        assert want[j][2].any() and not want[j][2].all()
    stream = vp(lib.gf2l_stream(ctx.handle))
    execs, streams = [], []
    for j in range(2):
        graph, ex, own = vp(), vp(), vp()
        hip("hipStreamBeginCapture", stream, RELAXED)
        decode(j)
        hip("hipStreamEndCapture", stream, ctypes.byref(graph))
        hip("hipGraphInstantiate", ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0))
        hip("hipGraphDestroy", graph)
        hip("hipStreamCreate", ctypes.byref(own))
        execs.append(ex)
        streams.append(own)
    for turn in range(4):
        print("[gpu-case] overlapping replays", turn, flush=True)
        for j in range(3):
            for b, (dtype, shape) in zip(outs[j], shapes):
                b.upload(np.zeros(shape, dtype))
        for ex, own in zip(execs, streams):
            hip("hipGraphLaunch", ex, own)
        decode(2)
        for own in streams:
            hip("hipStreamSynchronize", own)
        ctx.synchronize()
        for j in range(3):
            for b, s, w in zip(outs[j], shapes, want[j]):
                assert np.array_equal(b.download(*s), w), (turn, j)
    for ex, own in zip(execs, streams):
        hip("hipGraphExecDestroy", ex)
        hip("hipStreamDestroy", own)
