"""Device memory that a decode of a long general sparse code takes: the arrays of
the frames, in groups of 64 from three frames on, and no second set of them where
groups cannot be packed."""
import ctypes

import numpy as np
import pytest

from gf2_amd import _lib
from gf2_amd.device import DeviceBuffer
from gf2_amd.ldpc import Context, LdpcCode
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def free_bytes(ctx):
    ctx.synchronize()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _lib.load().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("frames,copies", [(1, 1), (2, 2), (3, 64), (64, 64), (130, 256)])
def test_workspace_of_a_long_code(frames, copies):
    orc.build()
    ctx, n, m, weight = Context(0), 120000, 40000, 3
    rng = np.random.default_rng(7)
    checks = rng.permutation(np.repeat(np.arange(m), weight * n // m))
    edges = np.unique(np.stack([checks, np.repeat(np.arange(n), weight)], axis=1), axis=0)
    code = LdpcCode.from_edges(m, n, edges, ctx)
    llr = ((1.0 + 0.4 * rng.standard_normal((frames, n))) * 12.5).astype(np.float32)
    kw = (code.k() + 63) // 64
    bufs = [DeviceBuffer.from_array(ctx, llr)] + [DeviceBuffer(ctx, b) for b in (8 * frames * kw, 4 * frames, frames,
                                                                                 frames)]
    before = free_bytes(ctx)
    print("[gpu-case] csr memory", frames, flush=True)
    _lib.check(ctx.handle, _lib.load().gf2l_decode_batch_device(ctx.handle, code.handle, bufs[0].ptr, frames, 12,
                                                                *[b.ptr for b in bufs[1:]]))
    taken = before - free_bytes(ctx)
    # messages, beliefs, LLRs and hard decisions (at most two bits a variable and
    # frame), 16 MiB for counters, lists and the allocator's pages
    assert taken <= copies * (4 * len(edges) + 8 * n + n // 4) + (16 << 20), taken
    msg, its, conv, ok = orc.Code(m, n, edges).decode_batch(llr[:2], 12, threads=2)
    assert np.array_equal(bufs[1].download(np.uint64, (frames, kw))[:2], msg)
    assert np.array_equal(bufs[2].download(np.uint32, frames)[:2], its)
