"""Short general sparse codes: several groups of frames beside each other on an
XCD, groups packed by many waves, and the early question after the first
iteration, against the oracle and the frame-contiguous kernels."""
import numpy as np
import pytest

from gf2_amd import _lib
from gf2_amd.ldpc import Context, LdpcCode, decode_batch_arrays
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

HAMMING = np.argwhere(np.array([[1, 0, 1, 0, 1, 0, 1], [0, 1, 1, 0, 0, 1, 1], [0, 0, 0, 1, 1, 1, 1]]))


@pytest.fixture(scope="module")
def ctx():
    orc.build()
    return Context(0)


def decode(ctx, code, llr, max_it, mode=0):
    ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, mode)
    try:
        return decode_batch_arrays(code, llr, max_it)
    finally:
        ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, 0)


def same(a, b, what):
    for name, x, y in zip(["msg", "iterations", "converged", "syndrome_ok"], a, b):
        assert np.array_equal(x, y), f"{what}: {name} differs at {np.nonzero(np.asarray(x) != y)[0][:8]}"


def edge_list(rng, n, m, weight):
    checks = rng.permutation(np.repeat(np.arange(m), -(-weight * n // m)))[:weight * n]
    return np.unique(np.stack([checks, np.repeat(np.arange(n), weight)], axis=1), axis=0)


# frames: whole rounds of eight groups and groups left over, more groups than one
# wave of the packing holds
@pytest.mark.parametrize("n,m,counts", [(7, 3, (1, 2, 5000, 150001)), (64, 32, (3, 511, 40000)),
                                        (300, 150, (1, 448, 512, 12345)), (1100, 500, (2, 3000))])
def test_short_codes(ctx, n, m, counts):
    rng = np.random.default_rng(n)
    edges = HAMMING if n == 7 else edge_list(rng, n, m, 3)
    code, oc = LdpcCode.from_edges(m, n, edges, ctx), orc.Code(m, n, edges)
    frames = max(counts)
    sigma = rng.choice([0.3, 0.7, 0.8, 1.2], size=(frames, 1), p=[0.6, 0.2, 0.1, 0.1])
    llr = ((1.0 + sigma * rng.standard_normal((frames, n))) * 2.0 / sigma**2).astype(np.float32)
    want = oc.decode_batch(llr[:600], 25, threads=8)
    for count in counts:
        for max_it in (25, 2, 1):
            print("[gpu-case] csr short codes", n, count, max_it, flush=True)
            got = decode(ctx, code, llr[:count], max_it)
            same(got, decode(ctx, code, llr[:count], max_it, 1), (n, count, max_it, "contiguous"))
            if max_it == 25:
                same([x[:600] for x in got], [x[:count] for x in want], (n, count, "oracle"))
