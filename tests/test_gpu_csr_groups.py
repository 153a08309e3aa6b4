"""General sparse codes decoded 64 frames interleaved, against the oracle and
against the frame-contiguous kernels: batch sizes around the group of 64, the
round of eight groups and the pass of several groups, and batches whose frames
stop at different iterations (running frames are packed into fewer groups)."""
import numpy as np
import pytest

from gf2_amd import _lib
from gf2_amd.ldpc import Context, LdpcCode, decode_batch_arrays
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


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


def mixed_llrs(rng, frames, n):
    """Zero codeword in noise from light to hopeless, zeros of both signs,
    infinities and NaN in some frames."""
    sigma = rng.choice([0.5, 0.75, 0.8, 1.5], size=(frames, 1), p=[0.5, 0.2, 0.2, 0.1])
    llr = ((1.0 + sigma * rng.normal(size=(frames, n))) * 2.0 / sigma**2).astype(np.float32)
    llr[rng.random(llr.shape) < 0.002] = -0.0
    llr[rng.random(llr.shape) < 0.002] = 0.0
    llr[0, :3] = [np.inf, -np.inf, 1e38]
    if frames > 2:
        llr[2, 5] = np.nan
    return llr


# n, checks, ones per variable: check degrees to 8, 16 and 30; a k that is no
# multiple of 64; more checks than variables of a wave's share
@pytest.mark.parametrize("n,m,weight", [(130, 65, 3), (1000, 500, 3), (500, 100, 3), (300, 40, 4)])
def test_batch_sizes_match_oracle(ctx, n, m, weight):
    rng = np.random.default_rng(n)
    edges = edge_list(rng, n, m, weight)
    code, oc = LdpcCode.from_edges(m, n, edges, ctx), orc.Code(m, n, edges)
    llr = mixed_llrs(rng, 650, n)
    for frames, max_it in ((1, 30), (1, 1), (63, 30), (64, 4), (65, 5), (130, 30), (512, 30), (650, 30), (650, 2)):
        print("[gpu-case] csr groups", n, m, weight, frames, max_it, flush=True)
        got = decode(ctx, code, llr[:frames], max_it)
        same(got, oc.decode_batch(llr[:frames], max_it, threads=8), (n, frames, max_it))
        same(got, decode(ctx, code, llr[:frames], max_it, 1), (n, frames, max_it, "contiguous"))


def test_several_passes(ctx):
    n, m = 100000, 300
    rng = np.random.default_rng(3)
    bits = rng.choice(n, 3000, replace=False)
    edges = np.stack([np.repeat(np.arange(m), 10), bits], axis=1)
    code = LdpcCode.from_edges(m, n, edges, ctx)
    llr = np.tile(mixed_llrs(rng, 60, n), (72, 1))  # 4320 frames of 100,000 LLRs: two passes
    print("[gpu-case] csr groups passes", llr.shape, flush=True)
    got = decode(ctx, code, llr, 6)
    same([x[:60] for x in got], orc.Code(m, n, edges).decode_batch(llr[:60], 6, threads=8), "first")
    same(got, [np.tile(np.asarray(x)[:60], (72,) + (1,) * (np.asarray(x).ndim - 1)) for x in got], "repeated")
