"""NaN LLRs of either sign bit, and NaN from infinite ones, in the layered
learned decoder: both kernels count a NaN input of a check as the comparisons of
the oracle's rule do."""
import numpy as np
import pytest

from gf2_amd import _lib, codes
from gf2_amd.ldpc import Context, LdpcCode
from gf2_amd.nms import NmsDecoder
from oracle import oracle as orc
from tests import frames

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    orc.build()
    return Context(0)


@pytest.mark.parametrize("kernel", [_lib.LAYERED_GENERAL, _lib.LAYERED_STAIRCASE])
@pytest.mark.parametrize("fb_it", [0, 10])
@pytest.mark.parametrize("which", ["n2304", "n64800"])
def test_nan_llrs(ctx, which, kernel, fb_it):
    spec = codes.n2304_r12() if which == "n2304" else codes.n64800_r12()
    base = spec.base_matrix()
    nbe = int((base >= 0).sum())
    _, _, llr = frames.random_frames(base, spec.z, 14, 3.0, seed=61)
    rng = np.random.default_rng(62)
    bits = llr.view(np.uint32)
    for f in range(10):  # a handful to a hundredth of the LLRs, positive, negative or both
        at = rng.choice(spec.n, 4 if f < 6 else spec.n // 100, replace=False)
        bits[f, at] = 0x7FC00000
        if f % 3:
            bits[f, at[::f % 3]] = 0xFFC00000
    llr[10] *= np.inf  # every LLR infinite, wrong ones among them: infinite minus infinite
    llr[11, rng.random(spec.n) < 0.7] *= np.inf
    w = rng.uniform(0.6, 1.0, size=(4, nbe)).astype(np.float32)
    dec = NmsDecoder(LdpcCode(spec.qc(), ctx), 4, weights=w, schedule="layered")
    print("[gpu-case] layered nan", which, kernel, flush=True)
    ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, kernel)
    try:
        got = dec.decode(llr, fallback_max_it=fb_it)
    finally:
        ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, _lib.LAYERED_AUTO)
    want = orc.layered_decode_batch(base, spec.z, llr, w, fb_it)
    for name, x, y in zip(["msg", "iterations", "converged", "syndrome_ok", "fallback"], got, want):
        assert np.array_equal(x, y), f"{name} differs at {np.nonzero(np.asarray(x) != np.asarray(y))[0][:8]}"
