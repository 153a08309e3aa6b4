"""Gradient of the layered decoder by the staircase kernels against the general
layered kernels, which the double-precision oracle checks."""
import numpy as np
import pytest

from gf2_amd import _lib
from gf2_amd.device import generate_frames
from gf2_amd.ldpc import Context, LdpcCode, QuasiCyclicLdpc, qc_ira_base_matrix
from gf2_amd.nms import NmsDecoder

pytestmark = pytest.mark.gpu

# (mb, nb, z, information column weights): both row degrees, both numbers of
# layers ahead (mb a multiple of 6, or of 10 only), whole and ragged waves, one
# wave, the largest lift
SHAPES = {"degree-6-by-6": (12, 24, 96, [6] * 4 + [3] * 8), "degree-6-by-5": (20, 40, 100, [4] * 20),
          "degree-7-by-5": (20, 40, 333, [5] * 20), "degree-7-by-6-one-wave": (18, 36, 64, [5] * 18),
          "largest-lift": (18, 30, 512, [8] * 6 + [7] * 6)}


@pytest.fixture(scope="module")
def ctx():
    return Context(0)


@pytest.mark.parametrize("frames", [1, 300])
@pytest.mark.parametrize("shape", SHAPES)
def test_staircase_gradient_equals_general(ctx, shape, frames):
    mb, nb, z, weights = SHAPES[shape]
    code = LdpcCode(QuasiCyclicLdpc(qc_ira_base_matrix(5, mb, nb, z, weights), z), ctx)
    T = 3 if frames > 1 else 1
    rng = np.random.default_rng(8)
    nbe = len(code.qc.to_edges()) // z
    w = rng.uniform(0.5, 1.1, size=(T, nbe)).astype(np.float32)
    dec = NmsDecoder(code, T, w, schedule="layered")
    d_llr, d_cw = generate_frames(code, 9, 0, frames, 1.0, 3.0)
    out = {}
    for kernel in (_lib.LAYERED_GENERAL, _lib.LAYERED_STAIRCASE):
        print("[gpu-case] layered gradient", shape, frames, kernel, flush=True)
        ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, kernel)
        try:
            if kernel == _lib.LAYERED_STAIRCASE:
                assert dec.layered_columns == nb - mb  # the structure is there
            out[kernel] = dec.gradient(d_llr, d_cw, frames)
            again = dec.gradient(d_llr, d_cw, frames)
        finally:
            ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, _lib.LAYERED_AUTO)
        assert np.array_equal(out[kernel][0], again[0]) and out[kernel][1] == again[1]
    # The forward passes are the same operations, so the subgradients take the
    # same branches: what differs is the rounding of sums of up to 512 lanes and
    # of the derivative (log2(512) + a few steps of 6e-8, times the ratio of
    # the terms' magnitudes to their sum, below 100 here)
    (ga, la), (gb, lb) = out[_lib.LAYERED_GENERAL], out[_lib.LAYERED_STAIRCASE]
    assert np.linalg.norm(ga - gb) <= 1e-4 * np.linalg.norm(ga)
    assert abs(la - lb) <= 1e-5 * abs(la)
