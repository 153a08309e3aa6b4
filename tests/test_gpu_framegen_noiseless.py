"""Generated frames without noise to speak of: an Eb/N0 that leaves sigma no
double gives infinite LLRs with the codeword's signs."""
import numpy as np
import pytest

from gf2_amd import codes
from gf2_amd.device import generate_frames, generate_zero_frames
from gf2_amd.ldpc import Context, LdpcCode
from tests import frames

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ebn0", [300.0, 3000.0, 3081.0, 3084.0, 1e5])
def test_noiseless_frames(ebn0):
    ctx, spec, F = Context(0), codes.n2304_r12(), 3
    code = LdpcCode(spec.qc(), ctx)
    print("[gpu-case] noiseless frames", ebn0, flush=True)
    d_llr, d_cw = generate_frames(code, 5, 0, F, ebn0, ebn0)
    llr = d_llr.download(np.float32, (F, spec.n))
    bits = frames.unpack_words(d_cw.download(np.uint64, (F, spec.n // 64)), spec.n)
    signs = 1.0 - 2.0 * bits.astype(np.float32)
    zero = generate_zero_frames(code, 5, 0, F, ebn0, ebn0).download(np.float32, (F, spec.n))
    if ebn0 < 380.0:  # 4 R Eb/N0, finite in float32 (4 R = 2)
        np.testing.assert_allclose(llr, signs * np.float32(2e30), rtol=1e-5)
        np.testing.assert_allclose(zero, np.full_like(zero, 2e30), rtol=1e-5)
    else:
        assert np.array_equal(llr, signs * np.inf) and np.array_equal(zero, np.full_like(zero, np.inf))
