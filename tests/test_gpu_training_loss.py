"""Training loss of confident outputs: every output's share counts, however far
below one it is."""
import numpy as np
import pytest

from gf2_amd import _lib
from gf2_amd.device import DeviceBuffer
from gf2_amd.ldpc import Context, LdpcCode, QuasiCyclicLdpc, qc_ira_base_matrix
from gf2_amd.nms import NmsDecoder
from oracle import oracle as orc
from tests import frames

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    orc.build()
    return Context(0)


# Eb/N0 in dB: soft outputs around 10, 30, 70
@pytest.mark.parametrize("ebn0", [4.0, 9.0, 13.0])
@pytest.mark.parametrize("kernel", [_lib.LAYERED_GENERAL, _lib.LAYERED_STAIRCASE])
def test_loss_of_confident_outputs(ctx, kernel, ebn0):
    mb, nb, z, T, F = 12, 24, 96, 10, 3
    base = qc_ira_base_matrix(5, mb, nb, z, [6] * 4 + [3] * 8)
    code = LdpcCode(QuasiCyclicLdpc(base, z), ctx)
    nbe = int((base >= 0).sum())
    w = np.random.default_rng(6).uniform(0.6, 1.0, size=(T, nbe)).astype(np.float32)
    dec = NmsDecoder(code, T, w, schedule="layered")
    _, bits, llr = frames.random_frames(base, z, F, ebn0, seed=9)
    words = np.zeros((F, nb * z // 64), dtype=np.uint64)
    for f in range(F):
        words[f] = np.packbits(bits[f].astype(np.uint8), bitorder="little").view(np.uint64)
    d_llr, d_cw = DeviceBuffer(ctx, llr.nbytes), DeviceBuffer(ctx, words.nbytes)
    d_llr.upload(llr)
    d_cw.upload(words)
    want = np.mean([orc.layered_loss_grad(base, z, llr[f], bits[f], w.astype(np.float64))[0] for f in range(F)])
    print("[gpu-case] training loss", kernel, ebn0, want, flush=True)
    ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, kernel)
    try:
        _, loss = dec.gradient(d_llr, d_cw, F)
    finally:
        ctx.set_tuning(_lib.TUNE_LAYERED_KERNEL, _lib.LAYERED_AUTO)
    # The outputs that make up the loss are below 55; ten layered iterations leave
    # them a few 1e-6 of themselves off (float32, some 30 additions), which an
    # exponential turns into 55 times that of its value.  The sum adds 1e-6.
    assert abs(loss - want) <= 2e-4 * abs(want), (loss, want)
