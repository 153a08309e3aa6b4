"""The default route of codes that may run in teams of workgroups: batches below
and above the number of teams, with full and with nearly empty last turns, of
quasi-cyclic codes without a staircase and of DVB codes in noise and in a quiet
channel, against the general kernels and the oracle."""
import numpy as np
import pytest

from gf2_amd import _lib, codes
from gf2_amd.ldpc import CodeRate, Context, LdpcCode, QuasiCyclicLdpc, decode_batch_arrays
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

GENERAL, TEAM_NO_WAIT = 1, 4


@pytest.fixture(scope="module")
def ctx():
    orc.build()
    return Context(0)


def decode(ctx, code, llr, max_it, mode):
    ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, mode)
    try:
        return decode_batch_arrays(code, llr, max_it)
    finally:
        ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, 0)


def same(a, b, what):
    for name, x, y in zip(["msg", "iterations", "converged", "syndrome_ok"], a, b):
        assert np.array_equal(x, y), f"{what}: {name} differs at {np.nonzero(np.asarray(x) != y)[0][:8]}"


def zero_codeword_llrs(rng, frames, n, sigma):
    s = np.broadcast_to(np.asarray(sigma, dtype=np.float64).reshape(-1, 1), (frames, 1))
    return ((1.0 + s * rng.standard_normal((frames, n))) * 2.0 / s**2).astype(np.float32)


def base_without_staircase(seed, mb, nb, z, weight):
    rng = np.random.default_rng(seed)
    base = np.full((mb, nb), -1, dtype=np.int32)
    order = rng.permutation(np.tile(np.arange(mb), weight * nb // mb + 1))[:weight * nb].reshape(nb, weight)
    for c in range(nb):
        for r in order[c]:
            base[r, c] = rng.integers(0, z)
    return base


# (mb, nb, z): teams of two, 128 at a time, and one workgroup a frame
@pytest.mark.parametrize("mb,nb,z,counts", [(40, 80, 400, (12, 140, 250)), (120, 240, 100, (12, 140, 250)),
                                            (240, 480, 48, (12, 140)), (24, 48, 500, (1, 300))])
def test_codes_without_staircase(ctx, mb, nb, z, counts):
    base = base_without_staircase(3, mb, nb, z, 3)
    code, oc = LdpcCode(QuasiCyclicLdpc(base, z), ctx), orc.Code.from_qc(base, z)
    assert ctx.code_path(code) == _lib.PATH_STATE
    rng = np.random.default_rng(4)
    llr = zero_codeword_llrs(rng, max(counts), nb * z, rng.choice([0.4, 0.7, 0.76, 1.0], max(counts)))
    want = oc.decode_batch(llr[:12], 15, threads=8)
    for count in counts:
        print("[gpu-case] team route", mb, nb, z, count, flush=True)
        got = decode(ctx, code, llr[:count], 15, 0)
        same(got, decode(ctx, code, llr[:count], 15, GENERAL), (z, count))
        same([x[:12] for x in got], [x[:count] for x in want], (z, count, "oracle"))


# teams of three (85 at a time) and two (128 at a time); checks up to 8, 16 and 27
@pytest.mark.parametrize("rate,counts", [(0, (86, 128, 520)), (2, (129, 200)), (4, (250,))])
@pytest.mark.parametrize("quiet", [0.0, 0.1, 0.4])  # share of frames that one iteration decodes
def test_dvb_batches_of_several_turns(ctx, rate, counts, quiet):
    code, s = LdpcCode.dvb_t2_normal(CodeRate(rate), ctx), codes.dvb_t2(1, rate)
    oc = orc.Code(s.m, s.n, orc.dvb_edges(s.table, s.n, s.k, s.q))
    rng = np.random.default_rng(5)
    noisy = zero_codeword_llrs(rng, 40, s.n, {0: 0.75, 2: 0.6, 4: 0.53}[rate])
    llr = noisy[rng.integers(0, 40, max(counts))]
    llr[rng.random(max(counts)) < quiet] = 10.0
    llr[rng.random(llr.shape) < 0.001] = -0.0
    llr[1, :3], llr[2, 7] = [np.inf, -np.inf, 1e38], np.nan
    for max_it in (2, 12):
        want = oc.decode_batch(llr[:4], max_it, threads=8)
        for count in counts:
            for mode in (0, TEAM_NO_WAIT):  # with and without teams that leave after the first iteration
                print("[gpu-case] team turns", rate, count, quiet, max_it, mode, flush=True)
                got = decode(ctx, code, llr[:count], max_it, mode)
                same(got, decode(ctx, code, llr[:count], max_it, GENERAL), (rate, count, quiet, max_it, mode))
                same([x[:4] for x in got], want, (rate, count, quiet, max_it, mode, "oracle"))


# rows of 1 to 25 information inputs: mostly padding in the whole-frame kernel
@pytest.mark.parametrize("mb,kb,z,counts", [(40, 60, 128, (1, 70, 300)), (60, 120, 360, (1, 86, 200))])
def test_staircase_codes_of_uneven_rows(ctx, mb, kb, z, counts):
    rng = np.random.default_rng(6)
    base = np.full((mb, kb + mb), -1, dtype=np.int32)
    for r in range(mb):
        for c in rng.choice(kb, 25 if r % 10 == 3 else 1 + r % 4, replace=False):
            base[r, c] = rng.integers(0, z)
        base[r, kb + r] = 0
        if r:
            base[r, kb + r - 1] = 0
    n = (kb + mb) * z
    code, oc = LdpcCode(QuasiCyclicLdpc(base, z), ctx), orc.Code.from_qc(base, z)
    llr = zero_codeword_llrs(rng, max(counts), n, rng.choice([0.3, 0.5, 0.9], max(counts)))
    want = oc.decode_batch(llr[:8], 15, threads=8)
    for count in counts:
        print("[gpu-case] uneven rows", z, count, flush=True)
        got = decode(ctx, code, llr[:count], 15, 0)
        same(got, decode(ctx, code, llr[:count], 15, GENERAL), (z, count))
        same([x[:8] for x in got], [x[:count] for x in want], (z, count, "oracle"))
