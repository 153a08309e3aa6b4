"""Teams of workgroups per frame against the oracle and the general kernels:
team sizes from one workgroup to the most, several frames per team, ragged
lifts, DVB codes, and the way back to the general kernels."""
import numpy as np
import pytest

from gf2_amd import _lib, codes
from gf2_amd.ldpc import CodeRate, Context, LdpcCode, QuasiCyclicLdpc, decode_batch_arrays, qc_ira_base_matrix
from oracle import oracle as orc
from tests import frames

pytestmark = pytest.mark.gpu

GENERAL, TEAM, TEAM_NO_WAIT = 1, 3, 4

# (mb, nb, z, information column weights, Eb/N0)
SHAPES = {
    "one-wave-rows": (24, 60, 64, [3] * 36, 3.0),
    "ragged-lift": (9, 60, 200, [3] * 51, 4.0),
    "lift-not-a-multiple-of-32": (6, 40, 401, [3] * 34, 4.0),
    "degree-27-checks": (4, 104, 360, [1] * 100, 6.0),
    "degree-16-columns": (20, 60, 360, [16] * 2 + [3] * 38, 3.0),
}


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


def with_odd_values(llr, seed):
    """Zeros of both signs everywhere; infinities, NaN and a hopeless frame."""
    rng = np.random.default_rng(seed)
    llr[rng.random(llr.shape) < 0.002] = -0.0
    llr[rng.random(llr.shape) < 0.002] = 0.0
    if len(llr) > 3:
        llr[1, :3] = [np.inf, -np.inf, 1e38]
        llr[2, 7] = np.nan
    llr[-1] = rng.normal(0, 1, llr.shape[1]).astype(np.float32)
    return llr


@pytest.mark.parametrize("shape", SHAPES)
def test_quasi_cyclic_codes(ctx, shape):
    mb, nb, z, weights, ebn0 = SHAPES[shape]
    base = qc_ira_base_matrix(5, mb, nb, z, weights)
    code = LdpcCode(QuasiCyclicLdpc(base, z), ctx)
    oc = orc.Code.from_qc(base, z)
    _, _, llr = frames.random_frames(base, z, 12, ebn0, seed=21)
    llr = with_odd_values(llr, 22)
    for count, max_it in ((1, 20), (12, 1), (12, 2), (12, 20)):
        print("[gpu-case] team", shape, count, max_it, flush=True)
        got = decode(ctx, code, llr[-count:], max_it, TEAM)
        same(got, oc.decode_batch(llr[-count:], max_it, threads=8), (shape, count, max_it))
    many = np.tile(llr, (50, 1))  # 600 frames: teams of one take several
    print("[gpu-case] team", shape, "600", flush=True)
    same(decode(ctx, code, many, 8, TEAM), decode(ctx, code, many, 8, GENERAL), (shape, 600))


@pytest.mark.parametrize("short,rate,counts", [(True, 0, (1, 9, 300)), (True, 5, (1, 300)), (False, 0, (1, 60, 100)),
                                               (False, 3, (1, 100, 300)), (False, 5, (2, 130))])
def test_dvb_codes(ctx, short, rate, counts):
    make = LdpcCode.dvb_t2_short if short else LdpcCode.dvb_t2_normal
    code = make(CodeRate(rate), ctx)
    s = codes.dvb_t2(0 if short else 1, rate)
    oc = orc.Code(s.m, s.n, orc.dvb_edges(s.table, s.n, s.k, s.q))
    rng = np.random.default_rng(31)
    sigma = 0.45 if rate else 0.75
    llr = (2.0 / sigma**2 * (1.0 + sigma * rng.normal(size=(max(counts), s.n)))).astype(np.float32)
    llr[4::3] = 10.0  # frames that stop after one iteration
    llr = with_odd_values(llr, 32)
    want = oc.decode_batch(llr[:4], 12, threads=8)
    for count in counts:
        for mode in (0, TEAM, TEAM_NO_WAIT):
            print("[gpu-case] team dvb", short, rate, count, mode, flush=True)
            got = decode(ctx, code, llr[:count], 12, mode)
            same(got, decode(ctx, code, llr[:count], 12, GENERAL), (short, rate, count, mode))
        same([x[:4] for x in got], [x[:count] for x in want], (short, rate, count, "oracle"))


def test_default_route_of_small_batches(ctx):
    spec = codes.n64800_r12()
    base = spec.base_matrix()
    code = LdpcCode(spec.qc(), ctx)
    _, _, llr = frames.random_frames(base, spec.z, 8, 1.65, seed=41)
    print("[gpu-case] team default", flush=True)
    got = decode(ctx, code, llr, 50, 0)
    same(got, decode(ctx, code, llr, 50, GENERAL), "default")
    same(got, decode(ctx, code, llr, 50, TEAM), "team")
    same(got, decode(ctx, code, llr, 50, TEAM_NO_WAIT), "no wait")
