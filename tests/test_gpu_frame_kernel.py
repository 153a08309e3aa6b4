"""The whole-frame flooding kernel against the oracle: one workgroup per frame
on staircase quasi-cyclic codes, bit-exact, over the shapes where its row
tables, wave layout and LDS split differ."""
import numpy as np
import pytest

from gf2_amd import _lib, codes
from gf2_amd.ldpc import Context, LdpcCode, QuasiCyclicLdpc, decode_batch_arrays, qc_ira_base_matrix
from gf2_amd.mixed import CodeSet, decode_mixed_arrays
from oracle import oracle as orc
from tests import frames

pytestmark = pytest.mark.gpu

# (mb, nb, z, information column weights, Eb/N0)
SHAPES = {
    "two-rows-one-wave": (2, 5, 64, [2, 2, 1], 4.0),
    "odd-rows-ragged-lift": (3, 9, 100, [3, 3, 2, 2, 2, 1], 4.0),
    "short-lift-96": (12, 24, 96, [6] * 4 + [3] * 8, 2.2),
    "largest-lift": (7, 20, 384, [4] * 5 + [3] * 8, 3.0),
    "few-heavy-columns": (10, 14, 320, [10, 9, 5, 2], 2.0),
    "degree-25-columns-past-lds": (5, 120, 360, [1] * 115, 6.0),
    "columns-past-lds": (40, 160, 360, [7] * 30 + [3] * 90, 3.0),
    "lift-above-the-kernel": (6, 15, 400, [3] * 9, 3.0),  # runs the general kernels
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


@pytest.mark.parametrize("shape", SHAPES)
def test_matches_oracle(ctx, shape):
    mb, nb, z, weights, ebn0 = SHAPES[shape]
    base = qc_ira_base_matrix(5, mb, nb, z, weights)
    code = LdpcCode(QuasiCyclicLdpc(base, z), ctx)
    oc = orc.Code.from_qc(base, z)
    F = 6 if nb * z > 30000 else 37
    _, _, llr = frames.random_frames(base, z, F, ebn0, seed=11)
    rng = np.random.default_rng(12)
    llr[rng.random(llr.shape) < 0.002] = -0.0
    llr[rng.random(llr.shape) < 0.002] = 0.0
    llr[-1] = rng.normal(0, 1, llr.shape[1]).astype(np.float32)  # no codeword near: runs every iteration
    for count, max_it in ((1, 20), (F, 1), (F, 2), (F, 20)):
        print("[gpu-case] frame kernel", shape, count, max_it, flush=True)
        same(decode(ctx, code, llr[:count], max_it, 2), oc.decode_batch(llr[:count], max_it, threads=8),
             f"{shape} {count}x{max_it}")


def random_base(mb, nb, z, degree, seed):
    """Any base matrix: rows of up to `degree` circulants, no structure."""
    rng = np.random.default_rng(seed)
    base = -np.ones((mb, nb), dtype=np.int32)
    for r in range(mb):
        cols = rng.choice(nb, size=int(rng.integers(2, degree + 1)), replace=False)
        base[r, cols] = rng.integers(0, z, size=cols.size)
    return base


# (mb, nb, z, largest row degree): one check, checks and variables that fill
# no wave, a whole wave, both degree classes, columns without a check, the
# largest workgroups
SMALL = {"one-check": (1, 3, 1, 3), "under-a-wave": (4, 9, 7, 6), "one-wave": (3, 6, 64, 5),
         "degree-8": (9, 18, 65, 8), "many-columns": (6, 40, 50, 8), "n2304": (12, 24, 96, 6),
         "ten-waves": (16, 32, 120, 6), "fourteen-waves": (26, 52, 100, 3)}


@pytest.mark.parametrize("shape", SMALL)
def test_small_codes_match_oracle(ctx, shape):
    mb, nb, z, degree = SMALL[shape]
    base = random_base(mb, nb, z, degree, 21)
    code = LdpcCode(QuasiCyclicLdpc(base, z), ctx)
    assert ctx.code_path(code) == _lib.PATH_LDS
    oc = orc.Code.from_qc(base, z)
    rng = np.random.default_rng(22)
    llr = rng.normal(1.0, 1.4, size=(41, nb * z)).astype(np.float32)  # the zero codeword, noisy
    llr[rng.random(llr.shape) < 0.01] = -0.0
    llr[rng.random(llr.shape) < 0.01] = 0.0
    for count, max_it in ((1, 30), (41, 1), (41, 30)):
        print("[gpu-case] small-code kernel", shape, count, max_it, flush=True)
        same(decode(ctx, code, llr[:count], max_it, 0), oc.decode_batch(llr[:count], max_it, threads=8),
             f"{shape} {count}x{max_it}")


def test_small_codes_many_frames_and_special_llrs(ctx):
    """More frames than workgroups, twice (the frame counter starts over), with
    infinite, NaN and very large LLRs in some frames: as the general kernel."""
    spec = codes.n2304_r12()
    base = spec.base_matrix()
    code = LdpcCode(QuasiCyclicLdpc(base, spec.z), ctx)
    _, _, llr = frames.random_frames(base, spec.z, 300, 2.0, seed=6)
    rng = np.random.default_rng(7)
    for f, v in ((1, np.inf), (4, -np.inf), (7, np.nan), (9, 2e30), (10, -3.3e38), (12, -np.nan)):
        llr[f, rng.integers(0, spec.n, 9)] = v
    llr[11] *= np.float32(1e28)  # beliefs pass the limit while it iterates
    llr = np.tile(llr, (9, 1))
    print("[gpu-case] small-code kernel, 2700 frames", flush=True)
    ref = decode(ctx, code, llr, 50, 1)
    for _ in range(2):
        same(decode(ctx, code, llr, 50, 0), ref, "small")


@pytest.mark.parametrize("special", [False, True])
def test_mixed_codes(ctx, special):
    """Frames of codes of different length, row degree and LDS split in one
    call; with a NaN and an infinite LLR the call is left to the general
    kernels."""
    shapes = [(25, 45, 360, [8] * 5 + [3] * 15), (8, 45, 360, [8] + [3] * 36), (5, 120, 360, [1] * 115),
              (12, 30, 330, [5] * 18)]
    bases = [qc_ira_base_matrix(7 + i, mb, nb, z, w) for i, (mb, nb, z, w) in enumerate(shapes)]
    gcodes = [LdpcCode(QuasiCyclicLdpc(b, s[2]), ctx) for b, s in zip(bases, shapes)]
    ids = np.random.default_rng(2).permutation(np.arange(22) % 4).astype(np.uint16)
    rows = [frames.random_frames(bases[c], shapes[c][2], 1, (2.6, 3.3, 6.0, 3.0)[c], seed=50 + f)[2][0]
            for f, c in enumerate(ids)]
    if special:
        rows[3][5], rows[9][100:103] = np.nan, np.inf
    cs = CodeSet(gcodes)
    out = {}
    for mode in (1, 2):
        print("[gpu-case] frame kernel, mixed codes", special, mode, flush=True)
        ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, mode)
        try:
            out[mode] = decode_mixed_arrays(cs, ids, np.concatenate(rows), 30)
        finally:
            ctx.set_tuning(_lib.TUNE_FRAME_KERNEL, 0)
    for a, b in zip(out[1], out[2]):
        assert np.array_equal(a, b)
    msg, off, it, conv, synd, _ = out[2]
    for f, c in enumerate(ids):
        if np.isfinite(rows[f]).all():
            ref = orc.Code.from_qc(bases[c], shapes[c][2]).decode_batch(rows[f][None], 30)
            same([msg[off[f]:off[f + 1]][None], it[f:f + 1], conv[f:f + 1], synd[f:f + 1]], ref, f"frame {f}")


def test_more_frames_than_workgroups(ctx):
    """Frames are drawn from a counter: each workgroup decodes several."""
    spec = codes.QcIraSpec(16200, 7200, 360)
    base = spec.base_matrix()
    code = LdpcCode(QuasiCyclicLdpc(base, spec.z), ctx)
    _, _, llr = frames.random_frames(base, spec.z, 24, 2.6, seed=3)
    print("[gpu-case] frame kernel, 1200 frames", flush=True)
    ref = orc.Code.from_qc(base, spec.z).decode_batch(llr, 50, threads=8)
    got = decode(ctx, code, np.tile(llr, (50, 1)), 50, 0)
    same(got, [np.tile(r, (50, 1)) if r.ndim == 2 else np.tile(r, 50) for r in ref], "tiled")


def test_frames_it_leaves_to_the_general_kernels(ctx):
    """Infinite, NaN and very large LLRs: those frames come out as the general
    kernels decode them, the others as ever."""
    spec = codes.QcIraSpec(16200, 7200, 360)
    base = spec.base_matrix()
    code = LdpcCode(QuasiCyclicLdpc(base, spec.z), ctx)
    _, _, llr = frames.random_frames(base, spec.z, 12, 2.4, seed=4)
    rng = np.random.default_rng(5)
    for f, v in ((1, np.inf), (4, -np.inf), (7, np.nan), (9, 2e30), (10, -3.3e38)):
        llr[f, rng.integers(0, spec.n, 9)] = v
    llr[11] *= np.float32(1e28)  # beliefs pass the limit while it iterates
    print("[gpu-case] frame kernel, special LLRs", flush=True)
    got = decode(ctx, code, llr, 50, 2)
    same(got, decode(ctx, code, llr, 50, 1), "special")
    finite = [f for f in range(12) if np.isfinite(llr[f]).all()]
    ref = orc.Code.from_qc(base, spec.z).decode_batch(llr[finite], 50, threads=8)
    same([r[finite] for r in got], ref, "finite")
