"""Timed cases of the decoder: what programs that use this framework ask of it.

A receiver decodes frames as they arrive (one frame from host memory, through
the batch API or the SDR handle), a batch decoder works through LLRs resident
in HBM (plain min-sum BP, the layered learned decoder, DVB-T2 codes, mixed
codes, a code given as an edge list), and a training run generates frames and
takes gradients of the layered decoder.  Every kind of call is timed through
its public entry point: the C ABI of include/gf2ldpc.h on device buffers, the
Python mirror on host arrays.

A case is a dict of plain values:
  kind    "host" | "sdr" | "batch" | "learned" | "dvb" | "mixed" | "edges" |
          "gradient" | "generate"
  n, k    the quasi-cyclic code (gf2_amd.codes), or of the edge-list code
  frames  frames per call
  ebn0    Eb/N0 in dB (0 stands for error-free +-10 LLRs)
  short, rate   DVB-T2 frame size and rate index (kinds "sdr" and "dvb")

Inputs are random codewords sent as BPSK over AWGN, made with torch from the
seed alone.  Contexts, codes, decoder handles and learned weights are what a
program sets up once and keeps, so they are kept per process here too.
"""
from __future__ import annotations

import math
import os

import numpy as np
import torch

from gf2_amd import _lib, codes
from gf2_amd.dvb_bench import WATERFALL_DB
from gf2_amd.ldpc import CodeRate, LdpcCode, decode_batch_arrays, default_context
from gf2_amd.mixed import CodeSet
from gf2_amd.nms import NmsDecoder

MAX_IT = 50
WEIGHTS = os.path.join(os.path.dirname(os.path.abspath(codes.__file__)), "weights")
LAYERED = {(64800, 32400): "nms_n64800_layered_t10.npz", (2304, 1152): "nms_n2304_layered_t10.npz"}
# Eb/N0 where plain BP has a frame error rate of about 1e-2
WATERFALL = dict(codes.FER_1E2_EBN0)
WATERFALL[(2304, 1152)] = 1.9
QC = sorted(WATERFALL)


def listed():
    return [
        # the smallest call: one short frame from host memory, as LdpcDecoder.decode_iterative makes it
        {"name": "host-n2304-1", "kind": "host", "n": 2304, "k": 1152, "frames": 1, "ebn0": 2.0},
        # a software radio block: one DVB-T2 normal frame per call through the SDR handle
        {"name": "sdr-normal-1/2-1", "kind": "sdr", "short": False, "rate": 0, "frames": 1, "ebn0": 1.7},
        # a receiver with a few long frames in flight: latency of a small batch
        {"name": "batch-n64800-24", "kind": "batch", "n": 64800, "k": 32400, "frames": 24, "ebn0": 1.62},
        # bulk decoding of a short code
        {"name": "batch-n2304-16384", "kind": "batch", "n": 2304, "k": 1152, "frames": 16384, "ebn0": 2.0},
        # bulk decoding of the long code, bit-exact plain BP: the largest call
        {"name": "batch-n64800-4096", "kind": "batch", "n": 64800, "k": 32400, "frames": 4096, "ebn0": 1.62},
        # the same batch with the layered learned decoder (bench.py's headline)
        {"name": "learned-n64800-4096", "kind": "learned", "n": 64800, "k": 32400, "frames": 4096, "ebn0": 1.62},
        # the reference's own decode benchmark: 202 error-free DVB-T2 normal r3/5 frames
        {"name": "dvb-normal-3/5-202", "kind": "dvb", "short": False, "rate": 1, "frames": 202, "ebn0": 0.0},
        # DVB-T2 short frames at the waterfall
        {"name": "dvb-short-1/2-1000", "kind": "dvb", "short": True, "rate": 0, "frames": 1000, "ebn0": 1.5},
        # a stream of all twelve quasi-cyclic codes, one call per batch
        {"name": "mixed-2000", "kind": "mixed", "frames": 2000},
        # a general sparse code (no structure to use), a ragged batch
        {"name": "edges-n9000-500", "kind": "edges", "n": 9000, "k": 4500, "frames": 500, "ebn0": 2.2},
        # one training step's gradient of the layered decoder
        {"name": "gradient-n64800-256", "kind": "gradient", "n": 64800, "k": 32400, "frames": 256, "ebn0": 1.6},
        # frames for training and error-rate sweeps, generated on the device
        {"name": "generate-n64800-1000", "kind": "generate", "n": 64800, "k": 32400, "frames": 1000, "ebn0": 1.6},
    ]


def _spread(rng, lo, hi):
    """A size between lo and hi, spread over its logarithm, odd ones among them."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["host", "sdr", "batch", "batch", "batch", "learned", "dvb", "dvb", "mixed", "edges",
                       "gradient", "generate"])
    c = {"kind": kind}
    if kind in ("sdr", "dvb"):
        c["short"] = rng.random() < 0.5
        c["rate"] = rng.randrange(6)
        c["frames"] = _spread(rng, 1, 8) if kind == "sdr" else _spread(rng, 2, 1500)
        point = WATERFALL_DB[(0 if c["short"] else 1, c["rate"])]
        c["ebn0"] = 0.0 if rng.random() < 0.25 else round(point + rng.uniform(0.0, 0.6), 2)
        return c
    if kind == "mixed":
        c["frames"] = _spread(rng, 30, 3000)
        return c
    if kind == "edges":
        c["k"] = 2 * rng.randrange(500, 4000)
        c["n"] = 2 * c["k"]
        c["frames"] = _spread(rng, 1, 1000)
        c["ebn0"] = round(rng.uniform(2.1, 2.8), 2)
        return c
    if kind in ("learned", "gradient"):
        c["n"], c["k"] = rng.choice(sorted(LAYERED))
    else:
        c["n"], c["k"] = rng.choice(QC)
    most = {"host": 12, "batch": 3000, "learned": 4000, "gradient": 300, "generate": 1500}[kind]
    c["frames"] = _spread(rng, 1, most if c["n"] > 20000 else 4 * most)
    c["ebn0"] = round(WATERFALL[(c["n"], c["k"])] + rng.uniform(0.02, 0.6), 2)
    return c


# ---- what a program keeps ------------------------------------------------

_kept = {}


def _keep(key, make):
    if key not in _kept:
        _kept[key] = make()
    return _kept[key]


def _qc_spec(n, k):
    if (n, k) == (2304, 1152):
        return codes.n2304_r12()
    if (n, k) == (64800, 32400):
        return codes.n64800_r12()
    return next(s for s in codes.mixed_twelve() if (s.n, s.k) == (n, k))


def _qc(n, k):
    return _keep(("qc", n, k), lambda: LdpcCode(_qc_spec(n, k).qc(), default_context()))


def _learned(n, k):
    return _keep(("learned", n, k),
                 lambda: NmsDecoder.load(_qc(n, k), os.path.join(WEIGHTS, LAYERED[(n, k)])))


def _dvb(short, rate):
    make = LdpcCode.dvb_t2_short if short else LdpcCode.dvb_t2_normal
    return _keep(("dvb", short, rate), lambda: make(CodeRate(rate), default_context()))


def _edge_list(n, k):
    """A seeded random code with three checks per bit and rate 1/2."""
    rng = np.random.default_rng(n)
    m = n - k
    bits = np.repeat(np.arange(n), 3)
    checks = rng.permutation(np.repeat(np.arange(m), 3 * n // m))
    return np.unique(np.stack([checks, bits], axis=1), axis=0)


def _sdr(short, rate):
    make = _lib.load().gf2_ldpc_decoder_create
    return _keep(("sdr", short, rate), lambda: make(0 if short else 1, rate, MAX_IT))


# ---- inputs ----------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _encode_qc(n, k, frames, g):
    """Random codewords [frames, n] (uint8) of a staircase quasi-cyclic code."""
    spec = _qc_spec(n, k)
    base, z = _keep(("base", n, k), spec.base_matrix), spec.z
    kb = spec.nb - spec.mb
    u = torch.randint(0, 2, (frames, kb, z), generator=g, device="cuda", dtype=torch.uint8)
    out = torch.empty((frames, spec.nb, z), device="cuda", dtype=torch.uint8)
    out[:, :kb] = u
    p = torch.zeros((frames, z), device="cuda", dtype=torch.uint8)
    for br in range(spec.mb):
        for bc in range(kb):
            if base[br, bc] >= 0:
                p = p ^ torch.roll(u[:, bc], -int(base[br, bc]), dims=1)
        out[:, kb + br] = p
    return out.reshape(frames, n)


def _encode_dvb(short, rate, frames, g):
    """Random codewords of a DVB-T2 code (accumulator encoder)."""
    s = _keep(("dvb-table", short, rate), lambda: codes.dvb_t2(0 if short else 1, rate))
    u = torch.randint(0, 2, (frames, s.k), generator=g, device="cuda", dtype=torch.uint8)
    par = torch.zeros((frames, s.m // s.q, s.q), device="cuda", dtype=torch.uint8)
    for i, row in enumerate(s.table):
        block = u[:, i * s.z:(i + 1) * s.z]
        for a in row:  # bit j of the block meets check (a + j q) mod m
            par[:, :, a % s.q] ^= torch.roll(block, a // s.q, dims=1)
    par = (torch.cumsum(par.reshape(frames, s.m), dim=1, dtype=torch.int32) & 1).to(torch.uint8)
    return torch.cat([u, par], dim=1)


def _channel(bits, ebn0, rate, g):
    """BPSK over AWGN as channel LLRs; ebn0 0: error-free +-10."""
    x = 1.0 - 2.0 * bits.to(torch.float32)
    if not ebn0:
        return 10.0 * x
    s2 = 1.0 / (2.0 * rate * 10.0 ** (ebn0 / 10.0))
    noise = torch.randn(x.shape, generator=g, device="cuda", dtype=torch.float32)
    return ((x + math.sqrt(s2) * noise) * (2.0 / s2)).contiguous()


def _pack(bits):
    """[F, n] bits -> [F, ceil(n/64)] little-endian words."""
    F, n = bits.shape
    b = torch.nn.functional.pad(bits, (0, -n % 64)).reshape(F, -1, 64).to(torch.int64)
    return (b << torch.arange(64, device=bits.device)).sum(dim=2)


class _Buffer:
    """A device tensor where the Python API takes a device buffer."""

    def __init__(self, tensor):
        self.tensor, self.ptr = tensor, tensor.data_ptr()


def _outputs(frames, k):
    def make(shape, dtype):
        return torch.zeros(shape, device="cuda", dtype=dtype)
    return [make((frames, (k + 63) // 64), torch.int64), make(frames, torch.int32), make(frames, torch.uint8),
            make(frames, torch.uint8)]


# ---- the cases -------------------------------------------------------------

def prepare(case, seed):
    kind, frames = case["kind"], case.get("frames")
    g = _generator(seed)
    s = {"kind": kind, "frames": frames}
    if kind in ("host", "batch", "learned", "gradient"):
        n, k = case["n"], case["k"]
        bits = _encode_qc(n, k, frames, g)
        llr = _channel(bits, case["ebn0"], k / n, g)
        s["code"] = _qc(n, k)
        if kind == "host":
            s["llr"] = llr.cpu().numpy()
            return s
        s["llr"] = llr
        if kind == "gradient":
            s["words"] = _pack(bits)
            s["decoder"] = _learned(n, k)
            s["llr"], s["words"] = _Buffer(s["llr"]), _Buffer(s["words"])
            return s
        s["out"] = _outputs(frames, k)
        if kind == "learned":
            s["decoder"] = _learned(n, k)
            s["out"].append(torch.zeros(frames, device="cuda", dtype=torch.uint8))
    elif kind in ("sdr", "dvb"):
        bits = _encode_dvb(case["short"], case["rate"], frames, g)
        code = _dvb(case["short"], case["rate"])
        llr = _channel(bits, case["ebn0"], code.rate(), g)
        if kind == "sdr":
            s["llr"] = llr.cpu().numpy()
            s["handle"] = _sdr(case["short"], case["rate"])
            s["out"] = (np.zeros((frames, code.k()), dtype=np.uint8), np.zeros(frames, dtype=np.int32))
            return s
        s["code"], s["llr"], s["out"] = code, llr, _outputs(frames, code.k())
    elif kind == "edges":
        n, k = case["n"], case["k"]
        s["code"] = _keep(("edges", n, k), lambda: LdpcCode.from_edges(n - k, n, _edge_list(n, k), default_context()))
        # the zero codeword, as the reference's own error-rate example sends it
        s["llr"] = _channel(torch.zeros((frames, n), device="cuda", dtype=torch.uint8), case["ebn0"], k / n, g)
        s["out"] = _outputs(frames, k)
    elif kind == "mixed":
        specs = codes.mixed_twelve()
        s["set"] = _keep("mixed", lambda: CodeSet([_qc(x.n, x.k) for x in specs]))
        # equal shares in random order: the outputs' sizes do not depend on the seed
        ids = np.random.default_rng(seed).permutation(np.arange(frames) % len(specs)).astype(np.uint16)
        rows = [None] * frames
        for c, x in enumerate(specs):
            at = np.nonzero(ids == c)[0]
            if at.size:
                llr = _channel(_encode_qc(x.n, x.k, int(at.size), g), WATERFALL[(x.n, x.k)] + 0.05, x.k / x.n, g)
                for j, f in enumerate(at):
                    rows[f] = llr[j]
        s["ids"], s["llr"] = ids, torch.cat(rows)
        words = int(sum((specs[c].k + 63) // 64 for c in ids))
        s["out"] = [torch.zeros(words, device="cuda", dtype=torch.int64)] + _outputs(frames, 64)[1:]
    else:
        n, k = case["n"], case["k"]
        s["code"], s["seed"], s["ebn0"] = _qc(n, k), int(seed), case["ebn0"]
        s["out"] = [torch.zeros((frames, n), device="cuda", dtype=torch.float32),
                    torch.zeros((frames, (n + 63) // 64), device="cuda", dtype=torch.int64)]
    return s


def run(s):
    kind, lib = s["kind"], _lib.load()
    if kind == "host":
        msg, it, conv, synd = decode_batch_arrays(s["code"], s["llr"], MAX_IT)
        return msg.view(np.int64), it.view(np.int32), conv, synd
    if kind == "sdr":
        out, its = s["out"]
        rc = lib.gf2_ldpc_decode_frames(s["handle"], s["llr"].ctypes.data, s["frames"], out.ctypes.data,
                                        its.ctypes.data)
        if rc < 0:
            raise RuntimeError("gf2_ldpc_decode_frames")
        return out, its
    ctx = default_context()
    if kind in ("batch", "dvb", "edges"):
        _lib.check(ctx.handle, lib.gf2l_decode_batch_device(
            ctx.handle, s["code"].handle, s["llr"].data_ptr(), s["frames"], MAX_IT, *[o.data_ptr() for o in s["out"]]))
        return s["out"]
    if kind == "learned":
        s["decoder"].decode_device(_Buffer(s["llr"]), s["frames"], MAX_IT, *[_Buffer(o) for o in s["out"]])
        return s["out"]
    if kind == "mixed":
        s["set"].decode_device(s["ids"], s["llr"].data_ptr(), MAX_IT, *[o.data_ptr() for o in s["out"]])
        return s["out"]
    if kind == "gradient":
        return s["decoder"].gradient(s["llr"], s["words"], s["frames"])
    _lib.check(ctx.handle, lib.gf2l_frames_generate(
        ctx.handle, s["code"].handle, s["seed"], 0, s["frames"], s["ebn0"], s["ebn0"] + 0.4,
        s["out"][0].data_ptr(), s["out"][1].data_ptr()))
    return s["out"]


def work(case):
    """LLRs in and results out; per edge and iteration a subtraction, two
    comparisons, a sign, a selection and an addition (about 25 iterations of
    plain BP at the waterfall, 13 for the short code, 9 of the layered one)."""
    kind, frames = case["kind"], case.get("frames")
    if kind == "mixed":
        specs = codes.mixed_twelve()
        per = [(x.n, x.k, _edges(x)) for x in specs]
        n, k, e = (sum(p[i] for p in per) / len(per) for i in range(3))
        its = 20
    elif kind in ("sdr", "dvb"):
        s = codes.dvb_t2(0 if case["short"] else 1, case["rate"])
        n, k, e = s.n, s.k, 2 * s.m + 360 * sum(len(r) for r in s.table)
        its = 20 if case["ebn0"] else 1
    elif kind == "edges":
        n, k, e, its = case["n"], case["k"], 3 * case["n"], 20
    else:
        n, k = case["n"], case["k"]
        e = _edges(_qc_spec(n, k))
        its = {"learned": 9, "gradient": 30, "generate": 0}.get(kind, 13 if n == 2304 else 25)
    if kind == "generate":  # ten rounds of two 32-bit products and a Gaussian pair for every two LLRs
        return {"bytes": frames * (4 * n + n / 8), "flops": frames * n * 40.0}
    back = n / 8 if kind == "gradient" else k / 8 + 6
    return {"bytes": frames * (4.0 * n + back), "flops": 6.0 * e * its * frames}


def _edges(spec):
    return spec.z * (sum(spec.weights()) + 2 * spec.mb - 1)


# ---- the same in 64 bits ---------------------------------------------------

def exact(case, seed):
    if case["kind"] == "gradient":
        return _exact_gradient(case, seed)
    if case["kind"] == "generate":
        return _exact_frames(case, seed)
    return None  # every other kind returns bits, counts and flags


def _exact_gradient(case, seed):
    """Gradient and loss of the layered decoder by automatic differentiation
    in float64, a few frames at a time."""
    n, k, frames = case["n"], case["k"], case["frames"]
    spec = _qc_spec(n, k)
    base, z = spec.base_matrix(), spec.z
    g = _generator(seed)
    bits = _encode_qc(n, k, frames, g)
    llr = _channel(bits, case["ebn0"], k / n, g).double()
    y = 1.0 - 2.0 * bits.double()
    rows = [[(bc, int(base[br, bc])) for bc in range(spec.nb) if base[br, bc] >= 0] for br in range(spec.mb)]
    with np.load(os.path.join(WEIGHTS, LAYERED[(n, k)]), allow_pickle=False) as f:
        w = torch.tensor(f["weights"], dtype=torch.float64, device="cuda")
    T = w.shape[0]
    w = w.reshape(T, -1).requires_grad_()
    total = torch.zeros((), dtype=torch.float64, device="cuda")
    grad = torch.zeros_like(w)
    step = 64 if n > 20000 else 1024
    for a in range(0, frames, step):
        b = list(llr[a:a + step].reshape(-1, spec.nb, z).unbind(1))
        yy = y[a:a + step].reshape(-1, spec.nb, z)
        old = [None] * spec.mb
        loss = torch.zeros((), dtype=torch.float64, device="cuda")
        for t in range(T):
            e0 = 0
            for br, row in enumerate(rows):
                x = torch.stack([torch.roll(b[c], -s, dims=1) for c, s in row], dim=1)
                if old[br] is not None:
                    x = x - old[br]
                mag, at = torch.topk(x.abs(), 2, dim=1, largest=False)
                place = torch.arange(len(row), device="cuda").reshape(1, -1, 1)
                m = torch.where(place == at[:, :1], mag[:, 1:], mag[:, :1])
                sign = 1.0 - 2.0 * (x.detach() < 0).double()
                m = w[t, e0:e0 + len(row)].reshape(1, -1, 1) * m * sign * sign.prod(dim=1, keepdim=True)
                new = x + m
                for p, (c, s) in enumerate(row):
                    b[c] = torch.roll(new[:, p], s, dims=1)
                old[br] = m
                e0 += len(row)
            loss = loss + torch.nn.functional.softplus(-yy * torch.stack(b, dim=1)).sum()
        grad += torch.autograd.grad(loss, w)[0]
        total += loss.detach()
    scale = 1.0 / (T * n * frames)
    return (grad * scale).cpu().numpy(), float(total) * scale


def _philox(c0, c1, c2, c3, key):
    """Philox4x32-10 on int64 tensors holding 32-bit words: words 0 and 1."""
    low = 0xFFFFFFFF
    k0, k1 = key & low, (key >> 32) & low

    def mul(m, c):
        hi = (m * (c >> 16) + ((m * (c & 0xFFFF)) >> 16)) >> 16
        return hi & low, (m * c) & low

    for _ in range(10):
        h0, l0 = mul(0xD2511F53, c0)
        h1, l1 = mul(0xCD9E8D57, c2)
        c0, c1, c2, c3 = h1 ^ c1 ^ k0, l1, h0 ^ c3 ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & low, (k1 + 0xBB67AE85) & low
    return c0, c1


def _exact_frames(case, seed):
    """The generator's frames from its documented counters, in float64."""
    n, k, frames = case["n"], case["k"], case["frames"]
    spec = _qc_spec(n, k)
    base, z, kb = spec.base_matrix(), spec.z, spec.nb - spec.mb
    zw = (z + 63) // 64
    f = torch.arange(frames, device="cuda").reshape(-1, 1)
    zero = torch.zeros_like(f)

    def draw_words(count, stream):
        c = torch.arange(count, device="cuda").reshape(1, -1).expand(frames, -1)
        full = torch.zeros_like(c)
        return _philox(c, f + full, full, full + stream, int(seed))

    w0, w1 = draw_words(kb * zw, 0)
    word = torch.stack([w0, w1], dim=2).reshape(frames, kb, 2 * zw, 1)
    u = ((word >> torch.arange(32, device="cuda")) & 1).reshape(frames, kb, 64 * zw)[:, :, :z].to(torch.uint8)
    bits = torch.empty((frames, spec.nb, z), device="cuda", dtype=torch.uint8)
    bits[:, :kb] = u
    p = torch.zeros((frames, z), device="cuda", dtype=torch.uint8)
    for br in range(spec.mb):
        for bc in range(kb):
            if base[br, bc] >= 0:
                p = p ^ torch.roll(u[:, bc], -int(base[br, bc]), dims=1)
        bits[:, kb + br] = p
    bits = bits.reshape(frames, n)
    unit = 1.0 / 4294967296.0
    lo, hi = float(np.float32(case["ebn0"])), float(np.float32(case["ebn0"] + 0.4))
    e0, _ = _philox(zero, f, zero, zero + 2, int(seed))
    ebn0 = lo + (hi - lo) * ((e0.double() + 0.5) * unit)
    s2 = 1.0 / (2.0 * (k / n) * 10.0 ** (ebn0 / 10.0))
    pairs = (n + 1) // 2
    w0, w1 = draw_words(pairs, 1)
    r = torch.sqrt(-2.0 * torch.log((w0.double() + 0.5) * unit))
    th = 2.0 * math.pi * ((w1.double() + 0.5) * unit)
    noise = torch.stack([r * torch.cos(th), r * torch.sin(th)], dim=2).reshape(frames, -1)[:, :n]
    llr = 2.0 * ((1.0 - 2.0 * bits.double()) + torch.sqrt(s2) * noise) / s2
    return [llr, None]
