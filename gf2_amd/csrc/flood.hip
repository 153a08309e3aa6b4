// Whole-frame flooding min-sum decoder for staircase quasi-cyclic codes: one
// workgroup decodes a frame from its LLRs to its bits in one launch, with the
// same operations in the same order as the STATE path (bit-exact with
// decode_iterative, crates/gf2-coding/src/ldpc/core.rs:889-938).
//
// A belief is L + the messages of its checks in ascending block-row order, so
// it can be accumulated while the block-rows are processed in that order: the
// variable update needs no pass of its own, and a check's compressed state is
// read and written once per iteration instead of once per edge.  Per frame
// and iteration:
//   - the accumulators of the information block-columns (beliefs being formed)
//     live in LDS; the beliefs of the iteration before are read from the
//     workgroup's scratch rows (L2), the channel LLRs in iteration 1;
//   - parity block-column j only meets block-rows j and j+1 with shift 0, so
//     its belief is private to one lane: L + its message from block-row j is
//     handed to block-row j+1 through an LDS slot;
//   - the check states (12 bytes) stay in the workgroup's scratch rows.
// Two groups of ceil(z/64) waves take the even and the odd block-rows.  A row
// is computed (loads one row of the group ahead, check rule) at any time, but
// its messages are added only after those of every earlier row: `done` counts
// the waves that have added, in row order, and a wave of row r waits for
// r * waves of them.  Row r waits only for rows below r and every wave of a
// workgroup is resident, so each wait ends.
//
// Scratch is per workgroup, not per frame: 256 workgroups of the N=64800 code
// use 170 MB, which stays in the 256 MB last-level cache.
//
// What bounds it (N=64800 r1/2, 4096 frames at 1.62 dB, 101,500
// frame-iterations): memory behind L2.  A frame-iteration moves 1.83 MB (states
// 0.78, LLRs 0.26, parity beliefs 0.26, information beliefs 0.13 written and
// 0.40 read: L2 holds part of them between their reads) at 6.9 TB/s: 0.266 us.
// The batch takes 27.0 ms; the check and variable kernels it replaces took
// 57.8 ms (0.57 us per frame-iteration).  A workgroup alone on the chip needs
// 53 us per iteration.  Measured and left out: streaming (non-temporal) marks
// on the states and LLRs, 34.1 ms: rows are not whole cache lines, and the
// parts of a line shared by two waves were fetched and written twice.
//
// Arithmetic.  With sign-carrying magnitudes (m1, m2 with the product of all
// input signs on their sign bit) the message to position p is the selected
// magnitude with p's own input sign flipped in: one three-input bit operation.
// The selection compares |x_p| with the minimum: where several inputs tie,
// m2 = m1 and the choice does not matter.  Signs of zeros differ from the
// general kernels' rule only where a magnitude is zero; a zero's sign reaches
// no sum's value, no magnitude and no `< 0` test, so bits, iteration counts
// and flags are the same.  An infinity or a NaN would not be: a frame with an
// LLR or a belief of magnitude 1e30 or more (or NaN) is put on a list instead,
// and the general kernels decode it from its LLRs.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "device_common.h"
#include "gf2ldpc.h"

namespace gf2l {
namespace {

constexpr uint32_t kFloodGroups = 2;
constexpr uint32_t kFloodThreads = 768;  // two groups of up to 384 lanes
constexpr float kFloodLimit = 1e30f;
// Information inputs per row of the instantiations.  Each runs rows of its number
// and of one less without guards (rows of a balanced code differ by one); a code
// between two of them runs the larger one, padded.
#define GF2L_FLOOD_DEGREES                                                                              \
    GF2L_FLOOD(4) GF2L_FLOOD(5) GF2L_FLOOD(6) GF2L_FLOOD(8) GF2L_FLOOD(9) GF2L_FLOOD(10) GF2L_FLOOD(11) \
    GF2L_FLOOD(13) GF2L_FLOOD(15) GF2L_FLOOD(17) GF2L_FLOOD(21) GF2L_FLOOD(25)

__device__ __forceinline__ bool too_large(float v) { return !(fabsf(v) < kFloodLimit); }

// Waits until `target` row parts have been added (see the file comment).
__device__ __forceinline__ void wait_rows(const lds_u32 *done, uint32_t target) {
    while (uni(*(const volatile lds_u32 *)done) < target) {
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// What one lane of a block-row reads, loaded a row ahead.
// Rows of many inputs compute the offsets twice instead of keeping them over
// the wait: they would not fit the 168 vector registers of three waves per
// SIMD.
constexpr int kFloodKeep = 11;
template <int ND>
struct FloodIn {
    uint32_t ad[ND <= kFloodKeep ? ND : 1];  // byte offset of each information input in a [columns][z] array
    uint32_t po, so;  // byte offsets of parity column r-1 in a [nb][z] array and of the state
    float b[ND];      // beliefs (LLRs in iteration 1)
    float bp, bo;     // beliefs of parity columns r-1 and r
    float lp;         // LLR of parity column r
    uint3 st;
};

// Arrays of one frame, all uniform: 32-bit byte offsets from them take the
// scalar-base addressing form.
struct FloodBase {
    const float *info;  // [kb][z] beliefs of the information columns (the LLRs in iteration 1)
    const float *par;   // [nb][z], parity columns only (likewise)
    const float *llr;   // [nb][z]
};

// Offsets of the first NI information inputs of block-row r at lane i.
template <int ND, int NI>
__device__ __forceinline__ void flood_offsets(const FloodPlan &pl, uint32_t r, uint32_t i, uint32_t z4, uint32_t *ad) {
#pragma unroll
    for (int p = 0; p < NI; ++p) {
        const uint2 t = ldc(pl.edge + r * ND + p);
        ad[p] = 4u * i + t.x - (i >= t.y ? z4 : 0u);
    }
}

template <int ND>
__device__ __forceinline__ void flood_load(const FloodPlan &pl, FloodIn<ND> &in, uint32_t r, uint32_t i, uint32_t kb,
                                           uint32_t z, const FloodBase &B, const uint3 *st) {
    const uint32_t i4 = 4u * i, z4 = 4u * z;
    uint32_t ad[ND];
    flood_offsets<ND, ND>(pl, r, i, z4, ad);
    in.po = i4 + uni((kb + r - 1u) * z4);
    in.so = 12u * i + uni(3u * (r * z4));
    in.st = ldb(st, in.so);
#pragma unroll
    for (int p = 0; p < ND; ++p) {
        in.b[p] = ldb(B.info, ad[p]);
        if constexpr (ND <= kFloodKeep) in.ad[p] = ad[p];
    }
    in.bp = ldb(B.par, in.po);
    in.bo = ldb(B.par, in.po + z4);
    in.lp = ldb(B.llr, in.po + z4);
}

// Check update: c[0..NI-1] messages to the information inputs, cp and co to
// parity columns r-1 and r, and the new state {m1, m2, argmin | input signs <<
// 5} (inputs in the order own, previous, information; the last one's sign at
// bit 5).  GENERAL: only the first ninfo information inputs exist and the
// previous parity column only with has_prev; a missing input counts as
// +infinity, which changes nothing for the rest.
template <int ND, int NI, bool GENERAL>
__device__ __forceinline__ uint3 flood_check(const FloodIn<ND> &in, uint32_t ninfo, bool has_prev, bool first,
                                             float *c, float &cp, float &co) {
    constexpr int D = NI + 2;
    // iteration 1: old messages -0, so that x = b - (-0) = b + 0 (b exactly, -0 as +0)
    const float m1o = first ? -0.0f : __uint_as_float(in.st.x), m2o = first ? -0.0f : __uint_as_float(in.st.y);
    const uint32_t mo = first ? 0u : in.st.z, io = mo & 31u;
    float x[D];
#pragma unroll
    for (int p = 0; p < D; ++p) {
        const float mag = (uint32_t)p == io ? m2o : m1o;
        const uint32_t old = __float_as_uint(mag) ^ ((mo << (26 - (D - 1 - p))) & 0x80000000u);
        x[p] = (p == 0 ? in.bo : p == 1 ? in.bp : in.b[p >= 2 ? p - 2 : 0]) - __uint_as_float(old);
        if constexpr (GENERAL) {
            if (p == 1 ? !has_prev : p >= 2 && p - 2 >= (int)ninfo) x[p] = __builtin_inff();
        }
    }
    float m1 = __builtin_fminf(fabsf(x[0]), fabsf(x[1])), m2 = __builtin_fmaxf(fabsf(x[0]), fabsf(x[1]));
#pragma unroll
    for (int p = 2; p < D; ++p) {
        const float a = fabsf(x[p]);
        m2 = __builtin_amdgcn_fmed3f(m1, a, m2);
        m1 = __builtin_fminf(m1, a);
    }
    uint32_t sg = 0;
#pragma unroll
    for (int p = 0; p < D; ++p) sg = __builtin_amdgcn_alignbit(sg, __float_as_uint(x[p]), 31);
    const uint32_t all = (uint32_t)__popc(sg) << 31;
    const float m1s = __uint_as_float(__float_as_uint(m1) ^ all), m2s = __uint_as_float(__float_as_uint(m2) ^ all);
    uint32_t idx = 0;
#pragma unroll
    for (int p = 0; p < D; ++p) {
        const bool is1 = fabsf(x[p]) == m1;
        idx = is1 ? (uint32_t)p : idx;
        const uint32_t v = __float_as_uint(is1 ? m2s : m1s) ^ (__float_as_uint(x[p]) & 0x80000000u);
        (p == 0 ? co : p == 1 ? cp : c[p >= 2 ? p - 2 : 0]) = __uint_as_float(v);
    }
    return make_uint3(__float_as_uint(m1s), __float_as_uint(m2s), idx | (sg << 5));
}

// LDS of one workgroup.
struct FloodLds {
    lds_float *acc;      // [X][z] beliefs being formed
    lds_float *carry;    // [4][lanes] L + message of the row above, parity columns; one unused row
    lds_u64 *hb;         // [nb][zw] hard decisions
    lds_u32 *chk;        // nbe: hard-decision word of the block-column | shift << 16
    lds_u32 *rp;         // mb + 1
    uint32_t unused;     // this lane's byte offset of the unused row from acc
    lds_u32 *done, *bad; // rows added (waves); per wave: unsatisfied | too large << 1
};

struct FloodFrame {
    const CodeView &cv;
    const FloodPlan &pl;
    const FloodLds &S;
    const float *llr;
    uint3 *st;    // [mb][z]
    float *info;  // [kb][z]
    float *par;   // [nb][z]: parity columns; column kb-1 takes block-row 0's store and is never read
    uint32_t g, lane, wave, i, nw, kb;
    bool act;
    uint64_t lanes;  // the wave's lanes below z
};

template <typename T>
__device__ __forceinline__ void stb(T *base, uint32_t off, T v) {
    *reinterpret_cast<T *>(reinterpret_cast<char *>(base) + off) = v;
}

// Adds a row's messages to the accumulators.  Read, add and write: an LDS
// float atomic (ds_add_f32) would need no order within the row, but measured
// three times slower for the whole kernel (96 ms against 30 ms per 4096-frame
// batch of the N=64800 code).
template <int NI, bool GUARD>
__device__ __forceinline__ void flood_add(lds_float *acc, const uint32_t *ad, const float *c, uint32_t nlds) {
    auto at = [&](int p) { return (lds_float *)((__attribute__((address_space(3))) char *)acc + ad[p]); };
    float v[NI];
#pragma unroll
    for (int p = 0; p < NI; ++p)
        if (!GUARD || p < (int)nlds) v[p] = *at(p);
#pragma unroll
    for (int p = 0; p < NI; ++p)
        if (!GUARD || p < (int)nlds) *at(p) = v[p] + c[p];
}

// Hard-decision word of a column from its final beliefs (one per lane);
// returns the lanes whose belief is too large.
__device__ __forceinline__ uint64_t flood_word(const FloodFrame &F, uint32_t c, float b) {
    const uint64_t m = __builtin_amdgcn_ballot_w64(b < 0.0f) & F.lanes;
    if (F.lane == 0) F.S.hb[c * F.cv.zw + F.wave] = m;
    return __builtin_amdgcn_ballot_w64(too_large(b)) & F.lanes;
}

// One block-row of the group: check update, then the ordered part.  Returns
// the lanes with a belief too large.
template <int ND, int NI, bool GENERAL, bool EXTRA>
__device__ __forceinline__ uint64_t flood_row(const FloodFrame &F, const FloodIn<ND> &in, uint32_t r, uint32_t ninfo,
                                              uint32_t nlds, bool first) {
    const CodeView &cv = F.cv;
    float c[ND], cp, co;
    uint3 ns = flood_check<ND, NI, GENERAL>(in, ninfo, r > 0, first, c, cp, co);
    float own = in.lp + co;
    uint32_t ad[NI];
    if constexpr (ND <= kFloodKeep) {
#pragma unroll
        for (int p = 0; p < NI; ++p) ad[p] = in.ad[p];
    } else {
        flood_offsets<ND, NI>(F.pl, r, F.i, 4u * cv.z, ad);
    }
    // everything above is computed before the wait: left to itself the
    // compiler moves it behind, into the part that the rows run one by one
#pragma unroll
    for (int p = 0; p < NI; ++p) __asm__ volatile("" : "+v"(c[p]));
    __asm__ volatile("" : "+v"(cp), "+v"(own), "+v"(ns.x), "+v"(ns.y), "+v"(ns.z));
    const uint32_t lanes = F.nw * 64u;
    lds_float *slot = F.S.carry + (r & 3u) * lanes + F.i;
    const lds_float *above = F.S.carry + ((r + 3u) & 3u) * lanes + F.i;
    wait_rows(F.S.done, r * F.nw);
    float prev = 0.0f;
    if (F.act) {
        prev = *above;
        if constexpr (GENERAL) {
            flood_add<NI, true>(F.S.acc, ad, c, nlds);
        } else {
            // messages to columns past the LDS go to an unused row: a select
            // each, where a branch each split the row's reads and writes
            if constexpr (EXTRA) {
#pragma unroll
                for (int p = 0; p < NI; ++p) ad[p] = p < (int)nlds ? ad[p] : F.S.unused;
            }
            flood_add<NI, false>(F.S.acc, ad, c, nlds);
        }
        *slot = own;
    }
    // a wave's LDS operations complete in order: the count lands after the adds
    if (F.lane == 0)
        __asm__ volatile("ds_add_u32 %0, %1" ::"v"((uint32_t)(size_t)F.S.done), "v"(1u) : "memory");
    const float fin = prev + cp;  // parity column r-1, final (row 0: column kb-1's unused slot)
    const uint32_t col = F.kb + r - 1u;
    uint64_t big = 0;
    if (F.act) {
        stb(F.par, in.po, fin);
        stb(F.st, in.so, ns);
    }
    if (!GENERAL || r > 0) big = flood_word(F, col, fin);
    if (r + 1 == cv.mb) {
        big |= flood_word(F, col + 1u, own);
        if (F.act) stb(F.par, in.po + 4u * cv.z, own);
    }
    return big;
}

// Block-rows with ND or ND - 1 information inputs (all but one or two rows of
// the codes here) run code of their exact degree; the others, and block-row
// 0, the guarded form.  The row word's third byte is the degree whose state
// layout the row uses.
template <int ND, bool EXTRA>
__device__ __forceinline__ uint64_t flood_row(const FloodFrame &F, const FloodIn<ND> &in, uint32_t r, bool first) {
    const uint32_t rw = uni(ldc(F.pl.row + r));
    const uint32_t ninfo = rw & 0xffu, nlds = (rw >> 8) & 0xffu;
    if (r > 0 && ninfo == (uint32_t)ND - 1u) return flood_row<ND, ND - 1, false, EXTRA>(F, in, r, ninfo, nlds, first);
    if (r > 0 && ninfo == (uint32_t)ND) return flood_row<ND, ND, false, EXTRA>(F, in, r, ninfo, nlds, first);
    return flood_row<ND, ND, true, EXTRA>(F, in, r, ninfo, nlds, first);
}

// Unsatisfied checks over the hard-decision words (this thread's share).
__device__ __forceinline__ bool flood_unsat(const CodeView &cv, const FloodLds &S) {
    const uint32_t z = cv.z, zw = cv.zw;
    uint64_t bad = 0;
    for (uint32_t u = threadIdx.x; u < cv.mb * zw; u += blockDim.x) {
        const uint32_t br = u / zw, w = u - br * zw;
        uint64_t acc = 0;
        for (uint32_t e = S.rp[br]; e < S.rp[br + 1]; ++e) {
            const uint32_t r = S.chk[e];
            acc ^= cyc64_lds(S.hb + (r & 0xffffu), z, zw, wrap_add(64u * w, r >> 16, z));
        }
        if (w == zw - 1 && (z & 63u)) acc &= (1ull << (z & 63u)) - 1;
        bad |= acc;
    }
    return bad != 0;
}

// Combines the flags over the workgroup (uniform result).
__device__ __forceinline__ uint32_t flood_flags(const FloodLds &S, bool unsat, uint64_t big) {
    const uint64_t u = __builtin_amdgcn_ballot_w64(unsat);
    if ((threadIdx.x & 63u) == 0) S.bad[threadIdx.x >> 6] = (u != 0 ? 1u : 0u) | (big != 0 ? 2u : 0u);
    __syncthreads();
    uint32_t r = 0;
    for (uint32_t w = 0; w < blockDim.x / 64u; ++w) r |= S.bad[w];
    return uni(r);
}

// Columns that did not fit the LDS: c, c + 2, ... (kFloodCols of them), from
// the new states of their checks, four states of each column in flight.
constexpr uint32_t kFloodCols = 3;
__device__ __forceinline__ uint64_t flood_columns(const FloodFrame &F, uint32_t c0) {
    const uint32_t z = F.cv.z;
    float v[kFloodCols];
    uint32_t q0[kFloodCols], q1[kFloodCols], most = 0;
#pragma unroll
    for (uint32_t k = 0; k < kFloodCols; ++k) {
        const uint32_t c = min(c0 + k * kFloodGroups, F.kb - 1u);
        v[k] = ldu(F.llr + c * z, F.i);
        q0[k] = uni(ldc(F.pl.xptr + (c - F.pl.X)));
        q1[k] = uni(ldc(F.pl.xptr + (c - F.pl.X) + 1));
        most = max(most, q1[k] - q0[k]);
    }
    for (uint32_t d = 0; d < most; d += 4) {
        uint3 s[kFloodCols][4];
        uint32_t w[kFloodCols][4];
#pragma unroll
        for (uint32_t k = 0; k < kFloodCols; ++k)
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {  // (lists are followed by four words of padding)
                const uint2 t = ldc(F.pl.xedge + q0[k] + min(d, q1[k] - q0[k]) + j);
                w[k][j] = t.y;
                s[k][j] = ldb(F.st, t.x + 12u * wrap_sub(F.i, t.y & 0xffffu, z));
            }
#pragma unroll
        for (uint32_t k = 0; k < kFloodCols; ++k)
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                const uint32_t mag = (w[k][j] >> 16 & 0xffu) == (s[k][j].z & 31u) ? s[k][j].y : s[k][j].x;
                const float m = __uint_as_float(mag ^ ((s[k][j].z << (w[k][j] >> 24)) & 0x80000000u));
                if (q0[k] + d + j < q1[k]) v[k] = v[k] + m;
            }
    }
    uint64_t big = 0;
#pragma unroll
    for (uint32_t k = 0; k < kFloodCols; ++k) {
        const uint32_t c = c0 + k * kFloodGroups;
        if (c < F.kb) {
            big |= flood_word(F, c, v[k]);
            if (F.act) stu(F.info + c * z, F.i, v[k]);
        }
    }
    return big;
}

// Decodes one frame; returns the iterations run, or ~0u when the frame has to
// be left to the general kernels.  conv: its last iteration satisfied every
// check.  The hard-decision words of the last iteration are in S.hb.
template <int ND, bool EXTRA>
__device__ __forceinline__ uint32_t flood_frame(FloodFrame &F, uint32_t max_it, bool &conv) {
    const CodeView &cv = F.cv;
    const uint32_t z = cv.z, X = F.pl.X, kb = F.kb, nthr = blockDim.x;
    uint64_t big = 0;
    for (uint32_t v0 = 0; v0 < cv.n; v0 += 8u * nthr) {  // accumulators start at the LLRs
        float l[8];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) l[k] = F.llr[min(v0 + k * nthr + threadIdx.x, cv.n - 1u)];
#pragma unroll
        for (uint32_t k = 0; k < 8; ++k) {
            const uint32_t v = v0 + k * nthr + threadIdx.x;
            big |= __builtin_amdgcn_ballot_w64(too_large(l[k]));
            if (v < X * z) F.S.acc[v] = l[k];
        }
    }
    if (threadIdx.x == 0) *F.S.done = 0;
    if (flood_flags(F.S, false, big)) return ~0u;
    for (uint32_t t = 1;; ++t) {
        const bool first = t == 1;
        const FloodBase B{first ? F.llr : F.info, first ? F.llr : F.par, F.llr};
        big = 0;
        FloodIn<ND> a, b;
        flood_load<ND>(F.pl, a, F.g, F.i, kb, z, B, F.st);
        for (uint32_t r = F.g;;) {  // two rows per turn: the slots of a and b alternate
            flood_load<ND>(F.pl, b, min(r + kFloodGroups, cv.mb - 1u), F.i, kb, z, B, F.st);
            big |= flood_row<ND, EXTRA>(F, a, r, first);
            r += kFloodGroups;
            if (r >= cv.mb) break;
            flood_load<ND>(F.pl, a, min(r + kFloodGroups, cv.mb - 1u), F.i, kb, z, B, F.st);
            big |= flood_row<ND, EXTRA>(F, b, r, first);
            r += kFloodGroups;
            if (r >= cv.mb) break;
        }
        __syncthreads();  // every message added, every state stored
        if (threadIdx.x == 0) *F.S.done = 0;
        for (uint32_t c0 = F.g; c0 < X; c0 += 4u * kFloodGroups) {
            float l[4], v[4];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t c = min(c0 + k * kFloodGroups, X - 1u);
                l[k] = ldu(F.llr + c * z, F.i);
                v[k] = F.S.acc[c * z + F.i];
            }
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const uint32_t c = c0 + k * kFloodGroups;
                if (c < X) {
                    big |= flood_word(F, c, v[k]);
                    if (F.act) {
                        stu(F.info + c * z, F.i, v[k]);
                        F.S.acc[c * z + F.i] = l[k];
                    }
                }
            }
        }
        if constexpr (EXTRA)
            for (uint32_t c = X + F.g; c < kb; c += kFloodCols * kFloodGroups) big |= flood_columns(F, c);
        __syncthreads();  // hard decisions and beliefs complete
        const uint32_t fl = flood_flags(F.S, flood_unsat(cv, F.S), big);
        if (fl & 2u) return ~0u;
        conv = !(fl & 1u);
        if (conv || t == max_it) return t;
    }
}

// LDS layout of a workgroup for one code, and the copy of its parity checks.
__device__ __forceinline__ FloodLds flood_lds(const CodeView &cv, const FloodPlan &pl, uint64_t *smem,
                                              uint32_t *done, uint32_t *bad) {
    FloodLds S;
    S.acc = (lds_float *)smem;  // first: its address folds into the offsets of the accesses
    S.hb = (lds_u64 *)(S.acc + ((pl.X * cv.z + 1u) & ~1u));
    S.carry = (lds_float *)(S.hb + cv.nb * cv.zw);
    const uint32_t lanes = blockDim.x / kFloodGroups;
    S.chk = (lds_u32 *)(S.carry + 5u * lanes);
    S.rp = S.chk + cv.nbe;
    S.unused = (uint32_t)((size_t)S.carry - (size_t)S.acc) + 4u * (4u * lanes + threadIdx.x % lanes);
    S.done = (lds_u32 *)done;
    S.bad = (lds_u32 *)bad;
    for (uint32_t e = threadIdx.x; e < cv.nbe; e += blockDim.x) {
        const uint2 r = cv.row_edge[e];
        S.chk[e] = r.x * cv.zw | (r.y << 16);
    }
    for (uint32_t r = threadIdx.x; r <= cv.mb; r += blockDim.x) S.rp[r] = cv.row_ptr[r];
    return S;
}

// A workgroup's place in the frame: group, wave and lane, and its scratch rows.
__device__ __forceinline__ FloodFrame flood_place(const CodeView &cv, const FloodPlan &pl, const FloodLds &S,
                                                  uint3 *state, float *bel) {
    const uint32_t kb = cv.nb - cv.mb, w = uni(threadIdx.x >> 6), nw = blockDim.x / 64u / kFloodGroups;
    const uint32_t g = w / nw, wave = w - g * nw, i = wave * 64u + (threadIdx.x & 63u);
    return FloodFrame{cv, pl, S, nullptr, state, bel, bel + (size_t)kb * cv.z, g, threadIdx.x & 63u, wave,
                      min(i, cv.z - 1u), nw, kb, i < cv.z, __builtin_amdgcn_ballot_w64(i < cv.z)};
}

// EXTRA: some information columns do not fit the LDS.
template <int ND, bool EXTRA>
__global__ void __launch_bounds__(kFloodThreads) flood_kernel(FloodArgs a) {
    extern __shared__ __align__(16) uint64_t smem[];
    __shared__ uint32_t s_f, s_done, s_bad[kFloodThreads / 64];
    const CodeView &cv = a.cv;
    const FloodLds S = flood_lds(cv, a.plan, smem, &s_done, s_bad);
    FloodFrame F = flood_place(cv, a.plan, S, reinterpret_cast<uint3 *>(a.state) + (size_t)blockIdx.x * cv.m,
                               a.bel + (size_t)blockIdx.x * (cv.n + (size_t)(cv.nb - cv.mb) * cv.z));
    const uint32_t kw = (cv.k + 63) / 64;
    for (;;) {
        __syncthreads();  // the previous frame is done with the LDS
        if (threadIdx.x == 0) s_f = atomicAdd(a.ctr, 1u);
        __syncthreads();
        const uint32_t f = uni(s_f);
        if (f >= a.frames) break;
        F.llr = a.llr + (size_t)f * cv.n;
        bool conv = false;
        const uint32_t its = flood_frame<ND, EXTRA>(F, a.max_it, conv);
        if (its == ~0u) {
            if (threadIdx.x == 0) a.list[atomicAdd(a.count, 1u)] = f;
            continue;
        }
        frame_message(cv, (const uint64_t *)S.hb, a.msg + (size_t)f * kw);
        if (threadIdx.x == 0) {
            a.iters[f] = its;
            a.conv[f] = (uint8_t)conv;
            a.synd[f] = (uint8_t)conv;
            atomicAdd(a.ctr + 1, its);
        }
    }
}

// Value of a uniform struct in memory that no running kernel writes, through
// scalar loads.
template <typename T>
__device__ __forceinline__ T ld_uniform(const T *p) {
    static_assert(sizeof(T) % 4 == 0, "read by words");
    uint32_t w[sizeof(T) / 4];
#pragma unroll
    for (uint32_t k = 0; k < sizeof(T) / 4; ++k) w[k] = uni(ldc(reinterpret_cast<const uint32_t *>(p) + k));
    T v;
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Frames of several codes in one launch: each workgroup draws the next frame
// (the longest codes come first) and runs its code's instantiation.  The
// registers are those of the largest instantiation, which costs nothing: three
// waves per SIMD are also what the LDS of a long code allows.  One launch,
// because a launch per code leaves each with fewer frames than compute units.
// 2000 frames of the twelve Z=360 codes: 9.6 ms, against 22.8 ms for the
// iteration graph of the general kernels.
__global__ void __launch_bounds__(kFloodThreads) flood_mix_kernel(FloodMixArgs a) {
    extern __shared__ __align__(16) uint64_t smem[];
    __shared__ uint32_t s_f, s_done, s_bad[kFloodThreads / 64];
    uint3 *state = reinterpret_cast<uint3 *>(a.state) + (size_t)blockIdx.x * a.state_stride;
    float *bel = a.bel + (size_t)blockIdx.x * a.bel_stride;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) s_f = atomicAdd(a.ctr, 1u);
        __syncthreads();
        const uint32_t j = uni(s_f);
        if (j >= a.frames) break;
        const SlotInfo si = ld_uniform(a.jobs + j);
        const FloodCode fc = ld_uniform(a.codes + si.code);
        const FloodLds S = flood_lds(fc.cv, fc.plan, smem, &s_done, s_bad);
        FloodFrame F = flood_place(fc.cv, fc.plan, S, state, bel);
        F.llr = a.llr + si.llr;
        bool conv = false;
        uint32_t its = ~0u;
        const bool extra = fc.plan.X < fc.cv.nb - fc.cv.mb;
#define GF2L_FLOOD(ND)                                                                            \
    case ND:                                                                                      \
        its = extra ? flood_frame<ND, true>(F, a.max_it, conv) : flood_frame<ND, false>(F, a.max_it, conv); \
        break;
        switch (fc.plan.nd) {
            GF2L_FLOOD_DEGREES
            default: break;
        }
#undef GF2L_FLOOD
        if (its == ~0u) {
            if (threadIdx.x == 0) atomicAdd(a.count, 1u);
            continue;
        }
        frame_message(fc.cv, (const uint64_t *)S.hb, a.msg + si.msg);
        if (threadIdx.x == 0) {
            a.iters[si.frame] = its;
            a.conv[si.frame] = (uint8_t)conv;
            a.synd[si.frame] = (uint8_t)conv;
        }
    }
}

__global__ void clear_words_kernel(uint32_t *p, uint32_t n) {
    for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0;
}

// LDS bytes besides the accumulators.
size_t flood_fixed_bytes(const CodeView &cv, uint32_t lanes) {
    return (size_t)cv.nb * cv.zw * 8 + 5ull * lanes * sizeof(float) + (size_t)cv.nbe * 4 + (cv.mb + 1ull) * 4 + 4;
}

uint32_t flood_lanes(uint32_t z) { return (z + 63u) & ~63u; }

}  // namespace

hipError_t launch_clear_words(uint32_t *words, uint32_t count, hipStream_t s) {
    hipLaunchKernelGGL(clear_words_kernel, dim3((count + 255) / 256), dim3(256), 0, s, words, count);
    return hipGetLastError();
}

size_t flood_bytes(const CodeView &cv, const FloodPlan &pl) {
    return flood_fixed_bytes(cv, flood_lanes(cv.z)) + (size_t)pl.X * cv.z * sizeof(float);
}

int build_flood_plan(gf2l_ctx *ctx, gf2l_code *c) {
    const CodeView &cv = c->view;
    if (cv.dvb_q || cv.nb <= cv.mb || cv.mb < 2 || cv.z < 64 || cv.z > kFloodThreads / kFloodGroups ||
        cv.nb * cv.zw > 0xffffu)
        return GF2L_OK;
    const uint32_t kb = cv.nb - cv.mb;
    uint32_t most = 0, inputs = 0;
    for (uint32_t br = 0; br < cv.mb; ++br) {
        const uint32_t e0 = c->h_row_ptr[br], d = c->h_row_ptr[br + 1] - e0, np = br > 0 ? 2u : 1u;
        if (d <= np) return GF2L_OK;
        const uint2 last = c->h_row_edge[e0 + d - 1], prev = c->h_row_edge[e0 + d - np];
        if (last.x != kb + br || last.y != 0 || prev.x + 1 != kb + br + (br > 0 ? 0u : 1u) || prev.y != 0)
            return GF2L_OK;
        if (c->h_row_edge[e0 + d - np - 1].x >= kb) return GF2L_OK;
        most = std::max(most, d - np);
        inputs += d - np;
    }
    uint32_t nd = 0;
#define GF2L_FLOOD(ND) nd = !nd && ND >= most ? ND : nd;
    GF2L_FLOOD_DEGREES
#undef GF2L_FLOOD
    // Rows are loaded padded to nd inputs.  Where two thirds of them are padding the
    // other kernels are faster from 256 frames on (N = 64800, rows of 1 to 25 inputs,
    // 4.0 on average: 256 frames 1154 -> 1560 us, 7.4 on average: 1368 -> 1397, at
    // high Eb/N0 308 -> 399; rows of 4 to 17, 12 on average: 1511 -> 1026).
    if (cv.mb * nd > 3u * inputs) return GF2L_OK;
    const size_t fixed = flood_fixed_bytes(cv, flood_lanes(cv.z)) + 256;
    if (!nd || fixed >= ctx->lds_limit) return GF2L_OK;
    const uint32_t X = (uint32_t)std::min<size_t>(kb, (ctx->lds_limit - fixed) / (cv.z * sizeof(float)));
    std::vector<uint2> edge((size_t)cv.mb * nd, make_uint2(0, cv.z));
    std::vector<uint32_t> row(cv.mb);
    for (uint32_t br = 0; br < cv.mb; ++br) {
        const uint32_t e0 = c->h_row_ptr[br], ni = c->h_row_ptr[br + 1] - e0 - (br > 0 ? 2u : 1u);
        uint32_t nl = 0;
        for (uint32_t p = 0; p < ni; ++p) {
            const uint2 e = c->h_row_edge[e0 + p];
            edge[(size_t)br * nd + p] = make_uint2(4u * (e.x * cv.z + e.y), cv.z - e.y);
            nl += e.x < X ? 1u : 0u;
        }
        const uint32_t exact = br > 0 && ni + 1 >= nd ? ni : nd;  // the state layout's degree (flood_row)
        row[br] = ni | (nl << 8) | (exact << 16);
    }
    // the columns past X: {byte offset of the block-row's states, shift |
    // position in the check << 16 | shift of its sign bit << 24}
    std::vector<uint32_t> xptr(kb - X + 1, 0);
    std::vector<uint2> xedge;
    for (uint32_t bc = X; bc < kb; ++bc) {
        for (uint32_t q = c->h_col_ptr[bc]; q < c->h_col_ptr[bc + 1]; ++q) {
            const uint4 ci = c->h_col_info[q];
            xedge.push_back(make_uint2(12u * ci.x * cv.z,
                                       ci.z | ((ci.y + 2u) << 16) | ((27u - (row[ci.x] >> 16) + ci.y) << 24)));
        }
        xptr[bc - X + 1] = (uint32_t)xedge.size();
    }
    for (int k = 0; k < 4; ++k) xedge.push_back(make_uint2(0, 0));
    edge.insert(edge.end(), xedge.begin(), xedge.end());
    row.insert(row.end(), xptr.begin(), xptr.end());
    const size_t b_e = edge.size() * sizeof(uint2), b_r = row.size() * sizeof(uint32_t);
    char *d = nullptr;
    GF2L_HIP(ctx, hipMalloc(&d, b_e + b_r));
    hipError_t e = hipMemcpy(d, edge.data(), b_e, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(d + b_e, row.data(), b_r, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        hipFree(d);
        return fail(ctx, GF2L_ERR_HIP, std::string("code upload: ") + hipGetErrorString(e));
    }
    c->d_flood = d;
    c->flood.edge = reinterpret_cast<const uint2 *>(d);
    c->flood.xedge = c->flood.edge + (size_t)cv.mb * nd;
    c->flood.row = reinterpret_cast<const uint32_t *>(d + b_e);
    c->flood.xptr = c->flood.row + cv.mb;
    c->flood.nd = nd;
    c->flood.X = X;
    return GF2L_OK;
}

// Workgroups of a launch: the registers allow three or four waves per SIMD.
uint32_t flood_grid(const CodeView &cv, const FloodPlan &pl, uint32_t frames, int num_cus) {
    const uint32_t waves = flood_lanes(cv.z) / 64u * kFloodGroups;
    const uint32_t per_cu = (uint32_t)std::max<size_t>(
        1, std::min<size_t>(12u / waves, (160 * 1024) / (flood_bytes(cv, pl) + 256)));
    return std::max(1u, std::min(frames, (uint32_t)num_cus * per_cu));
}

hipError_t launch_flood_mix(const FloodMixArgs &a, size_t lds, uint32_t block, uint32_t grid, hipStream_t s) {
    auto k = flood_mix_kernel;
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(k, dim3(grid), dim3(block), lds, s, a);
    return hipGetLastError();
}

uint32_t flood_block(const CodeView &cv) { return flood_lanes(cv.z) * kFloodGroups; }

hipError_t launch_flood(const FloodArgs &a, uint32_t grid, hipStream_t s) {
    const size_t bytes = flood_bytes(a.cv, a.plan);
    const uint32_t block = flood_block(a.cv);
#define GF2L_FLOOD(ND)                                                                                       \
    case ND: {                                                                                               \
        auto k = a.plan.X < a.cv.nb - a.cv.mb ? flood_kernel<ND, true> : flood_kernel<ND, false>;            \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),                          \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);    \
        if (e != hipSuccess) return e;                                                                       \
        hipLaunchKernelGGL(k, dim3(grid), dim3(block), bytes, s, a);                                         \
        break;                                                                                               \
    }
    switch (a.plan.nd) {
        GF2L_FLOOD_DEGREES
        default: return hipErrorInvalidValue;
    }
#undef GF2L_FLOOD
    return hipGetLastError();
}

}  // namespace gf2l
