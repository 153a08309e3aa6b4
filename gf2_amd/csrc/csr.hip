// General sparse (CSR/CSC) path of the min-sum decoder, for codes built from
// an arbitrary edge list: LdpcCode::from_edges (crates/gf2-coding/src/ldpc/
// core.rs:96-104) -> SpBitMatrixDual::from_coo (crates/gf2-core/src/sparse.rs:
// 166-204, 297-331, 441-445).  Same arithmetic contract as the quasi-cyclic
// paths: check message = sign_product * min over the other inputs (AVX2
// lane / remainder sign rule), belief = L + c2v in ascending check order,
// v2c = belief - c2v recomputed from the stored belief and message.
//
// Per frame in HBM: c2v [nnz] in CSR order, beliefs [n], hard decisions
// [ceil(n/64)] in the linear BitVec layout.  One thread per check (check
// kernel) and per variable (variable kernel); degrees vary per thread, so
// the loops are runtime-bounded.
//
// Where memory allows, frames run in groups of 64, one frame per lane (the
// second half of this file): with no structure in the code, the frames are what
// neighbouring lanes can share.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "device_common.h"
#include "gf2ldpc.h"
#include "host_codes.h"

namespace gf2l {
namespace {

__global__ void __launch_bounds__(256)
cn_csr_kernel(CsrView cv, const uint32_t *__restrict__ list, const uint32_t *__restrict__ count_ptr,
              float *__restrict__ c2v, const float *__restrict__ belief) {
    const uint32_t chunks = (cv.m + blockDim.x - 1) / blockDim.x;
    const uint32_t items = *count_ptr * chunks;
    for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
        const uint32_t f = list[item / chunks];
        const uint32_t r = (item % chunks) * blockDim.x + threadIdx.x;
        if (r >= cv.m) continue;
        float *fc = c2v + (size_t)f * cv.nnz;
        const float *fb = belief + (size_t)f * cv.n;
        const uint32_t e0 = cv.row_ptr[r], d = cv.row_ptr[r + 1] - e0;
        CheckAcc acc;
        acc.init();
        for (uint32_t p = 0; p < d; ++p) acc.add(p, fb[cv.col_idx[e0 + p]] - fc[e0 + p]);
        for (uint32_t p = 0; p < d; ++p) fc[e0 + p] = acc.out(d, p);
    }
}

__global__ void __launch_bounds__(256)
vn_csr_kernel(CsrView cv, const uint32_t *__restrict__ list, const uint32_t *__restrict__ count_ptr,
              const float *__restrict__ c2v, float *__restrict__ belief, const float *__restrict__ llr,
              uint64_t *__restrict__ hb, uint32_t *__restrict__ next_count) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *next_count = 0;
    const uint32_t chunks = (cv.n + blockDim.x - 1) / blockDim.x;
    const uint32_t items = *count_ptr * chunks;
    const uint32_t nw = (cv.n + 63) / 64;
    for (uint32_t item = blockIdx.x; item < items; item += gridDim.x) {
        const uint32_t f = list[item / chunks];
        const uint32_t v = (item % chunks) * blockDim.x + threadIdx.x;
        float bel = 0.0f;
        if (v < cv.n) {
            const float *fc = c2v + (size_t)f * cv.nnz;
            bel = llr[(size_t)f * cv.n + v];
            for (uint32_t q = cv.col_ptr[v]; q < cv.col_ptr[v + 1]; ++q) bel = bel + fc[cv.csc_edge[q]];
            belief[(size_t)f * cv.n + v] = bel;
        }
        const uint64_t mask = __ballot(v < cv.n && bel < 0.0f);
        if ((threadIdx.x & 63) == 0 && v < cv.n) hb[(size_t)f * nw + (v >> 6)] = mask;
    }
}

// One workgroup per frame: syndrome from the linear hard-decision words, then
// retire (first k bits are the message) or keep the frame running.  A frame's
// checks are dependent table and bit lookups: up to sixteen waves, as many as have
// checks, hide what one wave waited for (4,500 checks, 500 frames: 4.01 -> 2.57 ms
// for the decode).
constexpr uint32_t kSynThreads = 1024;
__global__ void __launch_bounds__(kSynThreads)
syn_csr_kernel(CsrView cv, const uint32_t *__restrict__ list, const uint32_t *__restrict__ count_ptr,
               uint32_t *__restrict__ next_list, uint32_t *__restrict__ next_count,
               const uint64_t *__restrict__ hb, uint32_t it_report, int last,
               uint64_t *__restrict__ msg, uint32_t *__restrict__ iters, uint8_t *__restrict__ conv,
               uint8_t *__restrict__ synd) {
    extern __shared__ uint64_t sh[];
    const uint32_t count = *count_ptr;
    const uint32_t nw = (cv.n + 63) / 64, kw = (cv.k + 63) / 64;
    for (uint32_t item = blockIdx.x; item < count; item += gridDim.x) {
        const uint32_t f = list[item];
        for (uint32_t w = threadIdx.x; w < nw; w += blockDim.x) sh[w] = hb[(size_t)f * nw + w];
        __syncthreads();
        uint32_t bad = 0;
        for (uint32_t r = threadIdx.x; r < cv.m; r += blockDim.x) {
            uint32_t par = 0;
            for (uint32_t e = cv.row_ptr[r]; e < cv.row_ptr[r + 1]; ++e) {
                const uint32_t v = cv.col_idx[e];
                par ^= (uint32_t)(sh[v >> 6] >> (v & 63u)) & 1u;
            }
            bad |= par;
        }
        const int unsat = __syncthreads_or(bad != 0);
        if (!unsat || last) {
            for (uint32_t w = threadIdx.x; w < kw; w += blockDim.x) {
                uint64_t word = sh[w];
                if (64u * w + 64u > cv.k) word &= (1ull << (cv.k - 64u * w)) - 1;
                msg[(size_t)f * kw + w] = word;
            }
            if (threadIdx.x == 0) {
                iters[f] = it_report;
                conv[f] = (uint8_t)!unsat;
                synd[f] = (uint8_t)!unsat;
            }
        } else if (threadIdx.x == 0) {
            next_list[atomicAdd(next_count, 1u)] = f;
        }
        __syncthreads();
    }
}

__global__ void csr_init_kernel(uint32_t *list, uint32_t *counts, uint32_t frames) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < frames) list[t] = t;
    if (t == 0) {
        counts[0] = frames;
        counts[1] = 0;
    }
}

// ---------------------------------------------------------------------------
// Groups of 64 frames.  Per group: messages [nnz][64], beliefs and LLRs
// [n][64], hard decisions [n] words (bit = lane).  A wave takes one check (one
// variable) of a group, so the code tables are scalar loads, every access is
// one row of 64 floats, and a parity is an XOR of lane masks for 64 frames.  A
// group runs while one of its frames does; when half of the groups would do for
// the running frames, they are packed into new groups.  Two kernels an
// iteration (a small batch costs launches, not work): the syndrome comes with
// the next check pass, which reads the beliefs anyway.  At n = 9,000, 500 frames
// the check pass moves 162 MB in 23 us, near what memory gives; a decode takes
// 0.89 ms, 4.01 before with a frame's arrays contiguous.

constexpr uint32_t kGroupThreads = 512;  // of the check and variable passes

// Workgroup split (workgroup b runs on XCD b % 8): whole rounds of eight groups
// go one group to an XCD, whose L2 then serves the repeated reads of the
// group's beliefs; there `share` workgroups take a group, and where a code has
// fewer rows than the XCD's workgroups have waves several groups run beside each
// other (one after the other, 65,536 frames of n = 64 took 5.0 ms for seven
// iterations, now 0.9; a million of n = 7 18.3, now 0.5).  The rows of the up to
// seven groups left over are spread over the chip (one group of 8,000 checks on
// one XCD took 60 us an iteration), each over its own part of it (split) where
// every row finds a wave there: 256 error-free frames of n = 300 58 -> 39 us.
// Calls f(group, first row, row stride, this workgroup's place among those of
// the group, their number).
struct GroupSplit {
    uint32_t share, split;
};
template <typename F>
__device__ __forceinline__ void each_group(uint32_t groups, GroupSplit sp, F &&f) {
    const uint32_t share = sp.share;
    const uint32_t x = blockIdx.x & 7u, b = blockIdx.x >> 3, per = blockDim.x >> 6, wave = uni(threadIdx.x >> 6);
    const uint32_t full = groups >> 3, beside = (gridDim.x >> 3) / share, at = b / share, place = b - at * share;
    if (at < beside)
        for (uint32_t t = at; t < full; t += beside) f(8u * t + x, place * per + wave, share * per, place, share);
    const uint32_t left = groups & 7u;
    if (left && sp.split) {
        const uint32_t part = gridDim.x / left, g = blockIdx.x / part, p = blockIdx.x - g * part;
        if (g < left) f(8u * full + g, p * per + wave, part * per, p, part);
        return;
    }
    for (uint32_t g = 8u * full; g < groups; ++g)
        f(g, 8u * (b * per + wave) + x, gridDim.x * per, blockIdx.x, gridDim.x);
}

// Check messages of one check for 64 frames: CheckAcc's rule.  Up to 8 inputs
// the sign rule is `< 0` for every input (no full 8-lane chunk among the
// others), and the signs are lane masks: products of signs are scalar XORs.
template <int D>
__device__ __forceinline__ void group_check(const float *x, float *out) {
    if constexpr (D == 1) {
        out[0] = 0.0f;
    } else if constexpr (D <= 8) {
        float m1 = __builtin_inff(), m2 = __builtin_inff();
        uint32_t idx = 0;
        uint64_t neg[D], all = 0;
#pragma unroll
        for (int p = 0; p < D; ++p) {
            const float a = fabsf(x[p]);
            const bool lt1 = a < m1, lt2 = a < m2;
            m2 = lt1 ? m1 : (lt2 ? a : m2);
            m1 = lt1 ? a : m1;
            idx = lt1 ? (uint32_t)p : idx;
            neg[p] = __builtin_amdgcn_ballot_w64(x[p] < 0.0f);
            all ^= neg[p];
        }
#pragma unroll
        for (int p = 0; p < D; ++p) {
            const float mag = (uint32_t)p == idx ? m2 : m1;
            out[p] = __builtin_amdgcn_inverse_ballot_w64(all ^ neg[p]) ? -mag : mag;
        }
    } else {
        CheckAcc acc;
        acc.init();
#pragma unroll
        for (int p = 0; p < D; ++p) acc.add_sel(p, x[p]);
        const uint32_t sg = acc.signs<D>(D);
#pragma unroll
        for (int p = 0; p < D; ++p) {
            const float mag = (uint32_t)p == acc.idx ? acc.min2 : acc.min1;
            out[p] = ((sg >> p) & 1u) ? -mag : mag;
        }
    }
}

// What an iteration's kernels share: running frames of a group and frames with
// an unsatisfied check (a word per workgroup of the check pass: or-ing them with
// atomics on one word, 4,500 waves of it, took 60 us).
struct GroupState {
    const uint64_t *act_in;
    uint64_t *act_out, *unsat;
    uint32_t *running;
};

// OR of the waves' (uniform) words over the workgroup.
__device__ __forceinline__ uint64_t group_or(uint64_t v, uint64_t *red) {
    __syncthreads();
    if ((threadIdx.x & 63u) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    uint64_t all = 0;
#pragma unroll
    for (uint32_t w = 0; w < kGroupThreads / 64u; ++w) all |= red[w];
    return all;
}

// Check pass of iteration it, and the parities of the beliefs of iteration
// it - 1 that it reads.  FIRST: beliefs are the LLRs, no old messages.
template <int MAXD, bool FIRST>
__global__ void __launch_bounds__(kGroupThreads)
cn_group_kernel(CsrView cv, uint32_t groups, GroupSplit sp, GroupState gs, float *__restrict__ c2v, const float *__restrict__ belief) {
    const uint32_t lane4 = 4u * (threadIdx.x & 63u);
    if (blockIdx.x == 0 && threadIdx.x == 0) *gs.running = 0;
    __shared__ uint64_t red[kGroupThreads / 64];
    each_group(groups, sp, [&](uint32_t g, uint32_t r0, uint32_t step, uint32_t slot, uint32_t) {
        if (ldc(gs.act_in + g) == 0) return;
        float *gc = c2v + (size_t)g * cv.nnz * 64u;
        const float *gb = belief + (size_t)g * cv.n * 64u;
        uint64_t bad = 0;
        for (uint32_t r = r0; r < cv.m; r += step) {
            const uint32_t e0 = uni(ldc(cv.row_ptr + r)), d = uni(ldc(cv.row_ptr + r + 1)) - e0;
            dispatch_degree<MAXD>(d, [&](auto DC) {
                constexpr int D = decltype(DC)::value, DA = D > 0 ? D : 1;
                float x[DA], o[DA];
#pragma unroll
                for (int p = 0; p < D; ++p) x[p] = ldb(gb, 256u * uni(ldc(cv.col_idx + e0 + p)) + lane4);
                if constexpr (!FIRST) {
                    float c[DA];
#pragma unroll
                    for (int p = 0; p < D; ++p) c[p] = ldb(gc, 256u * (e0 + p) + lane4);
                    uint64_t par = 0;
#pragma unroll
                    for (int p = 0; p < D; ++p) par ^= __builtin_amdgcn_ballot_w64(x[p] < 0.0f);
                    bad |= par;
#pragma unroll
                    for (int p = 0; p < D; ++p) x[p] = x[p] - c[p];
                }
                if constexpr (D > 0) group_check<D>(x, o);
                char *out = reinterpret_cast<char *>(gc);
#pragma unroll
                for (int p = 0; p < D; ++p) *reinterpret_cast<float *>(out + (256u * (e0 + p) + lane4)) = o[p];
            });
        }
        if constexpr (!FIRST) {
            const uint64_t all = group_or(bad, red);
            if (threadIdx.x == 0) gs.unsat[(size_t)g * gridDim.x + slot] = all;
        }
    });
}

// Variable pass of iteration it.  Before it, the frames whose checks were
// satisfied after iteration it - 1 (all frames in the pass after the last
// iteration) leave with the hard decisions of that iteration.
__global__ void __launch_bounds__(kGroupThreads)
vn_group_kernel(CsrView cv, uint32_t groups, GroupSplit sp, GroupState gs, const float *__restrict__ c2v,
                float *__restrict__ belief, const float *__restrict__ llr, const uint64_t *__restrict__ hb_in, uint64_t *__restrict__ hb_out,
                const uint32_t *__restrict__ map, uint32_t it, int last, uint64_t *__restrict__ msg,
                uint32_t *__restrict__ iters, uint8_t *__restrict__ conv, uint8_t *__restrict__ synd) {
    const uint32_t lane = threadIdx.x & 63u, lane4 = 4u * lane;
    __shared__ uint64_t red[kGroupThreads / 64];
    each_group(groups, sp, [&](uint32_t g, uint32_t v0, uint32_t step, uint32_t, uint32_t slots) {
        const uint64_t act = ldc(gs.act_in + g);
        if (act == 0) {  // uniform
            if (v0 == 0 && lane == 0) gs.act_out[g] = 0;
            return;
        }
        uint64_t bad = ~0ull;
        if (it > 1) {
            bad = 0;
            for (uint32_t t = threadIdx.x; t < slots; t += blockDim.x) bad |= gs.unsat[(size_t)g * gridDim.x + t];
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) bad |= (uint64_t)__shfl_xor((unsigned long long)bad, o, 64);
            bad = group_or(bad, red);
        }
        bad &= act;
        const uint64_t stop = last ? act : act & ~bad, run = act & ~stop;
        if (v0 == 0 && lane == 0) {
            gs.act_out[g] = run;
            if (run) atomicAdd(gs.running, (uint32_t)__popcll(run));
        }
        if (stop) {
            const uint32_t kw = (cv.k + 63u) / 64u, f = map[g * 64u + lane];
            const uint64_t *gh = hb_in + (size_t)g * cv.n;
            const bool mine = (stop >> lane) & 1ull;
            for (uint32_t w = v0; w < kw; w += step) {
                const uint32_t v = 64u * w + lane;
                const uint64_t bits = v < cv.k ? gh[v] : 0ull;
                uint64_t word = 0;  // of this lane's frame
                for (uint64_t s = stop; s; s &= s - 1) {  // uniform
                    const uint32_t t = (uint32_t)__builtin_ctzll(s);
                    const uint64_t m = __builtin_amdgcn_ballot_w64(((bits >> t) & 1ull) != 0);
                    word = lane == t ? m : word;
                }
                if (mine) msg[(size_t)f * kw + w] = word;
            }
            if (v0 == 0 && mine) {
                iters[f] = it - 1u;
                conv[f] = synd[f] = (uint8_t)(((bad >> lane) & 1ull) == 0);
            }
        }
        if (run == 0) return;
        const float *gc = c2v + (size_t)g * cv.nnz * 64u, *gl = llr + (size_t)g * cv.n * 64u;
        float *gb = belief + (size_t)g * cv.n * 64u;
        uint64_t *gh = hb_out + (size_t)g * cv.n;
        for (uint32_t v = v0; v < cv.n; v += step) {
            const uint32_t q0 = uni(ldc(cv.col_ptr + v)), q1 = uni(ldc(cv.col_ptr + v + 1));
            float b = ldb(gl, 256u * v + lane4);
            for (uint32_t q = q0; q < q1; q += 4) {  // four messages in flight, added in check order
                float c[4];
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    c[k] = ldb(gc, 256u * uni(ldc(cv.csc_edge + min(q + k, q1 - 1u))) + lane4);
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k)
                    if (q + k < q1) b = b + c[k];
            }
            *reinterpret_cast<float *>(reinterpret_cast<char *>(gb) + (256u * v + lane4)) = b;
            const uint64_t mask = __builtin_amdgcn_ballot_w64(b < 0.0f);
            if (lane == 0) gh[v] = mask;
        }
    });
}

__global__ void group_init_kernel(uint64_t *active, uint32_t *map, uint32_t groups, uint32_t frames) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t < groups * 64u) map[t] = min(t, frames - 1u);
    if (t < groups) active[t] = frames - t * 64u >= 64u ? ~0ull : (1ull << (frames - t * 64u)) - 1ull;
}

// [frames][n] LLRs to [groups][n][64] (lanes past the last frame: copies of it)
__global__ void __launch_bounds__(256)
group_llr_kernel(const float *__restrict__ llr, float *__restrict__ out, uint32_t frames, uint32_t n) {
    __shared__ float tile[64][65];
    const uint32_t g = blockIdx.y, v0 = blockIdx.x * 64u, lane = threadIdx.x & 63u;
    for (uint32_t f = threadIdx.x >> 6; f < 64; f += 4)
        if (v0 + lane < n) tile[f][lane] = llr[(size_t)min(g * 64u + f, frames - 1u) * n + v0 + lane];
    __syncthreads();
    for (uint32_t v = threadIdx.x >> 6; v < 64; v += 4)
        if (v0 + v < n) out[((size_t)g * n + v0 + v) * 64u + lane] = tile[lane][v];
}

// Packing: the running lanes in order get new slots; src[new] = old slot.
// One workgroup, a stretch of the groups per wave: the waves count theirs, then
// write from where the waves before them end, 64 masks in flight (one wave over
// all groups waited for each of them).
__global__ void __launch_bounds__(1024)
group_pack_kernel(uint64_t *__restrict__ active, uint32_t groups, const uint32_t *__restrict__ map,
                  uint32_t *__restrict__ new_map, uint32_t *__restrict__ src, uint32_t total) {
    __shared__ uint32_t s_sum[16];
    const uint32_t lane = threadIdx.x & 63u, wave = uni(threadIdx.x >> 6);
    const uint32_t new_groups = (total + 63u) / 64u;
    const uint32_t stretch = (groups + 15u) / 16u, g0 = min(wave * stretch, groups), g1 = min(g0 + stretch, groups);
    uint32_t sum = 0;
    for (uint32_t g = g0 + lane; g < g1; g += 64u) sum += (uint32_t)__popcll(active[g]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) sum += (uint32_t)__shfl_xor((int)sum, o, 64);
    if (lane == 0) s_sum[wave] = sum;
    __syncthreads();
    uint32_t base = 0, used = 0;  // used: all of them (total, as the host read it)
    for (uint32_t w = 0; w < 16u; ++w) {
        base += w < wave ? s_sum[w] : 0u;
        used += s_sum[w];
    }
    for (uint32_t gb = g0; gb < g1; gb += 64u) {
        const uint64_t mine = gb + lane < g1 ? active[gb + lane] : 0ull;
        const uint32_t count = min(64u, g1 - gb);
        for (uint32_t k = 0; k < count; ++k) {
            const uint64_t a = __shfl((unsigned long long)mine, (int)k, 64);
            if ((a >> lane) & 1ull) {
                const uint32_t at = base + (uint32_t)__popcll(a & ((1ull << lane) - 1ull));
                src[at] = (gb + k) * 64u + lane;
                new_map[at] = map[(gb + k) * 64u + lane];
            }
            base += (uint32_t)__popcll(a);
        }
    }
    __syncthreads();
    // the last group's free lanes repeat its last frame (masked off)
    for (uint32_t t = used + threadIdx.x; t < new_groups * 64u; t += blockDim.x) {
        src[t] = src[used - 1u];
        new_map[t] = new_map[used - 1u];
    }
    for (uint32_t g = threadIdx.x; g < groups; g += blockDim.x)
        active[g] = g >= new_groups ? 0ull : used - g * 64u >= 64u ? ~0ull : (1ull << (used - g * 64u)) - 1ull;
}

// Rows of the packed groups: out[g][row][lane] = in[src group][row][src lane];
// hb (may be null): the sign masks of the rows.
__global__ void __launch_bounds__(256)
group_move_kernel(const uint32_t *__restrict__ src, const float *__restrict__ in, float *__restrict__ out,
                  uint64_t *__restrict__ hb, uint32_t rows) {
    const uint32_t g = blockIdx.y, lane = threadIdx.x & 63u;
    const uint32_t s = src[g * 64u + lane];
    const float *p = in + (size_t)(s >> 6) * rows * 64u + (s & 63u);
    float *o = out + (size_t)g * rows * 64u + lane;
    for (uint32_t r = blockIdx.x * 4u + (threadIdx.x >> 6); r < rows; r += gridDim.x * 4u) {
        const float b = p[(size_t)r * 64u];
        o[(size_t)r * 64u] = b;
        if (hb) {
            const uint64_t mask = __builtin_amdgcn_ballot_w64(b < 0.0f);
            if (lane == 0) hb[(size_t)g * rows + r] = mask;
        }
    }
}

}  // namespace

// Codes whose group arrays are indexed by 32-bit byte offsets run in groups: two
// launches an iteration instead of three win where the launches bound (one frame
// of n = 2,000: 280 -> 201 us, of n = 300,000: 3.59 -> 3.39 ms), whole rows instead
// of gathered floats elsewhere (n = 9,000, 500 frames: 2.57 -> 0.89 ms against the
// kernels above).  A single frame of up to 128 variables has nothing to win: 86
// against 112 us for n = 7, 155 against 138 for n = 128.  One or two frames of 2^16
// variables and more gain little (n = 300,000: 2.09 -> 2.01 and 2.28 -> 2.01 ms;
// error-free 256 and 332 us stay below 385) and would take the memory of 64.
static bool use_groups(const CsrView &cv, uint32_t frames) {
    if ((frames == 1 && cv.n <= 128) || (frames <= 2 && cv.n >= (1u << 16))) return false;
    return cv.nnz > 0 && cv.m > 0 && cv.nnz < (1u << 20) && cv.n < (1u << 20);
}
static uint32_t group_grid_most(const gf2l_ctx *ctx) { return 8u * ((uint32_t)ctx->num_cus / 2u); }
// Whether each of the last groups of a pass (fewer than eight) has its own part of
// a full grid: every row of them finds a wave.
static bool groups_split(const gf2l_ctx *ctx, const CsrView &cv, uint32_t groups) {
    return (uint64_t)std::max(cv.m, cv.n) * (groups & 7u) <= (uint64_t)group_grid_most(ctx) * (kGroupThreads / 64u);
}
// Workgroups of a pass over `groups` groups: a multiple of 8, at most four to a
// compute unit, and no more than the rows of a round of groups, or of all the
// groups that are split (where they are not, more workgroups than one group needs
// cost 10%: n = 3,000, 130 frames 250 -> 290 us).
static uint32_t group_grid(const gf2l_ctx *ctx, const CsrView &cv, uint32_t groups) {
    const uint64_t waves = kGroupThreads / 64u, one = std::max(cv.m, cv.n),
                   rows = groups >= 8 ? one * ((groups + 7u) / 8u) : one * (groups_split(ctx, cv, groups) ? groups : 1u) / 8u;
    return 8u * (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>(group_grid_most(ctx) / 8u, (rows + waves - 1u) / waves));
}
// Workgroups of an XCD that share a group: four rows a wave, or fewer where there
// are fewer groups than that leaves room for.
static GroupSplit group_split(const gf2l_ctx *ctx, const CsrView &cv, uint32_t groups, uint32_t grid) {
    const uint32_t waves = kGroupThreads / 64u, rows = std::max(cv.m, cv.n), rounds = std::max(1u, groups / 8u);
    const uint32_t four = (rows + 4u * waves - 1u) / (4u * waves), one = (rows + waves - 1u) / waves;
    return {std::min(grid / 8u, std::min(one, std::max(four, grid / 8u / rounds))), groups_split(ctx, cv, groups) ? 1u : 0u};
}
// Floats of a row of 64 frames' arrays over `groups` groups: the groups themselves
// and, for the packed ones, half as many (a single group is never packed).
static size_t group_slots(uint32_t groups) { return 64 * ((size_t)groups + groups / 2); }
// Groups per pass: the workspace of a pass stays below 4 GiB (the longest codes:
// 1.2 GB a group), and groups fit a dimension of the grid.
static uint32_t groups_per_pass(const gf2l_ctx *ctx, const CsrView &cv) {
    const size_t per_group = ((size_t)cv.nnz + 2 * (size_t)cv.n) * 96 * sizeof(float) +
                             (2 * (size_t)cv.n + 2 + group_grid_most(ctx)) * sizeof(uint64_t) + 128 * sizeof(uint32_t);
    return (uint32_t)std::max<size_t>(1, std::min<size_t>(65535, ((size_t)4 << 30) / per_group));
}

static int decode_csr_groups(gf2l_ctx *ctx, const gf2l_code *code, const float *d_llr, uint32_t F, uint32_t max_it,
                             uint64_t *d_msg, uint32_t *d_iters, uint8_t *d_conv, uint8_t *d_synd) {
    const CsrView &cv = code->csr;
    hipStream_t s = ctx->stream;
    uint32_t groups = (uint32_t)(((uint64_t)F + 63u) / 64u);
    const size_t slots = (size_t)groups * 64u;
    // the second region of each array takes the packed groups (at most half)
    Workspace &ws = ctx->ws;
    float *c2v[2] = {ws.c2v, ws.c2v + slots * cv.nnz}, *bel[2] = {ws.belief, ws.belief + slots * cv.n},
          *llr[2] = {ws.llr_perm, ws.llr_perm + slots * cv.n};
    uint64_t *hb[2] = {ws.hb, ws.hb + (size_t)groups * cv.n}, *active[2] = {hb[1] + (size_t)groups * cv.n, nullptr};
    active[1] = active[0] + groups;
    uint64_t *unsat = active[1] + groups;
    uint32_t *map[2] = {ws.lists, ws.lists + slots}, *src = map[1] + (group_slots(groups) - slots), *running = ws.counts;
    uint32_t cur = 0;
    hipLaunchKernelGGL(group_init_kernel, dim3((groups * 64u + 255) / 256), dim3(256), 0, s, active[0], map[0], groups, F);
    hipLaunchKernelGGL(group_llr_kernel, dim3((cv.n + 63u) / 64u, groups), dim3(256), 0, s, d_llr, llr[0], F, cv.n);
    const uint32_t grid = group_grid(ctx, cv, groups);
    const uint32_t max_dc = code->view.max_dc;
    const uint32_t batch = (uint32_t)std::max(1, std::min(ctx->tune.graph_iters, kProfileSlots));
    // Few frames of a short code: launches are all there is, so those that one
    // iteration decodes are asked for at once (error-free: n = 2,000, 1 to 64 frames
    // 75 -> 36 us, n = 64, 4,096 frames 77 -> 39; in noise n = 2,000, 16 frames 200
    // -> 180; with n = 6,000, 100 frames, or n = 9,000, the question costs 2% to 8%
    // in noise).
    const bool quick = cv.n <= 6000 && (uint64_t)cv.n * groups < 10000;
    // the pass after the last iteration takes its parities and retires the rest
    for (uint64_t it = 1; it <= (uint64_t)max_it + 1; ++it) {
        const uint32_t in = (it - 1) & 1u, out = it & 1u;
        const bool last = it > max_it;
        const GroupState gs{active[in], active[out], unsat, running};
        const GroupSplit sp = group_split(ctx, cv, groups, grid);
        const float *b_in = it == 1 ? llr[cur] : bel[cur];
#define GF2L_CNG(MD, FI) \
    hipLaunchKernelGGL((cn_group_kernel<MD, FI>), dim3(grid), dim3(kGroupThreads), 0, s, cv, groups, sp, gs, c2v[cur], b_in)
#define GF2L_CNG_FIRST(MD) \
    do { if (it == 1) GF2L_CNG(MD, true); else GF2L_CNG(MD, false); } while (0)
        if (max_dc <= 8)
            GF2L_CNG_FIRST(8);
        else if (max_dc <= 16)
            GF2L_CNG_FIRST(16);
        else
            GF2L_CNG_FIRST(32);
#undef GF2L_CNG_FIRST
#undef GF2L_CNG
        hipLaunchKernelGGL(vn_group_kernel, dim3(grid), dim3(kGroupThreads), 0, s, cv, groups, sp, gs, c2v[cur], bel[cur], llr[cur],
                           hb[in], hb[out], map[cur], (uint32_t)it, (int)last, d_msg, d_iters, d_conv, d_synd);
        GF2L_HIP(ctx, hipGetLastError());
        if ((it % batch != 0 && !(quick && it == 2)) || last) continue;
        GF2L_HIP(ctx, hipMemcpyAsync(ws.h_count, running, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        GF2L_HIP(ctx, hipStreamSynchronize(s));
        const uint32_t left = ws.h_count[0];
        if (left == 0) break;
        const uint32_t packed = (left + 63u) / 64u;
        if (packed * 2u <= groups) {
            const uint32_t to = cur ^ 1u;
            hipLaunchKernelGGL(group_pack_kernel, dim3(1), dim3(1024), 0, s, active[out], groups, map[cur], map[to],
                               src, left);
            const uint32_t g_move = std::max<uint32_t>(1, std::min<uint32_t>(1024u, (uint32_t)ctx->num_cus * 8u / packed));
            auto move = [&](const float *from, float *dest, uint64_t *masks, uint32_t rows) {
                hipLaunchKernelGGL(group_move_kernel, dim3(g_move, packed), dim3(256), 0, s, src, from, dest, masks, rows);
            };
            move(c2v[cur], c2v[to], nullptr, cv.nnz);
            move(bel[cur], bel[to], hb[out], cv.n);
            move(llr[cur], llr[to], nullptr, cv.n);
            GF2L_HIP(ctx, hipGetLastError());
            groups = packed;
            cur = to;
        }
    }
    GF2L_HIP(ctx, hipStreamSynchronize(s));
    return GF2L_OK;
}

static int group_buffers(gf2l_ctx *ctx, const CsrView &cv, uint32_t groups) {
    // lists ([2][frames]): frame maps of both regions, sources of a packing
    const size_t slots = (size_t)groups * 64u, both = group_slots(groups);
    return ensure_buffers(ctx, slots, both * cv.nnz, 0, both * cv.n,
                          (size_t)groups * (2 * (size_t)cv.n + 2 + group_grid_most(ctx)), both * cv.n);
}

// Decoder driver of the CSR path (same semantics as decode_device's plain
// min-sum): device buffers, synchronizes the stream once per iteration.
int decode_csr(gf2l_ctx *ctx, const gf2l_code *code, const float *d_llr, uint32_t F, uint32_t max_it,
               uint64_t *d_msg, uint32_t *d_iters, uint8_t *d_conv, uint8_t *d_synd) {
    const CsrView &cv = code->csr;
    if (use_groups(cv, F) && ctx->tune.frame_kernel != 1) {
        const uint32_t pass = std::min(groups_per_pass(ctx, cv), (uint32_t)(((uint64_t)F + 63u) / 64u));
        if (group_buffers(ctx, cv, pass) == GF2L_OK) {
            const size_t kw = (cv.k + 63u) / 64u;
            for (uint64_t f0 = 0; f0 < F; f0 += 64ull * pass) {
                const int rc = decode_csr_groups(ctx, code, d_llr + (size_t)f0 * cv.n,
                                                 (uint32_t)std::min<uint64_t>(F - f0, 64ull * pass), max_it,
                                                 d_msg + f0 * kw, d_iters + f0, d_conv + f0, d_synd + f0);
                if (rc != GF2L_OK) return rc;
            }
            return GF2L_OK;
        }
        hipGetLastError();  // no memory for the groups: the frames' own arrays are smaller
    }
    hipStream_t s = ctx->stream;
    const size_t nw = (cv.n + 63) / 64;
    const uint32_t syn_threads = std::min(kSynThreads, std::max(1u, (cv.m + 63u) / 64u) * 64u);
    // the context's reusable workspace: c2v [F][nnz], beliefs [F][n], hard bits [F][nw]
    const int rc = ensure_buffers(ctx, F, (size_t)F * std::max<uint64_t>(cv.nnz, 1), 0, (size_t)F * cv.n,
                                  (size_t)F * nw, 0);
    if (rc != GF2L_OK) return rc;
    Workspace &ws = ctx->ws;
    float *c2v = ws.c2v, *bel = ws.belief;
    uint64_t *hb = ws.hb;
    uint32_t *lists = ws.lists, *counts = ws.counts, *h_count = ws.h_count;
    GF2L_HIP(ctx, hipMemcpyAsync(bel, d_llr, (size_t)F * cv.n * sizeof(float), hipMemcpyDeviceToDevice, s));
    GF2L_HIP(ctx, hipMemsetAsync(c2v, 0, (size_t)F * cv.nnz * sizeof(float), s));
    hipLaunchKernelGGL(csr_init_kernel, dim3((F + 255) / 256), dim3(256), 0, s, lists, counts, F);
    GF2L_HIP(ctx, hipGetLastError());
    const uint32_t grid = (uint32_t)ctx->num_cus * 4u;
    for (uint32_t it = 1; it <= max_it; ++it) {
        const uint32_t cur = (it - 1) & 1u, nxt = it & 1u;
        const uint32_t *list = lists + (size_t)cur * F;
        hipLaunchKernelGGL(cn_csr_kernel, dim3(grid), dim3(256), 0, s, cv, list, counts + cur, c2v, bel);
        hipLaunchKernelGGL(vn_csr_kernel, dim3(grid), dim3(256), 0, s, cv, list, counts + cur, c2v, bel,
                           d_llr, hb, counts + nxt);
        const uint32_t g_syn = std::min<uint32_t>(F, (uint32_t)ctx->num_cus * 8u);
        hipLaunchKernelGGL(syn_csr_kernel, dim3(g_syn), dim3(syn_threads), nw * sizeof(uint64_t), s, cv, list,
                           counts + cur, lists + (size_t)nxt * F, counts + nxt, hb, it, (int)(it == max_it),
                           d_msg, d_iters, d_conv, d_synd);
        GF2L_HIP(ctx, hipGetLastError());
        GF2L_HIP(ctx, hipMemcpyAsync(h_count, counts + nxt, sizeof(uint32_t), hipMemcpyDeviceToHost, s));
        GF2L_HIP(ctx, hipStreamSynchronize(s));
        if (*h_count == 0) break;
    }
    GF2L_HIP(ctx, hipStreamSynchronize(s));
    return GF2L_OK;
}

}  // namespace gf2l

using gf2l::fail;

extern "C" int gf2l_code_edges(gf2l_ctx *ctx, uint32_t m, uint32_t n, const uint32_t *rc_pairs,
                               size_t nnz, gf2l_code **out) {
    if (!ctx || !out) return GF2L_ERR_INVALID;
    *out = nullptr;
    return gf2l::guard(ctx, [&]() -> int {
        // SpBitMatrix::from_coo (sparse.rs:166-204): bounds checks, per-row sort,
        // duplicates cancel in pairs; then the stable transpose
        gf2l::host::Csr h;
        std::string err;
        const int hrc = gf2l::host::build_csr(m, n, rc_pairs, nnz, h, err);
        if (hrc != GF2L_OK) return fail(ctx, hrc, err);
        if (h.max_dc > gf2l::kMaxCheckDegree) return fail(ctx, GF2L_ERR_UNSUPPORTED, "check degree above 32");
        const std::vector<uint32_t> &row_ptr = h.row_ptr, &col_idx = h.col_idx, &col_ptr = h.col_ptr,
                                    &csc_edge = h.csc_edge;
        const uint32_t max_dc = h.max_dc;
        const uint32_t E = (uint32_t)col_idx.size();
        GF2L_HIP(ctx, hipSetDevice(ctx->device));
        const size_t b_rp = ((size_t)m + 1) * 4, b_ci = (size_t)std::max(E, 1u) * 4, b_cp = ((size_t)n + 1) * 4;
        auto al = [](size_t x) { return (x + 15) & ~(size_t)15; };
        const size_t o_ci = al(b_rp), o_cp = al(o_ci + b_ci), o_ce = al(o_cp + b_cp), total = o_ce + b_ci;
        std::vector<char> host(total, 0);
        std::memcpy(host.data(), row_ptr.data(), b_rp);
        if (E) std::memcpy(host.data() + o_ci, col_idx.data(), (size_t)E * 4);
        std::memcpy(host.data() + o_cp, col_ptr.data(), b_cp);
        if (E) std::memcpy(host.data() + o_ce, csc_edge.data(), (size_t)E * 4);
        gf2l_code *c = new gf2l_code;
        c->device = ctx->device;
        c->is_csr = true;
        hipError_t he = hipMalloc(&c->d_tables, total);
        if (he == hipSuccess) he = hipMemcpy(c->d_tables, host.data(), total, hipMemcpyHostToDevice);
        if (he != hipSuccess) {
            hipFree(c->d_tables);
            delete c;
            return fail(ctx, GF2L_ERR_HIP, std::string("code upload: ") + hipGetErrorString(he));
        }
        char *d = static_cast<char *>(c->d_tables);
        gf2l::CsrView &v = c->csr;
        v.m = m;
        v.n = n;
        v.k = n > m ? n - m : 0;
        v.nnz = E;
        v.row_ptr = reinterpret_cast<const uint32_t *>(d);
        v.col_idx = reinterpret_cast<const uint32_t *>(d + o_ci);
        v.col_ptr = reinterpret_cast<const uint32_t *>(d + o_cp);
        v.csc_edge = reinterpret_cast<const uint32_t *>(d + o_ce);
        // the QC view stays empty except the sizes used by the generic helpers
        c->view = gf2l::CodeView{};
        c->view.n = n;
        c->view.m = m;
        c->view.k = v.k;
        c->view.max_dc = max_dc;
        *out = c;
        return GF2L_OK;
    });
}
