// Whole-frame flooding min-sum decoder of small quasi-cyclic codes: the LDS
// path (one workgroup per frame, all iterations in one launch) with the work
// laid out so that nothing but the update itself is left in the loop.  Same
// operations in the same order as the other paths (bit-exact with
// decode_iterative, crates/gf2-coding/src/ldpc/core.rs:889-938).
//
// The m lifted checks and the n variables are dealt to the T threads in turn
// (thread t has checks t, t + T, ... and variables t, t + T, ...), whatever the
// lift, so no lane idles at the end of a block-row.  A thread keeps its checks
// for the whole call:
//   - the LDS addresses of their inputs and messages are computed once per
//     launch and stay in registers;
//   - their states (12 bytes) and the LLRs of its variables stay in registers;
//   - a message is written to LDS where the variable update reads it: the
//     column-order edge list, one row of z floats per block edge, so a
//     variable's messages lie z floats apart in ascending check order.
// Missing inputs (a row with fewer than DMAX, a thread's last checks) read a
// +infinity, which a check does not notice, and write to an unused word, so no
// access is guarded.  Two barriers an iteration.  The check pass also takes the
// parity of its inputs' hard decisions, the syndrome of the iteration before.
//
// Signs of zeros and the selection of the two minima are as in the large
// codes' kernel (flood.hip).  A frame with an LLR or a belief of magnitude 1e30
// or more, infinite or NaN is decoded (again) with SAFE set: a NaN input counts
// as +infinity, which is what the general rule's comparisons make of it, and
// hard decisions are comparisons.
//
// What bounds it: vector issue and, with the 12 waves per compute unit that
// 115 registers and 6-wave workgroups leave, LDS latency.  N=2304 (T = 384),
// 16384 frames at 2.0 dB: 1,987 vector and 395 LDS instructions per
// frame-iteration (6,915 and 887 in lds_decode_kernel), 1.21 ms against 2.65 ms;
// 1024 frames 158 against 427 us, one frame 44 against 99 us.  Measured and left
// out: registers for five waves per SIMD (20 spilled), 1.30 ms; input and
// output addresses as halves of one register, 1.31 ms.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"

namespace gf2l {
namespace {

constexpr uint32_t kChecks = 3, kVars = 6;  // checks and variables per thread
constexpr float kSmallLimit = 1e30f;

__device__ __forceinline__ bool too_large(float v) { return !(fabsf(v) < kSmallLimit); }

// One thread's part of the code.
template <int DMAX>
struct SmallPart {
    uint32_t in[kChecks][DMAX], out[kChecks][DMAX];  // LDS byte addresses
    uint32_t var[kVars];   // messages << 16 | word of the first
    uint32_t most[kVars];  // largest message count of the wave | 0x80 when all lanes have it (uniform)
    uint32_t a_bel, a_unused, n, T;

    // Belief of this thread's k-th variable (the unused word past the last one).
    __device__ uint32_t bel(uint32_t k) const {
        const uint32_t v = threadIdx.x + k * T;
        return v < n ? a_bel + 4u * v : a_unused;
    }
};

// Check pass: new states and (update) messages; returns whether a check of
// this thread is unsatisfied by the beliefs' hard decisions.
template <int DMAX, bool SAFE>
__device__ __forceinline__ bool small_checks(const SmallPart<DMAX> &P, uint3 *st, bool update) {
    uint32_t unsat = 0;
    float b[kChecks][DMAX];  // every read of the pass issued before the first use
#pragma unroll
    for (uint32_t k = 0; k < kChecks; ++k)
#pragma unroll
        for (int p = 0; p < DMAX; ++p) b[k][p] = lds_ld(P.in[k][p]);
#pragma unroll
    for (uint32_t k = 0; k < kChecks; ++k) {
        uint32_t par = 0;
#pragma unroll
        for (int p = 0; p < DMAX; ++p) par ^= SAFE ? (b[k][p] < 0.0f ? 0x80000000u : 0u) : __float_as_uint(b[k][p]);
        unsat |= par;
    }
    if (!update) return (unsat >> 31) != 0;
#pragma unroll
    for (uint32_t k = 0; k < kChecks; ++k) {
        float x[DMAX];
        const float m1o = __uint_as_float(st[k].x), m2o = __uint_as_float(st[k].y);
        const uint32_t mo = st[k].z, io = mo & 31u;
#pragma unroll
        for (int p = 0; p < DMAX; ++p) {
            const float mag = (uint32_t)p == io ? m2o : m1o;
            x[p] = b[k][p] - __uint_as_float(__float_as_uint(mag) ^ ((mo << (27 - DMAX + p)) & 0x80000000u));
            if constexpr (SAFE) x[p] = x[p] == x[p] ? x[p] : __builtin_inff();
        }
        float m1 = __builtin_fminf(fabsf(x[0]), fabsf(x[1])), m2 = __builtin_fmaxf(fabsf(x[0]), fabsf(x[1]));
#pragma unroll
        for (int p = 2; p < DMAX; ++p) {
            const float a = fabsf(x[p]);
            m2 = __builtin_amdgcn_fmed3f(m1, a, m2);
            m1 = __builtin_fminf(m1, a);
        }
        uint32_t sg = 0, idx = 0;
#pragma unroll
        for (int p = 0; p < DMAX; ++p) sg = __builtin_amdgcn_alignbit(sg, __float_as_uint(x[p]), 31);
        const uint32_t all = (uint32_t)__popc(sg) << 31;
        const uint32_t m1s = __float_as_uint(m1) ^ all, m2s = __float_as_uint(m2) ^ all;
#pragma unroll
        for (int p = 0; p < DMAX; ++p) {
            const bool is1 = fabsf(x[p]) == m1;
            idx = is1 ? (uint32_t)p : idx;
            lds_st(P.out[k][p], __uint_as_float((is1 ? m2s : m1s) ^ (__float_as_uint(x[p]) & 0x80000000u)));
        }
        st[k] = make_uint3(m1s, m2s, idx | (sg << 5));
    }
    return (unsat >> 31) != 0;
}

// Variable pass: belief = LLR + messages in ascending check order.  Returns
// the lanes with a belief too large.
template <int DMAX>
__device__ __forceinline__ uint64_t small_vars(const SmallPart<DMAX> &P, const float *llr, uint32_t z4) {
    uint64_t big = 0;
#pragma unroll
    for (uint32_t k = 0; k < kVars; ++k) {
        const uint32_t d = P.most[k] & 0x7fu;
        float v = llr[k];
        uint32_t ad = 4u * (P.var[k] & 0xffffu);
        if (P.most[k] & 0x80u) {
            uint32_t q = 0;
            for (; q + 3 <= d; q += 3) {
                const float c0 = lds_ld(ad), c1 = lds_ld(ad + z4), c2 = lds_ld(ad + 2u * z4);
                v = v + c0;
                v = v + c1;
                v = v + c2;
                ad += 3u * z4;
            }
            for (; q < d; ++q, ad += z4) v = v + lds_ld(ad);
        } else {
            const uint32_t own = P.var[k] >> 16;
            for (uint32_t q = 0; q < d; ++q, ad += z4) {
                const float c = q < own ? lds_ld(ad) : 0.0f;
                if (q < own) v = v + c;
            }
        }
        big |= __builtin_amdgcn_ballot_w64(too_large(v));
        lds_st(P.bel(k), v);
    }
    return big;
}

// Decodes the frame whose LLRs (canonical: no -0) are in `llr` and in the
// beliefs.  Returns the iterations, or ~0u when a belief grows too large.
// flag: four LDS words (zero on entry): unsatisfied and too large, each of the
// even and the odd passes.
template <int DMAX, bool SAFE>
__device__ __forceinline__ uint32_t small_decode(const SmallPart<DMAX> &P, const float *llr, uint32_t z4,
                                                 uint32_t max_it, lds_u32 *flag, bool &conv) {
    // the first messages are -0: x = b - (-0) = b + 0
    uint3 st[kChecks];
#pragma unroll
    for (uint32_t k = 0; k < kChecks; ++k) st[k] = make_uint3(0x80000000u, 0x80000000u, 0u);
    uint64_t big = 0;
    for (uint32_t it = 1;; ++it) {
        const bool update = it <= max_it;  // the pass after the last iteration only checks it
        const bool unsat = small_checks<DMAX, SAFE>(P, st, update);
        const uint64_t u = __builtin_amdgcn_ballot_w64(unsat);
        if ((threadIdx.x & 63u) == 0) {
            if (u) flag[it & 1u] = 1u;
            if (big) flag[2u + (it & 1u)] = 1u;
        }
        lds_barrier();
        const uint32_t f = uni(flag[it & 1u]), fb = uni(flag[2u + (it & 1u)]);
        if (!SAFE && fb) return ~0u;
        if (it > 1 && !f) {  // iteration it - 1 satisfied every check
            conv = true;
            return it - 1;
        }
        if (!update) {
            conv = false;
            return max_it;
        }
        if (threadIdx.x < 2) flag[((it + 1) & 1u) + 2u * threadIdx.x] = 0;
        big = small_vars<DMAX>(P, llr, z4);
        lds_barrier();
    }
}

template <int DMAX>
__global__ void __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(4))) small_kernel(CodeView cv, const float *__restrict__ llr, uint32_t frames,
                                                     uint32_t max_it, uint64_t *__restrict__ msg,
                                                     uint32_t *__restrict__ iters, uint8_t *__restrict__ conv_out,
                                                     uint8_t *__restrict__ synd, uint32_t *ctr) {
    extern __shared__ __align__(16) float sm[];
    __shared__ uint32_t s_flag[4], s_f;
    const uint32_t z = cv.z, E = cv.nbe * z, n = cv.n, T = blockDim.x, t = threadIdx.x;
    // [nbe][z] messages in column order, [n] beliefs, +infinity, unused word
    const uint32_t a_msg = (uint32_t)(size_t)(lds_float *)sm, a_bel = a_msg + 4u * E, a_inf = a_bel + 4u * n,
                   a_unused = a_inf + 4u;
    lds_u32 *flag = (lds_u32 *)s_flag;
    const uint32_t kw = (cv.k + 63) / 64, lane = t & 63u;
    // place in the column order of every block edge, in the message area
    uint32_t *inv = reinterpret_cast<uint32_t *>(sm);
    for (uint32_t q = t; q < cv.nbe; q += T) inv[cv.col_edge[q].x] = q;
    if (t == 0) sm[E + n] = __builtin_inff();
    __syncthreads();
    SmallPart<DMAX> P;
    P.a_bel = a_bel;
    P.a_unused = a_unused;
    P.n = n;
    P.T = T;
#pragma unroll
    for (uint32_t k = 0; k < kChecks; ++k) {
        const uint32_t c = t + k * T, r = c / z, i = c - r * z;
        const uint32_t e0 = c < cv.m ? cv.row_ptr[r] : 0u, d = c < cv.m ? cv.row_ptr[r + 1] - e0 : 0u;
#pragma unroll
        for (int p = 0; p < DMAX; ++p) {
            P.in[k][p] = a_inf;
            P.out[k][p] = a_unused;
            if (p < (int)d) {
                const uint2 re = cv.row_edge[e0 + p];
                const uint32_t j = wrap_add(i, re.y, z);
                P.in[k][p] = a_bel + 4u * (re.x * z + j);
                P.out[k][p] = a_msg + 4u * (inv[e0 + p] * z + j);
            }
        }
    }
#pragma unroll
    for (uint32_t k = 0; k < kVars; ++k) {
        const uint32_t v = t + k * T, bc = v / z, j = v - bc * z;
        const uint32_t q0 = v < n ? cv.col_ptr[bc] : 0u, own = v < n ? cv.col_ptr[bc + 1] - q0 : 0u;
        P.var[k] = (a_msg / 4u + q0 * z + j) | (own << 16);
        uint32_t most = own;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, o, 64));
        P.most[k] = uni(most | (__builtin_amdgcn_ballot_w64(own != most) == 0 ? 0x80u : 0u));
    }
    __syncthreads();  // inv is done with the message area
    for (uint32_t f = blockIdx.x;;) {
        if (f >= frames) break;
        const float *fl = llr + (size_t)f * n;
        float L[kVars];
        uint64_t big = 0;
#pragma unroll
        for (uint32_t k = 0; k < kVars; ++k) {
            const uint32_t v = t + k * T;
            L[k] = (v < n ? fl[v] : 0.0f) + 0.0f;  // -0 as +0
            big |= __builtin_amdgcn_ballot_w64(too_large(L[k]));
            lds_st(P.bel(k), L[k]);
        }
        if (t < 4) flag[t] = 0;
        if (t == 0) s_f = ctr ? gridDim.x + atomicAdd(ctr, 1u) : f + gridDim.x;  // the frame after this one
        const bool plain = __syncthreads_or(big != 0) == 0;
        bool conv = false;
        uint32_t its = ~0u;
        if (plain) its = small_decode<DMAX, false>(P, L, 4u * z, max_it, flag, conv);
        if (its == ~0u) {  // from the LLRs, with every special value minded
            __syncthreads();
#pragma unroll
            for (uint32_t k = 0; k < kVars; ++k) lds_st(P.bel(k), L[k]);
            if (t < 4) flag[t] = 0;
            __syncthreads();
            its = small_decode<DMAX, true>(P, L, 4u * z, max_it, flag, conv);
        }
        // message words: T is a multiple of 64, so a wave holds whole words
#pragma unroll
        for (uint32_t k = 0; k < kVars; ++k) {
            const uint32_t v = t + k * T;
            const uint64_t word = __ballot(v < cv.k && lds_ld(P.bel(k)) < 0.0f);
            if (lane == 0 && v < cv.k) msg[(size_t)f * kw + v / 64u] = word;
        }
        if (t == 0) {
            iters[f] = its;
            conv_out[f] = (uint8_t)conv;
            synd[f] = (uint8_t)conv;
        }
        const uint32_t next = uni(s_f);
        __syncthreads();  // the beliefs and s_f have been read
        f = next;
    }
    // the last workgroup leaves the counters at zero for the next launch
    if (ctr && t == 0) {
        __threadfence();
        if (atomicAdd(ctr + 1, 1u) == gridDim.x - 1u) {
            ctr[0] = 0;
            ctr[1] = 0;
        }
    }
}

size_t small_bytes(const CodeView &cv) { return ((size_t)cv.nbe * cv.z + cv.n + 2) * sizeof(float); }

}  // namespace

uint32_t small_threads(const gf2l_code *code) {
    const CodeView &cv = code->view;
    if (code->is_csr || cv.dvb_q || cv.max_dc > 8 || cv.n == 0 || small_bytes(cv) > 80 * 1024) return 0;
    for (uint32_t br = 0; br < cv.mb; ++br)
        if (code->h_row_ptr[br + 1] - code->h_row_ptr[br] < 2) return 0;  // a lone input's message is 0
    for (uint32_t t = 64; t <= 1024; t += 64)
        if (cv.m <= kChecks * t && cv.n <= kVars * t && cv.max_dv < 0x80u) return t;
    return 0;
}

hipError_t launch_small(const CodeView &cv, uint32_t threads, const float *llr, uint32_t frames, uint32_t max_it,
                        uint64_t *msg, uint32_t *iters, uint8_t *conv, uint8_t *synd, uint32_t *ctr, int num_cus,
                        hipStream_t s) {
    if (frames == 0) return hipSuccess;
    const size_t bytes = small_bytes(cv);
    const uint32_t waves = threads / 64u;
    // 16 waves are resident; a workgroup more per compute unit waits and takes
    // over where one ends early
    const uint32_t per_cu =
        (uint32_t)std::max<size_t>(1, std::min<size_t>(20u / waves, (160 * 1024) / (bytes + 256)));
    const uint32_t grid = std::min<uint32_t>(frames, (uint32_t)num_cus * per_cu);
    auto k = cv.max_dc <= 6 ? small_kernel<6> : small_kernel<8>;
    if (bytes > 65536) {
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(k),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(k, dim3(grid), dim3(threads), bytes, s, cv, llr, frames, max_it, msg, iters, conv, synd,
                       grid < frames ? ctr : nullptr);
    return hipGetLastError();
}

}  // namespace gf2l
