// Team kernel: a whole plain min-sum decode in one launch, a frame spread over a
// team of workgroups that meet twice an iteration (a batch that fills the chip
// has teams of one).
//
// A frame's iteration is a check pass and a variable pass with every edge
// crossing between them.  As kernels of their own they cost four launches and
// four drains of the chip an iteration (check, variable, syndrome, list: 13, 21,
// 8 and 4 us for one frame of N = 64800), for work of a few microseconds; that
// chain bounds a small batch.  Here the workgroups of a team stay on their
// compute units: check states and channel LLRs stay in LDS with the threads that
// own them (the LLRs in memory where LDS is short), messages (4 bytes an edge)
// and beliefs pass through memory, and a counter per team replaces the launches.
// The syndrome of an iteration is taken by the next check pass, which reads the
// beliefs anyway.  One frame of N = 64800: 850 -> 200 us at 22 iterations; 24
// frames: 1440 -> 480 us, bound by the exchange (3.4 MB a frame and iteration at
// 5 TB/s).
//
// Exchange: a team's workgroups may sit on different XCDs (workgroup b on XCD
// b % 8: they all share one only where the number of teams is a multiple of 8),
// whose L2s are not coherent within a kernel, so messages and beliefs are stored
// and loaded at agent scope, and a workgroup reports to the counter when its
// stores are done.
// Plain loads with an acquire fence at each meeting were slower (24 frames: 1.93
// ms, each fence drops the caches of the whole XCD).
//
// A team of one (SOLO) needs none of that: check states in LDS stand for the
// messages, beliefs stay in the XCD's L2, and meetings are barriers.  DVB-T2
// short r 1/2, 1000 frames: 5.0 -> 3.3 ms.
//
// A list of frames that the state kernels have run for one iteration goes on from
// their states and beliefs, in the same rows (RESUME: DVB-T2 normal r 2/3, 1000
// frames at the waterfall 15.0 -> 14.5 ms, 3 dB above it 3.68 -> 3.28).  With check
// degrees past 16 the two ways into the loop leave 18 registers to memory: such
// codes start again from the LLRs (r 4/5, 1000 frames 12.1 ms, resumed 14.0).
//
// Waiting is safe only when the whole team is resident.  The grid has at most
// one workgroup per compute unit, but other work may hold some of them: every
// wait is bounded, a team that does not meet in time marks the counter and
// leaves, and the caller decodes the batch by the general kernels.
//
// Same arithmetic as the state kernels: message = sign product * min of the
// other inputs, belief = LLR + messages in ascending check order.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_common.h"
#include "internal.h"

namespace gf2l {
namespace {

constexpr uint32_t kTeamThreads = 1024, kTeamWaves = kTeamThreads / 64;
constexpr int kTeamDv = 16;   // largest variable degree
constexpr int kTeamDc = 27;   // largest check degree (position and signs of a state in one word)
constexpr uint64_t kGaveUp = 1ull << 63;
constexpr int kTeamResumeDc = 16;  // largest degree class that goes on from states

template <bool SOLO>
__device__ __forceinline__ float ld_shared(const float *p, uint32_t i) {
    if constexpr (SOLO) return ldu(p, i);
    return __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <bool SOLO>
__device__ __forceinline__ void st_shared(float *p, uint32_t i, float v) {
    if constexpr (SOLO) {
        stu(p, i, v);
        return;
    }
    __hip_atomic_store(p + i, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// DVB belief sum at lane j of a block-column with nonzero shifts: the messages
// c, rotated so that slots whose check lane wrapped come first.  wrap: the
// column of the staircase's last parity bits, which has no edge from check 0
// (slots row0) to its last lane.  The same order as vn_state_item's, which keeps
// a copy inside its kernel (called from there it cost the kernel 40%).
template <int D, int N>
__device__ __forceinline__ float dvb_rotated_sum(float bel, float (&c)[N], const uint32_t *thr, uint32_t j, bool wrap,
                                                 bool last_lane, uint32_t row0) {
    constexpr int DA = N;
    uint32_t r = 0;
#pragma unroll
    for (int q = 0; q < D; ++q) r += (j < thr[q]) ? 1u : 0u;
#pragma unroll
    for (int k = 1; k < D; k <<= 1) {
        const bool rot = (r & (uint32_t)k) != 0;
        float t[DA];
#pragma unroll
        for (int q = 0; q < D; ++q) t[q] = rot ? c[(q + k) % DA] : c[q];
#pragma unroll
        for (int q = 0; q < D; ++q) c[q] = t[q];
    }
    if (wrap) {
        constexpr uint64_t full = D >= 64 ? ~0ull : (1ull << D) - 1;
        uint64_t live = full & ~(last_lane ? (uint64_t)row0 : 0ull);
        const uint32_t rr = r % (uint32_t)DA;
        live = ((live >> rr) | (live << ((DA - rr) % 64))) & full;
#pragma unroll
        for (int q = 0; q < D; ++q)
            if ((live >> q) & 1ull) bel = bel + c[q];
    } else {
#pragma unroll
        for (int q = 0; q < D; ++q) bel = bel + c[q];
    }
    return bel;
}

// The team meets: stores before it are seen by loads after it.  `bad` (any
// thread's) is counted in the upper word.  Returns the counter as every
// member sees it; kGaveUp set: leave.
template <bool SOLO>
__device__ __forceinline__ uint64_t team_meet(const TeamArgs &a, uint64_t *sync, uint32_t meeting, bool bad,
                                              uint32_t wait, uint64_t *s_word) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int any = __syncthreads_or(bad);
    if constexpr (SOLO) return any ? 1ull << 32 : 0ull;
    if (threadIdx.x == 0) {
        const uint32_t all = meeting * a.team;
        uint64_t v = __hip_atomic_fetch_add(sync, 1ull + (any ? 1ull << 32 : 0ull), __ATOMIC_RELAXED,
                                            __HIP_MEMORY_SCOPE_AGENT);
        const uint64_t t0 = wall_clock64();
        for (;;) {
            v = __hip_atomic_load(sync, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((v & kGaveUp) || (uint32_t)v >= all) break;
            if (wall_clock64() - t0 > wait) {
                __hip_atomic_fetch_or(sync, kGaveUp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(a.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                v |= kGaveUp;
                break;
            }
            __builtin_amdgcn_s_sleep(1);
        }
        *s_word = v;
    }
    __syncthreads();
    return *s_word;
}

template <int MAXC, bool DVB, bool SOLO, bool RESUME>
__global__ void __launch_bounds__(kTeamThreads)
team_kernel(TeamArgs a) {
    extern __shared__ uint32_t lds[];
    __shared__ uint64_t s_word;
    const CodeView &cv = a.cv;
    const uint32_t team = blockIdx.x % a.teams, member = blockIdx.x / a.teams;
    const uint32_t lane = threadIdx.x & 63u, id = uni(threadIdx.x >> 6) * a.team + member;
    const uint32_t waves = kTeamWaves * a.team;
    const uint32_t c_items = cv.mb * cv.zw, v_items = cv.nb * cv.zw;
    const uint32_t c_rounds = (c_items + waves - 1) / waves;
    const uint32_t plane = c_rounds * kTeamThreads;  // check states: three planes [c_rounds][threads]
    // [v_rounds][threads], in LDS or (llr_lds 0) in memory
    float *own_llr = reinterpret_cast<float *>(lds + c_rounds * 3u * kTeamThreads) + threadIdx.x;
    const uint32_t v_rounds = (v_items + waves - 1) / waves;
    float *mem_llr = a.llr_own + (size_t)blockIdx.x * v_rounds * kTeamThreads + threadIdx.x;
    float *msg = a.msg + (size_t)team * cv.nbe * cv.zp, *bel = a.bel + (size_t)team * cv.nb * cv.zp;
    uint64_t *sync = a.sync + (size_t)team * kTeamSyncStride;
    uint32_t meeting = 0, wait = a.first_wait;
    uint32_t bad_before = 0;  // upper word of the counter after the last check pass
    const uint32_t kw = (cv.k + 63u) / 64u;

    uint32_t next = a.frames;
    for (uint32_t slot = team; slot < a.frames; slot = next) {
        const uint32_t f = a.list ? ldc(a.list + slot) : slot;
        // the team's next frame, from the batch's counter: taken here by the
        // first member, read by all after the first meeting
        const bool more = a.frames > a.teams;
        if (more && member == 0 && threadIdx.x == 0) {
            const uint32_t n = a.teams + __hip_atomic_fetch_add(a.queue, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(sync + 8, (uint64_t)n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        const float *fl = a.llr + (size_t)f * cv.n;
        // LLR of lane j of a block-column, from the caller's order
        auto llr_at = [&](uint32_t bc, uint32_t j) {
            if (DVB && bc >= cv.dvb_kb) return ldu(fl, cv.k + (bc - cv.dvb_kb) + cv.dvb_q * j);
            return ldu(fl, bc * cv.z + j);
        };
        for (uint32_t item = id, r = 0; item < v_items; item += waves, ++r) {
            const uint32_t bc = item / cv.zw, j = (item - bc * cv.zw) * 64u + lane;
            const float l = j < cv.z ? llr_at(bc, j) : 0.0f;
            if (a.llr_lds)
                own_llr[r * kTeamThreads] = l;
            else
                mem_llr[r * kTeamThreads] = l;
        }
        if constexpr (RESUME) {  // states and beliefs of iteration 1, from the frame's rows
            bel = a.bel + (size_t)f * cv.nb * cv.zp;
            const uint3 *st = a.state + (size_t)f * cv.mb * cv.zp;
            for (uint32_t item = id, r = 0; item < c_items; item += waves, ++r) {
                const uint32_t br = item / cv.zw, i = (item - br * cv.zw) * 64u + lane;
                if (i >= cv.z) continue;
                const uint3 o = ldu(st, br * cv.zp + i);
                uint32_t *own = lds + (r * kTeamThreads + threadIdx.x);
                own[0] = o.x;
                own[plane] = o.y;
                own[2 * plane] = o.z;
            }
        }
        uint64_t word = 0;
        bool unsat = true;
        constexpr uint64_t it0 = RESUME ? 2 : 1;
        uint64_t it = it0;
        for (;; ++it) {
            bool bad = false;
            for (uint32_t item = id, r = 0; item < c_items; item += waves, ++r) {
                const uint32_t br = item / cv.zw, i = (item - br * cv.zw) * 64u + lane;
                const uint32_t e0 = uni(ldc(cv.row_ptr + br)), d = uni(ldc(cv.row_ptr + br + 1)) - e0;
                uint32_t *own = lds + (SOLO ? br * cv.zp + i : r * kTeamThreads + threadIdx.x);
                dispatch_degree<MAXC>(d, [&](auto DC) {
                    constexpr int D = decltype(DC)::value, DA = D > 0 ? D : 1;
                    if (i >= cv.z) return;
                    uint2 re[DA];
#pragma unroll
                    for (int p = 0; p < D; ++p) {
                        const uint2 e = ldc(cv.row_edge + e0 + p);
                        re[p] = make_uint2(uni(e.x), uni(e.y));
                    }
                    float x[DA];
                    if (!RESUME && it == 1) {
#pragma unroll
                        for (int p = 0; p < D; ++p) x[p] = llr_at(re[p].x, wrap_add(i, re[p].y, cv.z));
                    } else {
#pragma unroll
                        for (int p = 0; p < D; ++p) x[p] = ld_shared<SOLO>(bel, re[p].x * cv.zp + wrap_add(i, re[p].y, cv.z));
                    }
                    uint32_t skip = D;  // DVB: check 0 has no staircase edge to the last parity bit
                    if (DVB && br == 0 && i == 0) {
#pragma unroll
                        for (int p = 0; p < D; ++p)
                            if (re[p].x == cv.wrap_bc) skip = p;
                    }
                    if (RESUME || it > 1) {
                        const float m1 = __uint_as_float(own[0]), m2 = __uint_as_float(own[plane]);
                        const uint32_t meta = own[2 * plane];
                        uint32_t par = 0;
#pragma unroll
                        for (int p = 0; p < D; ++p) {
                            if (!DVB || (uint32_t)p != skip) par ^= x[p] < 0.0f ? 1u : 0u;
                            x[p] = x[p] - recon_or(m1, m2, meta, p);
                        }
                        bad = bad || par;
                    }
                    float m1, m2;
                    uint32_t meta;
                    if constexpr (D <= 8) {
                        // no full 8-lane chunk among the other inputs: a sign is `< 0` everywhere
                        m1 = m2 = __builtin_inff();
                        uint32_t idx = 0, lt = 0;
#pragma unroll
                        for (int p = 0; p < D; ++p) {
                            if (DVB && (uint32_t)p == skip) continue;
                            const float v = fabsf(x[p]);
                            const bool lt1 = v < m1, lt2 = v < m2;
                            m2 = lt1 ? m1 : (lt2 ? v : m2);
                            m1 = lt1 ? v : m1;
                            idx = lt1 ? (uint32_t)p : idx;
                            lt |= (x[p] < 0.0f ? 1u : 0u) << p;
                        }
                        meta = idx | ((((__popc(lt) & 1u) ? (1u << D) - 1u : 0u) ^ lt) << 5);
                    } else {
                        CheckAcc acc;
                        acc.init();
#pragma unroll
                        for (int p = 0; p < D; ++p) {
                            if (DVB && (uint32_t)p == skip) continue;
                            acc.add_sel(p, x[p]);
                        }
                        m1 = acc.min1;
                        m2 = acc.min2;
                        if constexpr (DVB)
                            meta = acc.idx | (dvb_signs<D>(cv, acc, cv.row_edge + e0, i, skip) << 5);
                        else
                            meta = acc.idx | (acc.signs<D>(D) << 5);
                    }
                    if constexpr (D == 1) {
                        m1 = 0.0f;
                        m2 = 0.0f;
                        meta = 0;
                    }
                    own[0] = __float_as_uint(m1);
                    own[plane] = __float_as_uint(m2);
                    own[2 * plane] = meta;
                    if constexpr (!SOLO) {
#pragma unroll
                        for (int p = 0; p < D; ++p) st_shared<SOLO>(msg, (e0 + p) * cv.zp + i, recon_or(m1, m2, meta, p));
                    }
                });
            }
            word = team_meet<SOLO>(a, sync, ++meeting, bad, wait, &s_word);
            wait = a.wait;
            if (word & kGaveUp) return;
            if (it == it0 && more)
                next = (uint32_t)__hip_atomic_load(sync + 8, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            unsat = (uint32_t)(word >> 32) != bad_before;
            if (!SOLO) bad_before = (uint32_t)(word >> 32);
            if ((RESUME || it > 1) && (!unsat || it > a.max_it)) break;

            for (uint32_t item = id, r = 0; item < v_items; item += waves, ++r) {
                const uint32_t bc = item / cv.zw, j = (item - bc * cv.zw) * 64u + lane;
                const uint32_t c0 = uni(ldc(cv.col_ptr + bc)), dv = uni(ldc(cv.col_ptr + bc + 1)) - c0;
                dispatch_degree<kTeamDv>(dv, [&](auto DC) {
                    constexpr int D = decltype(DC)::value, DA = D > 0 ? D : 1;
                    if (j >= cv.z) return;
                    float c[DA];
                    uint32_t sh[DA], row0 = 0;  // shifts; slots of block-row 0
                    if constexpr (SOLO) {
                        uint2 ce[DA];  // {block-row * zp, shift << 5 | position}
#pragma unroll
                        for (int q = 0; q < D; ++q) {
                            const uint2 e = ldc(cv.col_pack + c0 + q);
                            ce[q] = make_uint2(uni(e.x), uni(e.y));
                            sh[q] = ce[q].y >> 5;
                            row0 |= (ce[q].x == 0 ? 1u : 0u) << q;
                        }
#pragma unroll
                        for (int q = 0; q < D; ++q) {
                            const uint32_t *o = lds + (ce[q].x + wrap_sub(j, sh[q], cv.z));
                            c[q] = recon(__uint_as_float(o[0]), __uint_as_float(o[plane]), o[2 * plane], ce[q].y & 31u);
                        }
                    } else {
                        uint32_t e[DA];  // row-order edges
                        const uint32_t e_row1 = DVB ? uni(ldc(cv.row_ptr + 1)) : 0u;
#pragma unroll
                        for (int q = 0; q < D; ++q) {
                            const uint2 t = ldc(cv.col_edge + c0 + q);
                            e[q] = uni(t.x);
                            sh[q] = uni(t.y);
                            row0 |= (e[q] < e_row1 ? 1u : 0u) << q;
                        }
#pragma unroll
                        for (int q = 0; q < D; ++q) c[q] = ld_shared<SOLO>(msg, e[q] * cv.zp + wrap_sub(j, sh[q], cv.z));
                    }
                    float b = a.llr_lds ? own_llr[r * kTeamThreads] : mem_llr[r * kTeamThreads];
                    bool ordered = true;  // every lane sums in slot order
                    if constexpr (DVB) {
#pragma unroll
                        for (int q = 0; q < D; ++q) ordered = ordered && sh[q] == 0;
                    }
                    if (ordered) {
#pragma unroll
                        for (int q = 0; q < D; ++q) b = b + c[q];
                    } else if constexpr (DVB && D > 0) {
                        uint32_t thr[DA];
#pragma unroll
                        for (int q = 0; q < D; ++q) thr[q] = sh[q] ? sh[q] : cv.z;
                        b = dvb_rotated_sum<D>(b, c, thr, j, bc == cv.wrap_bc, j == cv.z - 1, row0);
                    }
                    st_shared<SOLO>(bel, bc * cv.zp + j, b);
                });
            }
            word = team_meet<SOLO>(a, sync, ++meeting, false, wait, &s_word);
            if (word & kGaveUp) return;
        }
        // the hard decisions of iteration it - 1
        for (uint32_t w = id; w < kw; w += waves) {
            const uint32_t v = 64u * w + lane, bc = v / cv.z;
            const bool one = v < cv.k && ld_shared<SOLO>(bel, bc * cv.zp + (v - bc * cv.z)) < 0.0f;
            const uint64_t bits = __builtin_amdgcn_ballot_w64(one);
            if (lane == 0) a.msg_out[(size_t)f * kw + w] = bits;
        }
        if (member == 0 && threadIdx.x == 0) {
            a.iters[f] = (uint32_t)(it - 1);
            a.conv[f] = a.synd[f] = (uint8_t)!unsat;
        }
    }
}

// LDS words of a thread in a team of g: check states, channel LLRs.
struct TeamRounds {
    size_t c, v;
};
TeamRounds team_rounds(const CodeView &cv, uint32_t g) {
    const size_t waves = (size_t)kTeamWaves * g;
    return {(cv.mb * cv.zw + waves - 1) / waves, (cv.nb * cv.zw + waves - 1) / waves};
}

}  // namespace

bool team_shape(const CodeView &cv, uint32_t frames, uint32_t max_it, int num_cus, size_t lds_limit, TeamArgs &a) {
    if (cv.max_dc > (uint32_t)kTeamDc || cv.max_dv > (uint32_t)kTeamDv || cv.mb == 0 || !frames) return false;
    const uint32_t cus = (uint32_t)num_cus;
    const size_t words = (lds_limit - 64) / (kTeamThreads * sizeof(uint32_t));
    // a wave per item of the check pass at most
    const uint32_t most = std::max(1u, (cv.mb * cv.zw + kTeamWaves - 1) / kTeamWaves);
    uint32_t g = std::max(1u, std::min(most, cus / std::min(frames, cus)));
    while (g <= cus && 3 * team_rounds(cv, g).c > words) ++g;
    if (g > cus) return false;
    const TeamRounds r = team_rounds(cv, g);
    a.team = g;
    a.teams = std::min(frames, cus / g);
    a.llr_lds = 3 * r.c + r.v <= words;
    a.llr_words = a.llr_lds ? 0 : (size_t)a.teams * g * r.v * kTeamThreads;
    a.lds = (uint32_t)((3 * r.c + (a.llr_lds ? r.v : 0)) * kTeamThreads * sizeof(uint32_t));
    // the counter's two words hold every meeting of a team
    const uint64_t most_frames = frames - a.teams + 1;
    return g == 1 || most_frames <= (1u << 31) / (((uint64_t)max_it + 1) * 2 * g);
}

bool team_resumes(const CodeView &cv) { return cv.dvb_q && cv.max_dc <= (uint32_t)kTeamResumeDc; }

hipError_t launch_team(const TeamArgs &a, hipStream_t s) {
    const uint32_t lds = a.lds;
#define GF2L_TEAM_AS(MD, DV, SO, RE)                                                                              \
    do {                                                                                                          \
        const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(team_kernel<MD, DV, SO, RE>),     \
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);           \
        if (e != hipSuccess) return e;                                                                            \
        hipLaunchKernelGGL((team_kernel<MD, DV, SO, RE>), dim3(a.team * a.teams), dim3(kTeamThreads), lds, s, a); \
    } while (0)
#define GF2L_TEAM(MD, DV)                    \
    do {                                     \
        if (a.team == 1)                     \
            GF2L_TEAM_AS(MD, DV, true, false);   \
        else if (DV && MD <= kTeamResumeDc && a.state) \
            GF2L_TEAM_AS(MD, DV, false, (DV && MD <= kTeamResumeDc)); \
        else                                 \
            GF2L_TEAM_AS(MD, DV, false, false);  \
    } while (0)
#define GF2L_TEAM_CLASS(DV)          \
    do {                             \
        if (a.cv.max_dc <= 8)        \
            GF2L_TEAM(8, DV);        \
        else if (a.cv.max_dc <= 16)  \
            GF2L_TEAM(16, DV);       \
        else                         \
            GF2L_TEAM(kTeamDc, DV);  \
    } while (0)
    if (a.cv.dvb_q)
        GF2L_TEAM_CLASS(true);
    else
        GF2L_TEAM_CLASS(false);
#undef GF2L_TEAM_CLASS
#undef GF2L_TEAM
#undef GF2L_TEAM_AS
    return hipGetLastError();
}

}  // namespace gf2l
