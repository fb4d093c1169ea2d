// gl3_seqsum.h — exact parallel evaluation of the strictly sequential binary32 sum
//     s = (((0 + a_0) + a_1) + ... + a_{n-1}),   a_k = x_k * x_k >= 0,
// i.e. InferenceCore.rmsnorm's `x.reduce(0f, (acc, xi) -> acc + xi * xi)` (J/inference/InferenceCore.java:41),
// bit for bit, without a 4096-step dependent chain (13 cycles / element on gfx950 = 22 us for dim 4096).
//
// Idea (CPU mirror with adversarial trials: tests/test_seqsum_mirror.py): while the running sum stays
// inside one binade it is N*u with an integer N, and adding a_k adds an integer that depends only on a_k
// (and, on an exact rounding tie, on the parity of N).  So a segment of m elements that (i) starts in the
// binade predicted by an approximate prefix sum, (ii) does not leave it and (iii) gives the same increment D
// from an even and from an odd start is a pure translation s -> s + D, and translations compose exactly
// (integer sums of D/u).  Each of 256 threads finds the D of its 4-element segments by running the real f32 chain from two
// representative starts; the few "hard" segments (a binade crossing, a parity-dependent tie, the first one;
// ~18 of 1024 four-element segments for Gaussian data) are replayed with real f32 adds from their true start = previous hard
// segment's end + (integer run sum) * u.  The premises are re-checked on the true values at every run
// boundary (values are monotone, so boundary checks cover the interior); on any violation the naive chain
// runs instead, so the result is always exactly the sequential sum.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gl3 {

#ifdef GL3_SS_TIMING
__device__ long long gl3_ss_stamp[16];
#define SS_STAMP(i) do { if ((threadIdx.x & 255) == 0) gl3_ss_stamp[i] = clock64(); } while (0)
#else
#define SS_STAMP(i)
#endif

constexpr int SS_T = 256;                          // threads that own a segment

__device__ __forceinline__ uint32_t f2u(float f) { return __builtin_bit_cast(uint32_t, f); }
__device__ __forceinline__ float u2f(uint32_t u) { return __builtin_bit_cast(float, u); }

// wave64 inclusive scan with DPP row shifts + row broadcasts (the sequence LLVM's atomic optimizer emits on gfx9)
__device__ __forceinline__ uint32_t wave_incl_scan_u32(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false);   // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);   // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);   // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);   // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);   // row_bcast15 -> rows 1,3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);   // row_bcast31 -> rows 2,3
    return v;
}
__device__ __forceinline__ float wave_incl_scan_f32(float v) {                        // predictor only (any order)
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x111, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x112, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x114, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x118, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xa, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xc, 0xf, false));
    return v;
}

// naive chain over x[k0..k1), executed redundantly by all lanes of one wavefront (LDS broadcast reads)
template <bool SQ = true>
__device__ __forceinline__ float naive_sumsq_lds(const float* x, int k0, int k1, float s) {
    int k = k0;
    for (; k + 4 <= k1; k += 4) {
        const float4 v = *reinterpret_cast<const float4*>(x + k);
        if (SQ) { s = s + v.x * v.x; s = s + v.y * v.y; s = s + v.z * v.z; s = s + v.w * v.w; }
        else { s = s + v.x; s = s + v.y; s = s + v.z; s = s + v.w; }
    }
    for (; k < k1; ++k) { const float v = x[k]; s = SQ ? s + v * v : s + v; }
    return s;
}

// Sequential part of exact_seqsum_lds, run by one wavefront.  Event j < nhard = hard segment j (in order) preceded by
// the easy run since the previous hard segment; event nhard = the trailing easy run.  Lane j gathers event j's
// run translation (exact: integer run sum * ulp) and its four terms in one parallel pass over LDS.
// ep[seg] = (prefix of D / ulp inside the segment's wavefront, predicted exponent | hard << 31); hl: the hard segments of every wavefront's
// span of S segments, from the span's own place on; w_nd, w_cnt: the wavefronts' totals.
constexpr int SS_EVENTS = 61;                      // events of one pass: the first, then four at a time
template <bool SQ>
__device__ __forceinline__ void replay_events(const float* x, int nseg, int S, const uint2* ep, const int* hl, const uint32_t* w_nd, const int* w_cnt, float& base, int& fail) {
    const int lane = threadIdx.x & 63;
    const int c0n = w_cnt[0], c1n = c0n + w_cnt[1], c2n = c1n + w_cnt[2], nhard = c2n + w_cnt[3];          // (nhard >= 1: the first segment is hard)
    // (sums of masked terms: a select between captures would put them all into scratch memory)
    const int o1 = S - c0n, o2 = S - (c1n - c0n), o3 = S - (c2n - c1n);
    auto place = [=](int j) { return j + (j >= c0n ? o1 : 0) + (j >= c1n ? o2 : 0) + (j >= c2n ? o3 : 0); };
    const uint32_t d1 = w_nd[0], d2 = w_nd[1], d3 = w_nd[2];
    auto before = [=](int seg) { return (seg >= S ? d1 : 0u) + (seg >= 2 * S ? d2 : 0u) + (seg >= 3 * S ? d3 : 0u); };
    const int edge = min(max(lane, 1) * S, nseg - 1);
    const uint32_t el = ep[edge - 1].y, er_ = ep[edge].y;
    if (lane >= 1 && lane < 4 && lane * S < nseg) fail |= (int)(!((el | er_) >> 31) && el != er_);          // easy segments on either side of two wavefronts' border: one binade
    for (int k0 = 0; k0 <= nhard; k0 += SS_EVENTS) {
        // everything is read unconditionally, from clamped places
        const int j = k0 + lane;
        const int hj = hl[place(min(j, nhard - 1))], hp = hl[place(min(max(j - 1, 0), nhard - 1))];
        const int h = j < nhard ? hj : nseg, ph = j > 0 ? hp : -1;
        const uint2 e1 = ep[max(h - 1, 0)], e0 = ep[max(ph, 0)];
        const uint32_t ef = ep[min(ph + 1, nseg - 1)].y & 0x7FFFFFFFu;
        float4 sq = *reinterpret_cast<const float4*>(x + 4 * h);
        if (SQ) { sq.x = sq.x * sq.x; sq.y = sq.y * sq.y; sq.z = sq.z * sq.z; sq.w = sq.w * sq.w; }
        const bool run = j <= nhard && h - 1 > ph && lane < SS_EVENTS;
        if (j >= nhard || lane >= SS_EVENTS) sq = make_float4(0.f, 0.f, 0.f, 0.f);          // the trailing event and the lanes behind it add nothing
        const uint32_t R = e1.x + before(h - 1) - (e0.x + before(ph)), er = run ? ef : 0u;          // 0 = no easy run before this event
        const float runadd = run ? (float)R * u2f((er - 23u) << 23) : 0.f;                          // exact: integer run sum * ulp
        SS_STAMP(4);
        // The sequential part.  Lane j already holds event j's operands, so instead of feeding one chain through v_readlane EVERY lane runs the event's five adds on its own operands and the
        // result moves one lane up (wave_shr:1, as an operand of the first add): at step k lane k has the true incoming value, from lane k - 1's step k - 1.  What a lane's own step made
        // is kept for the binade checks (beside the chain).  Steps go four at a time: lanes behind the last event add zeros, so the value that arrives there stays the chain's.
        const int nev = __builtin_amdgcn_readfirstlane(min(SS_EVENTS, 1 + ((min(SS_EVENTS, nhard + 1 - k0) + 2) & ~3)));
        auto terms = [=](float t) { t = t + sq.x; t = t + sq.y; t = t + sq.z; return t + sq.w; };
        float t2 = terms(base + runadd), made = t2;
        for (int k = 1; k < nev; k += 4) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                t2 = terms(u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(t2), 0x138, 0xf, 0xf, true)) + runadd);
                made = lane == k + u ? t2 : made;
            }
        }
        const float in = u2f((uint32_t)__builtin_amdgcn_update_dpp((int)f2u(base), (int)f2u(made), 0x138, 0xf, 0xf, false));          // (lane 0: base)
        if (er != 0u) {
            const float after_run = in + runadd;
            fail |= (int)((f2u(in) >> 23) != er) | (int)((f2u(after_run) >> 23) != er);
        }
        base = u2f((uint32_t)__builtin_amdgcn_readlane((int)f2u(t2), nev - 1));
    }
    fail = __builtin_amdgcn_ballot_w64(fail != 0) != 0;          // any lane's violation fails the wavefront
}

// Barrier functors for exact_sumsq_lds: `sync()` must be a barrier over exactly the 4 participating wavefronts.
struct BlockBarrier { __device__ __forceinline__ void operator()() const { __syncthreads(); } };

// Barrier over a subset of the workgroup's wavefronts through an LDS counter (gfx950 has no named barriers).
// ctr must be zero before first use; every participating wavefront calls operator() the same number of times.
struct SubBarrier {
    int* ctr; int nwaves; int target;
    __device__ __forceinline__ void operator()() {
        target += nwaves;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(ctr, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < target) {}     // busy poll: an s_sleep(1) quantum is 64 cycles
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    }
};

// scratch bytes needed for n elements (16-byte aligned): header + prefix, exponent and hard list per 4-element segment
__host__ __device__ constexpr size_t ss_scratch_bytes(int n) { return 128 + (size_t)3 * n; }
constexpr int SS_MAX_SPT = 5;                      // segments per thread: n <= 4 * 256 * 5 = 5120

// SQ = true: a_k = x_k * x_k (RMSNorm); SQ = false: a_k = x_k >= 0 (FloatTensor.sum of softmax numerators / probabilities,
// J/tensor/standard/FloatTensor.java:211-219).  start = value of the running sum before x[0] (chunked sums of long vectors).
// Bound: four lone wavefronts issue an instruction every ~5 cycles, so what counts is instructions in a row and barriers.  The segments of a thread are worked on side by side and without branches,
// prefixes and hard lists stay inside a wavefront (the replay adds the totals: three barriers instead of four), and the replay's step is five adds and no select.
// 4096 elements alone 3.56 us -> 2.60, 2048 3.08 -> 2.16.
template <bool SQ, typename Sync>
__device__ __forceinline__ float exact_seqsum_lds(const float* x, int n, uint8_t* scratch, const int t, Sync& sync, const float start) {
    const int lane = t & 63, wave = t >> 6;
    float* w_tot = reinterpret_cast<float*>(scratch);                    // [4]  predictor wave totals
    uint32_t* w_nd = reinterpret_cast<uint32_t*>(scratch + 16);          // [4]  run-sum wave totals
    int* w_cnt = reinterpret_cast<int*>(scratch + 32);                   // [4]  hard segments per wave
    int* w_bad = reinterpret_cast<int*>(scratch + 48);                   // [4]  neighbours in different binades
    float* result = reinterpret_cast<float*>(scratch + 64);              // [0]
    const int nseg = n >> 2;                                             // 4-element segments (one float4 each)
    uint2* ep = reinterpret_cast<uint2*>(scratch + 128);                 // [nseg]
    int* hl = reinterpret_cast<int*>(ep + nseg);                         // [nseg]
    const int spt = (nseg + SS_T - 1) / SS_T, seg0 = t * spt;            // segments per thread (uniform)
    constexpr int SPT = SS_MAX_SPT;
    SS_STAMP(0);

    // ---- predictor: approximate (any-order) f32 prefix of the terms before each of my segments.  All LDS reads are issued unconditionally (segments past the end read the zero padding behind
    // x[n]): reads under a lane-dependent condition are waited for one by one
    float4 a[SPT];
    float qs[SPT], qt = 0.f;
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        const float4 v = *reinterpret_cast<const float4*>(x + 4 * min(seg0 + i, nseg));
        if (SQ) { a[i].x = v.x * v.x; a[i].y = v.y * v.y; a[i].z = v.z * v.z; a[i].w = v.w * v.w; }
        else a[i] = v;
    }
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        if (i >= spt) break;
        qs[i] = (a[i].x + a[i].y) + (a[i].z + a[i].w);
        qt += qs[i];
    }
    const float incl = wave_incl_scan_f32(qt);
    if (lane == 63) w_tot[wave] = incl;
    sync();
    SS_STAMP(1);
    const float t0 = w_tot[0], t1 = w_tot[1], t2 = w_tot[2];
    float P = start + (incl - qt);
    if (wave > 0) P += t0;
    if (wave > 1) P += t1;
    if (wave > 2) P += t2;

    // ---- translation D of each segment from two representative starts (even / odd mantissa)
    uint32_t ev[SPT], nd[SPT], hmask = 0, ndt = 0;
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        ev[i] = 0x80000000u; nd[i] = ndt;
        if (i >= spt) continue;
        const uint32_t rb = f2u(P) & ~1u, e = rb >> 23;
        const float R0 = u2f(rb), R1 = u2f(rb | 1u), margin = u2f((e - 10u) << 23);         // 8192 ulp: keeps the fallback rare
        float E0 = R0, E1 = R1;
        E0 = E0 + a[i].x; E1 = E1 + a[i].x; E0 = E0 + a[i].y; E1 = E1 + a[i].y;
        E0 = E0 + a[i].z; E1 = E1 + a[i].z; E0 = E0 + a[i].w; E1 = E1 + a[i].w;
        const float D0 = E0 - R0, D1 = E1 - R1;
        const uint32_t leaves = (f2u(E0) ^ rb) | (f2u(E1) ^ rb) | (f2u(R0 - margin) ^ rb) | (f2u(E0 + margin) ^ rb);      // a bit from 23 on: another binade
        const bool easy = (D0 == D1) & (leaves < 1u << 23) & (e - 41u < 209u) & (seg0 + i > 0) & (seg0 + i < nseg);
        ev[i] = easy ? e : e | 0x80000000u;
        ndt += easy ? (uint32_t)(D0 * u2f((277u - e) << 23)) : 0u;           // D / ulp, exact integer < 2^24
        nd[i] = ndt;
        hmask |= (easy || seg0 + i >= nseg ? 0u : 1u) << i;
        P += qs[i];
    }
    SS_STAMP(2);
    // ---- inclusive prefix of nd inside the wavefront (mod 2^32: only differences inside one run are used), hard list, neighbours
    const uint32_t pin = wave_incl_scan_u32(ndt);
    uint32_t hin = 0, last = ev[0];                                      // hard segments of the lanes in front; the thread's last segment
    int hall = 0;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        if (i >= spt) break;
        const uint64_t hb = __builtin_amdgcn_ballot_w64((hmask >> i) & 1u);
        hin = __builtin_amdgcn_mbcnt_hi((uint32_t)(hb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)hb, hin));
        hall += __popcll(hb);
        bad |= !((last | ev[i]) >> 31) && last != ev[i];
        last = ev[i];
    }
    const uint32_t left = (uint32_t)__builtin_amdgcn_update_dpp((int)0x80000000u, (int)last, 0x138, 0xf, 0xf, false);          // wave_shr:1, lane 0: no neighbour here
    bad |= !((left | ev[0]) >> 31) && left != ev[0];
    const uint32_t nb0 = pin - ndt;
    int hpos = 64 * spt * wave + (int)hin;
#pragma unroll
    for (int i = 0; i < SPT; ++i) {
        if (i >= spt) break;
        if (seg0 + i < nseg) ep[seg0 + i] = make_uint2(nb0 + nd[i], ev[i]);
        if ((hmask >> i) & 1u) hl[hpos++] = seg0 + i;
    }
    const bool any_bad = __builtin_amdgcn_ballot_w64(bad) != 0;
    if (lane == 63) { w_nd[wave] = pin; w_cnt[wave] = hall; w_bad[wave] = any_bad; }
    sync();
    SS_STAMP(3);
    // ---- replay the hard segments in order (one wavefront), see replay_events
    if (wave == 0) {
        float base = start;
        int fail = 0;
        replay_events<SQ>(x, nseg, 64 * spt, ep, hl, w_nd, w_cnt, base, fail);
        if (fail | w_bad[0] | w_bad[1] | w_bad[2] | w_bad[3]) base = naive_sumsq_lds<SQ>(x, 0, n, start);       // never expected: plain chain
        if (lane == 0) result[0] = base;
        SS_STAMP(5);
    }
    sync();
    SS_STAMP(6);
    return result[0];
}
template <typename Sync>
__device__ __forceinline__ float exact_sumsq_lds(const float* x, int n, uint8_t* scratch, const int t, Sync& sync) {
    return exact_seqsum_lds<true>(x, n, scratch, t, sync, 0.f);
}

}  // namespace gl3
