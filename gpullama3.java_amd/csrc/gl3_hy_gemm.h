// gl3_hy_gemm.h — the layer-list family's matrix product for more than 8 tokens: C[m][n] = sum_k A[m][k] W[n][k], both operands K-contiguous
// rows of 16-byte aligned pieces, K a multiple of one 128-byte stage (64 bfloat16 / 32 float32).  Other shapes: hy_gemm_kernel.
//
// What bounds it.  A workgroup fills at most 160 KB of LDS, so at most that much can travel to a CU; behind HBM misses (1.3 - 1.7 us
// under load) that is 60 - 75 GB/s per CU, while 256 x 256 results need 60 GB/s to keep the matrix cores busy and 128 x 128 twice that.  So:
//   * operands go straight to LDS (global_load_lds, 16 bytes per lane: no staging registers, no store pass) into two rings, SA stages of A
//     (re-read by every workgroup: L2 hits, 0.4 us under load — a ring of two leaves it one stage's time, less than that in the small tiles) and SW > SA stages of
//     W (each row read once: HBM misses, hence the longer lead; the float32 tiles of 64 x 128 and 32 x 128 have as many of either, two and four workgroups of them share a CU);
//   * the barrier of a stage sits a quarter of a stage before its end: the last quarter's MFMAs run behind it while the next stage's first
//     fragments are read, and it waits with a counted vmcnt for everything but the loads that have a whole stage left to travel;
//   * the loads are spread between the MFMAs (issued in one go they hold the wavefront for ~1000 cycles: the address unit takes 16 cycles each);
//   * LDS rows are 128 bytes; 16-byte chunk c of row r stands at chunk c ^ (r / 2 % 8): 16 lanes of a fragment read cover the 64 banks once
//     (SQ_LDS_BANK_CONFLICT 0; with r % 8 half of the cycles were conflicts);
//   * XCD-aware order: the row tiles of A that share a tile of W run on one XCD, so W leaves HBM once.
// The tile is picked per shape (hy_ring_pick in gl3_hybrid.hip).  Measured against hy_gemm_kernel, 512 tokens, W cold in HBM (us):
//   28672 x 4096 220 -> 107 - 125, 18560 x 4096 200 -> 75 - 83, 10240 x 4096 98 -> 49, 4096 x 4096 50 -> 31 (K split in 2: 24), 4096 x 14336 157 -> 65 - 75;
//   88 tokens, 4096 x 14336: 56; 24 tokens, 28672 x 4096: 89 -> 52 (4.5 TB/s of weights).
// float32 matrices.  The float32 MFMAs (v_mfma_f32_32x32x2_f32) take 16 times as long per product as the bfloat16 ones AND the vector units' time with them (measured: the
// times of f32 MFMAs and of vector instructions of a SIMD add up, those of bfloat16 MFMAs overlap).  So an operand is split into three bfloat16 planes on its way from
// LDS (x = p0 + p1 + p2, every plane the rounded rest: all 24 bits
// of values above 2^-108, below which the planes run out of bfloat16's range: a matrix of size 2^-112 errs by 1.6e-7, of 2^-116 by 2.2e-6, of 2^-120 by 3.5e-5) and the plane products of at least 2^-16 go to v_mfma_f32_32x32x16_bf16: six, or three where the
// matrix's values are bfloat16 already (HyMat::b16: what most checkpoints hold; exact).  Only the largest plane product is added in the main chain, a rounding per 16 k, which goes to
// a second set of accumulators every HY_FLUSH stages (128 k); the others, 2^-8 of it and less, have a chain of their own (in one chain they are rounded to its size: 2.3e-7 below).
// Relative error of a product against 64 bits, weights of 24 bits / of bfloat16 values: 181 tokens, 8192 x 2048 0.93e-7 / 0.90e-7 (float32 MFMAs 2.1e-7), 2048 x 8192 1.1e-7 (2.2e-7),
// 512 tokens, 4096 x 512 0.8e-7 (2.1e-7); of positive operands 0.49e-7 / 0.47e-7 (0.58e-7).  An infinity's planes are not a number: tiles with a result that is not finite make it again in float32
// at the end (hy_tile_again).
// Bound now by issue: the one wavefront per SIMD of a 64 x 128 tile is at work 58 % of its cycles (148 vector instructions a stage with weights of one plane; planes made ahead by a kernel of their own,
// and the tile on eight wavefronts, were no faster).  Products alone, us, float32 MFMAs -> weights of one plane / of three: 181 tokens, 8192 x 2048 79 -> 40 / 60, 16384 x 2048 with the gate 135 -> 58 / 98,
// 2048 x 8192 with K split 79 -> 39 / 60, 512 tokens, 4096 x 512 23 -> 13 / 19.  Inside a request (float32 chat, 181 tokens): 8192 x 2048 with its activation 84 -> 50 / 76, experts 183 + 91 -> 121 + 64 / 143 + 75.
#pragma once
#include "gl3_hy_kernels.h"

typedef float hy_v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void hy_dma16(const void* src, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}
// The same for W; ONCE: past the caches (hy_ring_once).
template <bool ONCE>
__device__ __forceinline__ void hy_dma16_w(const void* src, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, ONCE ? 2 : 0);
}
// all but the newest N loads of this wavefront have landed, its LDS reads are done, and so are everybody's
template <int N> __device__ __forceinline__ void hy_wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

constexpr int HY_FLUSH = 4;
typedef float hy_v8f __attribute__((ext_vector_type(8)));
template <typename T> struct HyFrag;
template <> struct HyFrag<bf16_t> { typedef hy_v8bf V; static constexpr int K = 64; };
template <> struct HyFrag<float> { typedef hy_v4f V; static constexpr int K = 32; };
__device__ __forceinline__ void hy_mma(hy_v16f& c, const hy_v8bf& a, const hy_v8bf& b) { c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
typedef __bf16 hy_v2bf __attribute__((ext_vector_type(2)));
typedef float hy_v2f __attribute__((ext_vector_type(2)));
typedef uint32_t hy_v4u __attribute__((ext_vector_type(4)));
template <int I, int N, typename F> __device__ __forceinline__ void hy_static_for(F f) { if constexpr (I < N) { f(std::integral_constant<int, I>{}); hy_static_for<I + 1, N>(f); } }
// Two values as bfloat16, and (REST) what is left of them.  Three times over all 24 bits are held (see above); once for values that are bfloat16 already.
template <bool REST> __device__ __forceinline__ uint32_t hy_plane(float& x, float& y) {
    const uint32_t d = __builtin_bit_cast(uint32_t, __builtin_convertvector((hy_v2f{x, y}), hy_v2bf));
    if constexpr (REST) { x -= __uint_as_float(d << 16); y -= __uint_as_float(d & 0xffff0000u); }
    return d;
}
// Which of 32 rows hold a value that is not a number (bit r: row r); p: row lane % 32.
__device__ __forceinline__ uint32_t hy_nan_rows(const float* __restrict__ p, int n, int kh) {
    bool nan = false;
#pragma unroll 16
    for (int k = 0; k < n; k += 8) {
        const hy_v4f v = *reinterpret_cast<const hy_v4f*>(p + k + 4 * kh);
        nan |= __builtin_isunordered(v[0], v[1]) || __builtin_isunordered(v[2], v[3]);
    }
    const uint64_t b = __ballot(nan);
    return (uint32_t)b | (uint32_t)(b >> 32);
}
// The results `odd` (bit r: register r) of a 32 x 32 tile once more, in float32 MFMAs straight from memory: the planes of an infinity are not a number, and so is their product.  a, w: the
// lane's row (lane % 32) of either operand, n a multiple of 8.  Rows and columns with an operand that is not a number have their results already: a spoiled row costs the look at its operands
// (a prompt of 181 rows of 1024, none a number: 0.25 ms instead of 0.21; one lane's chain per result took 6.1 ms) and only infinities the products.
__device__ __attribute__((noinline)) hy_v16f hy_tile_again(hy_v16f c, uint32_t odd, const float* __restrict__ a, const float* __restrict__ w, int n, float scale) {
    const int lane = threadIdx.x & 63, r32 = lane & 31, kh = lane >> 5;
    const uint32_t na = hy_nan_rows(a, n, kh);
#pragma unroll
    for (int r = 0; r < 16; ++r) if (na >> (8 * (r >> 2) + 4 * kh + (r & 3)) & 1) odd &= ~(1u << r);
    if (!__any(odd)) return c;
    if (hy_nan_rows(w, n, kh) >> r32 & 1) odd = 0;
    if (!__any(odd)) return c;
    hy_v16f tot;
#pragma unroll
    for (int r = 0; r < 16; ++r) tot[r] = 0.f;
#pragma unroll 1
    for (int k0 = 0; k0 < n; k0 += 128) {
        hy_v16f d;
#pragma unroll
        for (int r = 0; r < 16; ++r) d[r] = 0.f;
#pragma unroll 4
        for (int k = k0; k < min(n, k0 + 128); k += 8) {
            const hy_v4f x = *reinterpret_cast<const hy_v4f*>(a + k + 4 * kh), y = *reinterpret_cast<const hy_v4f*>(w + k + 4 * kh) * scale;
#pragma unroll
            for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_32x32x2f32(x[e], y[e], d, 0, 0, 0);
        }
        tot += d;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) if (odd >> r & 1) c[r] = tot[r];
    return c;
}

// WM x WN wavefronts, BM x BN results; EPI, GR and HyGroup as for hy_gemm_kernel (GR: blockIdx.y = row tile of the list, BM rows at most).
// Grid: x = mt nt ks workgroups (row tiles x column tiles x K splits of kper) rounded up to a multiple of 8; GR: x = column tiles.
template <typename T, int BM, int BN, int WM, int WN, int SA, int SW, int EPI, int GR, int WP, bool ONCE>
static __global__ __launch_bounds__(WM * WN * 64, sizeof(T) == 4 ? 2 : 1) void hy_gemm_ring_kernel(const T* __restrict__ A, int lda, const T* __restrict__ Wt, int ldw, int M, int N, int K,
                                                                           float* __restrict__ C, int ldc, T* __restrict__ act, int ld_act, HyGlu glu, int mt, int nt, int ks,
                                                                           int kper, HyGroup grp = HyGroup{}) {
    constexpr int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32, BK = HyFrag<T>::K;
    constexpr int PA = BM / 8, PW = BN / 8, NPA = (PA + NW - 1) / NW, NPW = (PW + NW - 1) / NW, NP = NPA + NPW;      // 1 KB pieces (8 rows) of a stage, per wavefront
    constexpr int SZA = BM * 128, SZW = BN * 128, OW = SA * SZA;
    static_assert(SW >= SA + (sizeof(T) == 2) && SA >= 2 && NPA * NW < 2 * PA + NW && TM * WM * 32 == BM && TN * WN * 32 == BN, "tile layout");
    static_assert(SA * SZA + SW * SZW <= 160 * 1024, "LDS");
    __shared__ __attribute__((aligned(1024))) uint8_t smem[SA * SZA + SW * SZW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
    int m0, n0, z = 0;
    if constexpr (GR) {
        if ((int)blockIdx.y >= grp.ntiles[0]) return;
        const int* tl = grp.tiles + 3 * blockIdx.y;
        const int row0 = tl[0];
        M = tl[1];
        A += (size_t)row0 * lda;
        Wt += (size_t)tl[2] * grp.wstride;
        if (C) C += (size_t)row0 * ldc;
        if (act) act += (size_t)row0 * ld_act;
        m0 = 0; n0 = blockIdx.x * BN;
    } else {
        const int total = mt * nt * ks, per_xcd = (total + 7) >> 3;          // workgroups go to the XCDs in turn
        const int J = (blockIdx.x & 7) * per_xcd + (blockIdx.x >> 3);
        if (J >= total) return;
        m0 = (J % mt) * BM; z = (J / mt) % ks; n0 = (J / mt / ks) * BN;
    }
    const int kbeg = z * kper, n_it = (min(K, kbeg + kper) - kbeg) / BK;
    if constexpr (EPI == HY_EPI_STORE) C += (size_t)z * M * ldc;
    // this wavefront's pieces: byte offset of the lane's source in the operand (rows past the end repeat the last one: their results are
    // not stored), byte offset in the ring; wavefronts left without a piece of their own load one again (the same bytes to the same place)
    uint32_t offa[NPA], offw[NPW];
    int pa[NPA], pw[NPW];
#pragma unroll
    for (int u = 0; u < NPA; ++u) {
        const int p = (wave + NW * u) % PA, row = 8 * p + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        pa[u] = p * 1024;
        offa[u] = ((uint32_t)min(m0 + row, M - 1) * (uint32_t)lda + kbeg) * (uint32_t)sizeof(T) + 16 * c;
    }
#pragma unroll
    for (int u = 0; u < NPW; ++u) {
        const int p = (wave + NW * u) % PW, row = 8 * p + (lane >> 3), c = (lane & 7) ^ ((row >> 1) & 7);
        pw[u] = OW + p * 1024;
        offw[u] = ((uint32_t)min(n0 + row, N - 1) * (uint32_t)ldw + kbeg) * (uint32_t)sizeof(T) + 16 * c;
    }
    constexpr int WH = (NPW + 1) / 2;
    auto issue_a = [&](int it, int slot) {
        const uint8_t* a = (const uint8_t*)A + (size_t)it * 128;
#pragma unroll
        for (int u = 0; u < NPA; ++u) hy_dma16(a + offa[u], smem + slot * SZA + pa[u]);
    };
    auto issue_w = [&](int it, int slot, int u0, int u1) {
        const uint8_t* w = (const uint8_t*)Wt + (size_t)it * 128;
#pragma unroll
        for (int u = 0; u < NPW; ++u)
            if (u >= u0 && u < u1) hy_dma16_w<ONCE>(w + offw[u], smem + slot * SZW + pw[u]);
    };
    hy_v16f acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
    hy_v16f tot[sizeof(T) == 4 ? TM : 1][sizeof(T) == 4 ? TN : 1];
    if constexpr (sizeof(T) == 4) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) tot[i][j] = acc[i][j];
    }
    auto flush = [&]() {
        if constexpr (sizeof(T) == 4) {
#pragma unroll
            for (int i = 0; i < TM; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) { tot[i][j][r] += acc[i][j][r]; acc[i][j][r] = 0.f; }
        }
    };
    const int r32 = lane & 31, kh = lane >> 5;
    uint32_t ca[4];          // a stage is four quarters; a lane reads row lane % 32, chunk 2 quarter + lane / 32
#pragma unroll
    for (int q = 0; q < 4; ++q) ca[q] = ((2 * q + kh) ^ ((r32 >> 1) & 7)) * 16;
    const uint32_t aw = (wm * (BM / WM) + r32) * 128, ww = OW + (wn * (BN / WN) + r32) * 128;
    if constexpr (sizeof(T) == 4) {
        // Half a stage (16 k) at a time, three deep: while the MFMAs take half h's planes, half h + 1 is split and half h + 2 comes from LDS.  Barrier s finds the stage's last
        // chunks in registers, so the loads behind it (A's stage s + SA, W's s + SW) go into the stage's own slots.
        constexpr int LEFT = SW > SA ? NPW + (SA - 2) * NP : (SA - 2) * NP;          // loads started behind stage s + 1's when barrier s waits for them (a step starts A's, then W's)
        hy_v4f xa[2][TM][2], xw[2][TN][2];
        hy_v4u qa[2][TM][3], qw[2][TN][WP];
        auto rd = [&](int set, int sa, int sw, int h) {
#pragma unroll
            for (int u = 0; u < 2; ++u) {
#pragma unroll
                for (int j = 0; j < TN; ++j) xw[set][j][u] = *reinterpret_cast<const hy_v4f*>(smem + sw * SZW + ww + j * 4096 + ca[2 * h + u]);
#pragma unroll
                for (int i = 0; i < TM; ++i) xa[set][i][u] = *reinterpret_cast<const hy_v4f*>(smem + sa * SZA + aw + i * 4096 + ca[2 * h + u]);
            }
        };
        // the split of a half in UN steps, a plane of one pair of values each
        constexpr int UN = 4 * (WP * TN + 3 * TM);
        auto cut = [&](auto c, int set) {
            constexpr int u = decltype(c)::value, w = 4 * WP * TN, f = u < w ? u / (4 * WP) : (u - w) / 12, pl = u < w ? u / 4 % WP : (u - w) / 4 % 3, e = u % 4;
            if constexpr (u < w) qw[set][f][pl][e] = hy_plane<(pl + 1 < WP)>(*((float*)&xw[set][f][e / 2] + e % 2 * 2), *((float*)&xw[set][f][e / 2] + e % 2 * 2 + 1));
            else qa[set][f][pl][e] = hy_plane<(pl < 2)>(*((float*)&xa[set][f][e / 2] + e % 2 * 2), *((float*)&xa[set][f][e / 2] + e % 2 * 2 + 1));
        };
        // the products of at least 2^-16 (planes a + b <= 2); all but the largest add up in a chain of their own, where they are rounded to their size
        hy_v16f low[TM][TN];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) low[i][j] = acc[i][j];
        constexpr int NM = (WP == 3 ? 6 : 3) * TM * TN;
        auto mm = [&](auto c, int set) {
            constexpr int q = decltype(c)::value / (TM * TN), i = decltype(c)::value / TN % TM, j = decltype(c)::value % TN;
            constexpr int a_ = WP == 3 ? (q == 0 ? 2 : q == 1 || q == 3 ? 1 : 0) : 2 - q, b_ = WP == 3 ? (q == 1 || q == 4 ? 1 : q == 2 ? 2 : 0) : 0;
            hy_mma(a_ + b_ ? low[i][j] : acc[i][j], __builtin_bit_cast(hy_v8bf, qa[set][i][a_]), __builtin_bit_cast(hy_v8bf, qw[set][j][b_]));
        };
        // (pinned: left to the compiler the splits stand in one piece behind the MFMAs)
        auto both = [&](auto mset, int cset, auto load) {
            hy_static_for<0, NM>([&](auto c) {
                constexpr int q = decltype(c)::value, u0 = q * UN / NM, u1 = (q + 1) * UN / NM, h = NM * decltype(mset)::value, l0 = (h + q) * NP / (2 * NM), l1 = (h + q + 1) * NP / (2 * NM);
                mm(c, decltype(mset)::value);
                hy_static_for<l0, l1>(load);
                hy_static_for<u0, u1>([&](auto u) { cut(u, cset); });
                __builtin_amdgcn_sched_barrier(0);
            });
        };
        constexpr std::integral_constant<int, 0> H0{};
        constexpr std::integral_constant<int, 1> H1{};
#pragma unroll
        for (int s = -SW; s < 0; ++s) {
            if (s + SA >= 0 && s + SA < n_it) issue_a(s + SA, s + SA);
            if (s + SW < n_it) issue_w(s + SW, s + SW, 0, NPW);
        }
        if (n_it >= SW) hy_wait_barrier<LEFT + NP>(); else hy_wait_barrier<0>();
        int sa = 0, sw = 0, it = 0;
        rd(0, 0, 0, 0);
        rd(1, 0, 0, 1);
        hy_static_for<0, UN>([&](auto u) { cut(u, 0); });
        while (it < n_it - SW) {
            const int stop = min(n_it - SW, it + HY_FLUSH);
#pragma unroll 1
            for (; it < stop; ++it) {
                __builtin_amdgcn_s_waitcnt(0xc07f);          // lgkmcnt(0) where the compiler sees it: it would wait for the reads behind the barrier as well
                hy_wait_barrier<LEFT>();
                const uint8_t *na = (const uint8_t*)A + (size_t)(it + SA) * 128, *nw = (const uint8_t*)Wt + (size_t)(it + SW) * 128;
                uint8_t *da = smem + sa * SZA, *dw = smem + sw * SZW;
                auto load = [&](auto c) {          // piece c of this step
                    constexpr int u = decltype(c)::value;
                    if constexpr (u < NPA) hy_dma16(na + offa[u], da + pa[u]); else hy_dma16_w<ONCE>(nw + offw[u - NPA], dw + pw[u - NPA]);
                };
                if (++sa == SA) sa = 0;
                if (++sw == SW) sw = 0;
                rd(0, sa, sw, 0);
                __builtin_amdgcn_sched_barrier(0);
                both(H0, 1, load);
                rd(1, sa, sw, 1);
                __builtin_amdgcn_sched_barrier(0);
                both(H1, 0, load);
            }
            flush();
        }
        for (; it < n_it; ++it) {          // the last SW stages: nothing (A: little) left to load
            hy_wait_barrier<0>();
            if (it + SA < n_it) issue_a(it + SA, sa);
            if (++sa == SA) sa = 0;
            if (++sw == SW) sw = 0;
            const bool more = it + 1 < n_it;
            if (more) rd(0, sa, sw, 0);
            both(H0, 1, [](auto) {});
            if (more) rd(1, sa, sw, 1);
            both(H1, 0, [](auto) {});          // (nothing behind the last stage: the chunks are those of before, the planes unused)
        }
        flush();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = tot[i][j] + low[i][j];
    } else {
    // step s (behind barrier s) starts the loads of A's stage s + SA (into the slot the barrier freed) and, in the two quarters after it,
    // of W's stage s + SW; the steps before 0 are the prologue, the last one's W belongs to the loop's first round
    constexpr int LEFT = (SA - 2) * NP + NPW;          // loads started behind A's stage s + 1 when barrier s waits for it
#pragma unroll
    for (int s = -SW; s < 0; ++s) {
        if (s + SA >= 0 && s + SA < n_it) issue_a(s + SA, s + SA);
        if (s < -1 && s + SW < n_it) issue_w(s + SW, s + SW, 0, NPW);
    }
    if (n_it >= SW) hy_wait_barrier<(SA - 1) * NP>(); else hy_wait_barrier<0>();
    int sa = 0, sw = 0, sp = SW - 1, it = 0;          // slots of the current stage; sp: the W slot that the step before fills
    typedef typename HyFrag<T>::V V;
    V fa[2][TM], fw[2][TN];
    auto rd = [&](int set, int sa, int sw, int q) {
#pragma unroll
        for (int i = 0; i < TM; ++i) fa[set][i] = *reinterpret_cast<const V*>(smem + sa * SZA + aw + i * 4096 + ca[q]);
#pragma unroll
        for (int j = 0; j < TN; ++j) fw[set][j] = *reinterpret_cast<const V*>(smem + sw * SZW + ww + j * 4096 + ca[q]);
    };
    auto mm = [&](int set) {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) hy_mma(acc[i][j], fa[set][i], fw[set][j]);
    };
    // a quarter's order: fragment reads and the quarter's loads (ND of them) between the MFMAs
    constexpr int NR = TM + TN, NM = TM * TN;
#define HY_QUARTER(ND)                                                              \
    do {                                                                            \
        _Pragma("unroll") for (int q_ = 0; q_ < NR; ++q_) {                         \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      \
            if (q_ + 1 <= NM) __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     \
            if (q_ < (ND)) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);        \
        }                                                                           \
        if (NM > NR) __builtin_amdgcn_sched_group_barrier(0x8, NM - NR, 0);          \
        __builtin_amdgcn_sched_barrier(0);                                          \
    } while (0)
    rd(0, 0, 0, 0);
    for (; it < n_it - SW; ++it) {
        rd(1, sa, sw, 1); mm(0); issue_w(it - 1 + SW, sp, 0, WH); HY_QUARTER(WH);
        rd(0, sa, sw, 2); mm(1); issue_w(it - 1 + SW, sp, WH, NPW); HY_QUARTER(NPW - WH);
        rd(1, sa, sw, 3); mm(0); HY_QUARTER(0);
        hy_wait_barrier<LEFT>();
        const int freed = sa;
        sp = sw;
        if (++sa == SA) sa = 0;
        if (++sw == SW) sw = 0;
        rd(0, sa, sw, 0); mm(1); issue_a(it + SA, freed); HY_QUARTER(NPA);
    }
    if (it - 1 + SW < n_it) issue_w(it - 1 + SW, sp, 0, NPW);
    for (; it < n_it; ++it) {          // the last SW stages: nothing (A: little) left to load
        rd(1, sa, sw, 1); mm(0); HY_QUARTER(0);
        rd(0, sa, sw, 2); mm(1); HY_QUARTER(0);
        rd(1, sa, sw, 3); mm(0); HY_QUARTER(0);
        hy_wait_barrier<0>();
        if (it + SA < n_it) issue_a(it + SA, sa);
        if (++sa == SA) sa = 0;
        if (++sw == SW) sw = 0;
        if (it + 1 < n_it) rd(0, sa, sw, 0);
        mm(1);
        __builtin_amdgcn_sched_barrier(0);
    }
    }
#undef HY_QUARTER
    // lane holds column lane % 32 and rows 8 (r / 4) + 4 (lane / 32) + r % 4 of every 32 x 32 tile
    const int mb = m0 + wm * (BM / WM) + 4 * kh, nb = n0 + wn * (BN / WN) + r32;
    if constexpr (sizeof(T) == 4) {          // an operand or a sum that is not finite (rare)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                uint32_t odd = 0;
#pragma unroll
                for (int r = 0; r < 16; ++r) odd |= !(fabsf(acc[i][j][r]) < INFINITY) ? 1u << r : 0u;
                if (__builtin_expect(__any(odd), 0)) {
                    const int ma = m0 + wm * (BM / WM) + i * 32 + r32, n = nb + j * 32;
#pragma unroll
                    for (int r = 0; r < 16; ++r) if (mb + i * 32 + 8 * (r >> 2) + (r & 3) >= M || n >= N) odd &= ~(1u << r);          // (repeated rows: not stored)
                    if (__any(odd))
                        acc[i][j] = hy_tile_again(acc[i][j], odd, (const float*)A + (size_t)min(ma, M - 1) * lda + kbeg, (const float*)Wt + (size_t)min(n, N - 1) * ldw + kbeg, n_it * BK, 1.f);
                }
            }
    }
    if constexpr (EPI == HY_EPI_GLU) {
        static_assert(EPI != HY_EPI_GLU || TN % 2 == 0, "gate / up pairs need a wavefront tile of 64 features");
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j + 1 < TN; j += 2) {
                const int f = (n0 + wn * (BN / WN) + j * 32) / 2 + r32;        // feature of this lane's gate (tile j) and up (tile j + 1)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = mb + i * 32 + 8 * (r >> 2) + (r & 3);
                    if (m < M && f < ld_act && 2 * f < N) hy_st(act + (size_t)m * ld_act + f, hy_glu(acc[i][j][r], acc[i][j + 1][r], glu));
                }
            }
    } else {
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) {
                const int n = nb + j * 32;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int m = mb + i * 32 + 8 * (r >> 2) + (r & 3);
                    if (m < M && n < N) {
                        if constexpr (EPI == HY_EPI_STORE) C[(size_t)m * ldc + n] = acc[i][j][r];
                        else hy_st(act + (size_t)m * ld_act + n, hy_actmul<T>(acc[i][j][r], m, n, glu));
                    }
                }
            }
    }
}
