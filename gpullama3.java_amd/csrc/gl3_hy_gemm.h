// gl3_hy_gemm.h — the layer-list family's matrix product for more than 8 tokens: C[m][n] = sum_k A[m][k] W[n][k], both operands K-contiguous
// rows of 16-byte aligned pieces, K a multiple of one 128-byte stage (64 bfloat16 / 32 float32).  Other shapes: hy_gemm_kernel.
//
// What bounds it.  A workgroup fills at most 160 KB of LDS, so at most that much can travel to a CU; behind HBM misses (1.3 - 1.7 us
// under load) that is 60 - 75 GB/s per CU, while 256 x 256 results need 60 GB/s to keep the matrix cores busy and 128 x 128 twice that.  So:
//   * operands go straight to LDS (global_load_lds, 16 bytes per lane: no staging registers, no store pass) into two rings, SA stages of A
//     (re-read by every workgroup: L2 hits, 0.4 us under load — a ring of two leaves it one stage's time, less than that in the small tiles) and SW > SA stages of
//     W (each row read once: HBM misses, hence the longer lead);
//   * the barrier of a stage sits a quarter of a stage before its end: the last quarter's MFMAs run behind it while the next stage's first
//     fragments are read, and it waits with a counted vmcnt for everything but the loads that have a whole stage left to travel;
//   * the loads are spread between the MFMAs (issued in one go they hold the wavefront for ~1000 cycles: the address unit takes 16 cycles each);
//   * LDS rows are 128 bytes; 16-byte chunk c of row r stands at chunk c ^ (r / 2 % 8): 16 lanes of a fragment read cover the 64 banks once
//     (SQ_LDS_BANK_CONFLICT 0; with r % 8 half of the cycles were conflicts);
//   * XCD-aware order: the row tiles of A that share a tile of W run on one XCD, so W leaves HBM once.
// The tile is picked per shape (hy_ring_pick in gl3_hybrid.hip).  Measured against hy_gemm_kernel, 512 tokens, W cold in HBM (us):
//   28672 x 4096 220 -> 107 - 125, 18560 x 4096 200 -> 75 - 83, 10240 x 4096 98 -> 49, 4096 x 4096 50 -> 31 (K split in 2: 24), 4096 x 14336 157 -> 65 - 75;
//   88 tokens, 4096 x 14336: 56; 24 tokens, 28672 x 4096: 89 -> 52 (4.5 TB/s of weights).
// float32 matrices (v_mfma_f32_32x32x2_f32): a lane's 16-byte chunk holds 4 k of its row, so one read feeds four MFMAs (the half-wave's
// chunks pair up; k enters in the order 0, 4, 1, 5, ...); the accumulators are added to a second set every HY_FLUSH stages (128 k), so that the
// rounding of a long K grows with the number of blocks and not with K.
#pragma once
#include "gl3_hy_kernels.h"

typedef float hy_v4f __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void hy_dma16(const void* src, void* lds_wave_base) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src, (__attribute__((address_space(3))) void*)lds_wave_base, 16, 0, 0);
}
// all but the newest N loads of this wavefront have landed, its LDS reads are done, and so are everybody's
template <int N> __device__ __forceinline__ void hy_wait_barrier() { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory"); }

constexpr int HY_FLUSH = 4;
template <typename T> struct HyFrag;
template <> struct HyFrag<bf16_t> { typedef hy_v8bf V; static constexpr int K = 64; };
template <> struct HyFrag<float> { typedef hy_v4f V; static constexpr int K = 32; };
__device__ __forceinline__ void hy_mma(hy_v16f& c, const hy_v8bf& a, const hy_v8bf& b) { c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ void hy_mma(hy_v16f& c, const hy_v4f& a, const hy_v4f& b) {
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], b[e], c, 0, 0, 0);
}

// WM x WN wavefronts, BM x BN results; EPI, GR and HyGroup as for hy_gemm_kernel (GR: blockIdx.y = row tile of the list, BM rows at most).
// Grid: x = mt nt ks workgroups (row tiles x column tiles x K splits of kper) rounded up to a multiple of 8; GR: x = column tiles.
template <typename T, int BM, int BN, int WM, int WN, int SA, int SW, int EPI, int GR = 0>
static __global__ __launch_bounds__(WM * WN * 64) void hy_gemm_ring_kernel(const T* __restrict__ A, int lda, const T* __restrict__ Wt, int ldw, int M, int N, int K,
                                                                           float* __restrict__ C, int ldc, T* __restrict__ act, int ld_act, HyGlu glu, int mt, int nt, int ks,
                                                                           int kper, HyGroup grp = HyGroup{}) {
    constexpr int NW = WM * WN, TM = BM / WM / 32, TN = BN / WN / 32, BK = HyFrag<T>::K;
    constexpr int PA = BM / 8, PW = BN / 8, NPA = (PA + NW - 1) / NW, NPW = (PW + NW - 1) / NW, NP = NPA + NPW;      // 1 KB pieces (8 rows) of a stage, per wavefront
    constexpr int SZA = BM * 128, SZW = BN * 128, OW = SA * SZA;
    static_assert(SW > SA && SA >= 2 && NPA * NW < 2 * PA + NW && TM * WM * 32 == BM && TN * WN * 32 == BN, "tile layout");
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
            if (u >= u0 && u < u1) hy_dma16(w + offw[u], smem + slot * SZW + pw[u]);
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
    constexpr int NR = TM + TN, MPR = sizeof(T) == 2 ? 1 : 4, NM = TM * TN * MPR;
#define HY_QUARTER(ND)                                                              \
    do {                                                                            \
        _Pragma("unroll") for (int q_ = 0; q_ < NR; ++q_) {                         \
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                      \
            if ((q_ + 1) * MPR <= NM) __builtin_amdgcn_sched_group_barrier(0x8, MPR, 0); \
            if (q_ < (ND)) __builtin_amdgcn_sched_group_barrier(0x20, 1, 0);        \
        }                                                                           \
        if (NM > NR * MPR) __builtin_amdgcn_sched_group_barrier(0x8, NM - NR * MPR, 0); \
        __builtin_amdgcn_sched_barrier(0);                                          \
    } while (0)
    // step s (behind barrier s) starts the loads of A's stage s + SA (into the slot the barrier freed) and, in the two quarters after it,
    // of W's stage s + SW; the steps before 0 are the prologue, the last one's W belongs to the loop's first round
    constexpr int LEFT = (SA - 2) * NP + NPW;          // loads started behind A's stage s + 1 when barrier s waits for it
#pragma unroll
    for (int s = -SW; s < 0; ++s) {
        if (s + SA >= 0 && s + SA < n_it) issue_a(s + SA, s + SA);
        if (s < -1 && s + SW < n_it) issue_w(s + SW, s + SW, 0, NPW);
    }
    if (n_it >= SW) hy_wait_barrier<(SA - 1) * NP>(); else hy_wait_barrier<0>();
    rd(0, 0, 0, 0);
    int sa = 0, sw = 0, sp = SW - 1, it = 0;          // slots of the current stage; sp: the W slot that the step before fills
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
        if (sizeof(T) == 4 && it % HY_FLUSH == HY_FLUSH - 1) flush();
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
        if (sizeof(T) == 4 && it % HY_FLUSH == HY_FLUSH - 1) flush();
    }
    if constexpr (sizeof(T) == 4) {
        flush();
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = tot[i][j];
    }
#undef HY_QUARTER
    // lane holds column lane % 32 and rows 8 (r / 4) + 4 (lane / 32) + r % 4 of every 32 x 32 tile
    const int mb = m0 + wm * (BM / WM) + 4 * kh, nb = n0 + wn * (BN / WN) + r32;
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
