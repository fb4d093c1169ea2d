// gl3_hy_beside_kernels.h — one token: launches that nothing orders, side by side in one.
//
// A token's launches stand one behind the other, each with 1 us of boundary and 2 - 3 us until its loads answer and its last workgroup has left, and a mixer or a choice of experts
// keeps some dozens of CUs busy (or one) while the others wait.  Where two of them read the same row, their workgroups share a launch:
//   * parallel blocks (one norm feeds mixer and feed-forward): the mixer's workgroups and the gate / up product's; output and down projections, whose sums the next update adds;
//   * mixtures of experts with a shared expert: the choice of the experts and the shared gate / up product; the chosen experts' and the shared expert's down projections.
// Every product keeps its own kernel's arithmetic (hy_matvec), so results are the same bits as from the launches apart.  us, apart / together: gate and up beside a mixer in hy_mixer_up (gl3_hybrid.hip);
// output 2048 x 4096 and down 2048 x 8192 in bfloat16 5.4 + 7.7 / 10.3; choice of 4 of 32 and shared gate / up 8192 x 2048 in float32 4.4 + 13.4 / 13.7; down projections of four experts and the shared one
// 8.1 + 8.4 / 13.8.  One token, medians of 30 calls in turn (GL3_HY_APART): three layers of Kosusun 768 wide bfloat16 110 / 88, 1000 x 8192 136 / 107, 1B 164 / 145, behind 640 positions 169 / 143, 8B
// 355 / 348, behind 300 362 / 348; float32 1B 232 / 228, behind 640 243 / 235, 2048 x 16384 318 / 323, 8B 616 / 622, behind 300 625 / 621; Kugadra 1B float32 185 / 178, bfloat16 227 / 213.
// Bound: the weights' bytes; the mixers' chains hide behind them.
#pragma once
#include "gl3_hy_one_kernels.h"
#include "gl3_hy_plain_kernels.h"
#include "gl3_hy_pre_kernels.h"

template <typename T>
struct HyMv {                  // one token's product, as hy_matvec takes it
    const T* A; int lda;
    const T* W; int ldw, N, K;
    float* C; int ldc;
    T* act; int ld_act;
    HyGlu glu;
    const int* sel; size_t wstride; int a_div; const float* row_scale; int n_sel;          // grouped
};
template <typename T, int EPI, int KS, int GR, int SUB, bool ONCE>
__device__ __forceinline__ void hy_matvec(int bx, int by, const HyMv<T>& p) {
    hy_matvec<T, T, 1, EPI, KS, GR, SUB, ONCE>(bx, by, p.A, p.lda, p.W, p.ldw, 1, p.N, p.K, p.C, p.ldc, p.act, p.ld_act, p.glu, p.sel, p.wstride, p.a_div, p.row_scale, p.n_sel);
}

// Two products: workgroups 0 .. wp - 1 make p, the others q (GR: gx workgroups per pair).
template <typename T, int KS, int GR, bool ONCE>
static __global__ __launch_bounds__(256) void hy_matvec_two_kernel(HyMv<T> p, int wp, HyMv<T> q, int gx) {
    const int b = blockIdx.x;
    if (b < wp) { hy_matvec<T, HY_EPI_STORE, KS, 0, 1, ONCE>(b, 0, p); return; }
    if constexpr (GR) hy_matvec<T, HY_EPI_STORE, KS, 1, 1, ONCE>((b - wp) % gx, (b - wp) / gx, q);
    else hy_matvec<T, HY_EPI_STORE, KS, 0, 1, ONCE>(b - wp, 0, q);
}

// Gate and up rows by workgroups of sixteen wavefronts that stay: pairs wg 16 + wavefront, + 16 wgs .., a pair's next pieces on their way while the ones before are multiplied, the token's
// row in LDS.  Every lane's chain is hy_matvec's (KS = 1).  K a multiple of a piece, rows of at most HY_WALK_BYTES: with longer ones hy_matvec's wavefronts of one pair have enough on their way.  One token
// of three layers, us, one pair a wavefront / walked: bfloat16 1000 x 4128 100.0 / 95.3, 1000 x 16384 147 / 128, 2048 x 8192 147.8 / 144.9, 2048 x 16384 192 / 184, 3072 x 8192 181.7 / 177.3, 4096 x 14336
// 347.5 / 353.7; float32 1000 x 8192 144 / 138, 1536 x 8192 174.2 / 173.6, 2048 x 8192 227.9 / 231.2, 3072 x 8192 284.9 / 289.1.  (A mixer's registers leave a CU one workgroup.  A piece of
// either row at a time: two and four put more on the way than the mixers' loads can stand behind, whole requests 3845 us, 3960, 3925.)
constexpr int HY_WALK_BYTES = 6 * 1024;
template <typename T, bool ONCE>
__device__ __forceinline__ void hy_walk_glu(int wg, int wgs, const HyMv<T>& p) {
    constexpr int PE = HyPiece<T>::N, UN = 1, STEP = 64 * PE;
    __shared__ __attribute__((aligned(16))) T sh[HY_WALK_BYTES / sizeof(T)];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), K = p.K;
    const int pairs = p.N >> 1, first = wg * 16 + wave, stride = wgs * 16, chunks = (K + UN * STEP - 1) / (UN * STEP), todo = first < pairs ? ((pairs - 1 - first) / stride + 1) * chunks : 0;
    uint4 a[2][UN], b[2][UN];
    auto fetch = [&](int set, int q) {          // (places past K repeat the last one: not multiplied)
        const int pr = first + q / chunks * stride, k = q % chunks * UN * STEP + lane * PE;
        const T *w0 = p.W + (size_t)((pr >> 5) * 64 + (pr & 31)) * p.ldw, *w1 = w0 + (size_t)32 * p.ldw;
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int ku = min(k + u * STEP, K - PE);
            a[set][u] = hy_ld_weights<ONCE>(w0 + ku);
            b[set][u] = hy_ld_weights<ONCE>(w1 + ku);
        }
    };
    const uint4 row = *reinterpret_cast<const uint4*>(p.A + min(tid * PE, K - PE));          // first: the weights' answers come in order behind it
    __builtin_amdgcn_sched_barrier(0);
    if (todo > 0) fetch(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    if (tid * PE < K) *reinterpret_cast<uint4*>(sh + tid * PE) = row;
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");          // (without the wait for the weights that __syncthreads has)
    float a0 = 0.f, a1 = 0.f;
    auto take = [&](int set, int q) {
        const int c = q % chunks, k = c * UN * STEP + lane * PE;
        if (c == 0) a0 = a1 = 0.f;
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            if (k + u * STEP >= K) continue;
            float f0[PE], f1[PE], fx[PE];
            hy_widen(a[set][u], f0, (const T*)nullptr);
            hy_widen(b[set][u], f1, (const T*)nullptr);
            hy_widen(*reinterpret_cast<const uint4*>(sh + k + u * STEP), fx, (const T*)nullptr);
#pragma unroll
            for (int i = 0; i < PE; ++i) { a0 = fmaf(fx[i], f0[i], a0); a1 = fmaf(fx[i], f1[i], a1); }
        }
        if (c + 1 == chunks) {
            const float s0 = hy_wave_sum_vec(a0), s1 = hy_wave_sum_vec(a1);
            const int pr = first + q / chunks * stride;
            if (lane == 0 && pr < p.ld_act) hy_st(p.act + pr, hy_glu(s0, s1, p.glu));
        }
    };
    int q = 0;
    for (; q + 2 <= todo; q += 2) {
        fetch(1, q + 1);
        take(0, q);
        if (q + 2 < todo) fetch(0, q + 2);
        take(1, q + 1);
    }
    if (q < todo) take(0, q);
}

// A mixer (attention, a matrix memory or both: gl3_hy_one_kernels.h) in the first workgroups, gate and up rows of the feed-forward in the others, sixteen wavefronts each.
template <typename T, int NI, int QN, int KS, bool ONCE>          // KS = 0: hy_walk_glu
static __global__ __launch_bounds__(1024) void hy_mixer_up_kernel(HyAttnOne a, T* __restrict__ out_a, HyScanOut b, T* __restrict__ out_b, HyMv<T> f) {
    const int w = blockIdx.x, mixers = a.H + b.s.heads;
    if (w < a.H) hy_attn_one<T, NI>(a, out_a, w);
    else if (w < mixers) hy_scan_out<T, QN>(b, out_b, w - a.H);
    else if constexpr (KS == 0) hy_walk_glu<T, ONCE>(w - mixers, (int)gridDim.x - mixers, f);
    else hy_matvec<T, HY_EPI_GLU, KS, 0, 4, ONCE>(w - mixers, 0, f);
}

// The token's choice of experts in workgroup 0, gate and up rows of the shared expert in the others.
struct HyRouteArgs { const float* z; int ldz, parts; size_t pstride; int E, top; int* sel; float* wgt; int* pair_row; float* extra_out; HyRoute rt; };
template <typename T, int PER, int KS, bool ONCE>
static __global__ __launch_bounds__(256) void hy_route_up_kernel(HyRouteArgs r, HyMv<T> f) {
    if (blockIdx.x > 0) { hy_matvec<T, HY_EPI_GLU, KS, 0, 1, ONCE>((int)blockIdx.x - 1, 0, f); return; }
    if (threadIdx.x < 64) hy_route<PER>(0, r.z, r.ldz, r.parts, r.pstride, r.E, r.top, r.sel, r.wgt, r.pair_row, r.extra_out, r.rt);
}
