// gl3_hy_pre_kernels.h — one token's residual update and norm as the beginning of the product behind them.
//
// What it saves.  The update of a row (streams or plain residual, K-split parts, an optional norm of what joins) is a launch of one workgroup: 4 - 5 us with its boundary,
// four to six times a token, while a product of 8 MB waits.  Here every workgroup of the product makes the whole row itself (24 - 48 KB from L2, 16 bytes a thread) under
// the first weights it has already asked for; workgroup 0 keeps the new residual (in the other of two buffers: the others still read the old one) and the normed row for
// later readers.  That wants few workgroups (every one reads the row): one of sixteen wavefronts per CU, pairs of weight rows dealt out over the wavefronts, the next
// pair's pieces on their way while one is multiplied.
//
// Every sum is taken in the order of the kernels it stands for (hy_streams4_kernel or hy_resid_kernel on 1024 threads, then hy_matvec_kernel), to the bit: a plan's results do
// not depend on whether an update was deferred, and a lane's chain of products is no longer here than there.  So four wavefronts share a pair (KS = 4) where that kernel splits K:
// up to 16384 rows of 1024 columns and more; a lane of one wavefront alone would add K / 64 products in one chain instead of K / 256, an error of 1.2e-7 instead of 0.95e-7
// (K = 2048, float32 plans).  Both splits take the same time once the sums cross the wavefront in registers: 4608 - 12000 x 2048 in bfloat16 10.2 - 11.0 us (one wavefront a
// pair 10.8 - 11.3), 8192 x 2048 in float32 14.9 (15.1).
#pragma once
#include "gl3_hybrid.h"
#include "gl3_hy_kernels.h"
#include "gl3_hy_heads_kernels.h"

// hy_wave_sum without LDS, the same sums in the same order: lanes l ^ 32, l ^ 16, then within rows of 16, whose values repeat every 8, 4, 2 by then (a turn by as many is the exchange)
__device__ __forceinline__ float hy_wave_sum_vec(float v) {
    auto swap = [](uint32_t x, auto f) { const auto r = f(x); return __uint_as_float(r[0]) + __uint_as_float(r[1]); };
    v = swap(__float_as_uint(v), [](uint32_t x) { return __builtin_amdgcn_permlane32_swap(x, x, false, false); });
    v = swap(__float_as_uint(v), [](uint32_t x) { return __builtin_amdgcn_permlane16_swap(x, x, false, false); });
    v += hy_dpp<0x128>(v);          // row_ror 8, 4, 2, 1
    v += hy_dpp<0x124>(v);
    v += hy_dpp<0x122>(v);
    return v + hy_dpp<0x121>(v);
}

// UN: a wavefront's places of the walk that are loaded together
template <typename T, int S, int EPI, int KS, int UN, bool ONCE>
static __global__ __launch_bounds__(1024) void hy_matvec_pre_kernel(HyPre p, const T* __restrict__ Wt, int ldw, int N, float* __restrict__ C, T* __restrict__ act, int ld_act, HyGlu glu) {
    constexpr int PE = HyPiece<T>::N, STEP = KS * 64 * PE;
    __shared__ __attribute__((aligned(16))) T sh[4096];
    __shared__ float red[16], part[HY_PRE_SPLIT_PAIRS * 4][2];
    const int K = p.W, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pairs = (N + 1) >> 1, each = pairs / (int)gridDim.x, over = pairs % (int)gridDim.x;
    const int pair0 = (int)blockIdx.x * each + min((int)blockIdx.x, over), mine = each + ((int)blockIdx.x < over);          // pairs in a row, so that results leave in whole lines
    const int kp = wave % KS, slots = 16 / KS, first = wave / KS, chunks = (K + UN * STEP - 1) / (UN * STEP), todo = first < mine ? ((mine - 1 - first) / slots + 1) * chunks : 0;
    auto row0 = [&](int i) { const int pr = pair0 + i; return EPI == HY_EPI_GLU ? (pr >> 5) * 64 + (pr & 31) : 2 * pr; };
    auto row1 = [&](int r0) { return EPI == HY_EPI_GLU ? r0 + 32 : r0 + 1; };
    uint4 a[2][UN], b[2][UN];
    auto fetch = [&](int set, int q) {          // chunk q of this wavefront's walk (places past K repeat the last one: not multiplied)
        const int r0 = row0(first + q / chunks * slots), r1 = row1(r0), k = q % chunks * UN * STEP + (kp * 64 + lane) * PE;
        const T *w0 = Wt + (size_t)r0 * ldw, *w1 = Wt + (size_t)(r1 < N ? r1 : r0) * ldw;
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            const int ku = min(k + u * STEP, K - PE);
            a[set][u] = hy_ld_weights<ONCE>(w0 + ku);
            b[set][u] = hy_ld_weights<ONCE>(w1 + ku);
        }
    };
    const int w = 4 * tid;
    const bool on = w < K;
    float xs[S][4], yv[4] = {0.f, 0.f, 0.f, 0.f}, pw[4], nw[4];
    if (on) {          // the row first: the weights' answers come in order behind it
#pragma unroll
        for (int s = 0; s < S; ++s) hy_ldv<4>(p.x + s * p.xs + w, xs[s]);
        hy_ldv<4>(p.y + w, yv);
        hy_ldv<4>(p.norm_w + w, nw);
        if (p.post_w) hy_ldv<4>(p.post_w + w, pw);
    }
    if (todo > 0) fetch(0, 0);
    __builtin_amdgcn_sched_barrier(0);
    for (int z = 1; z < p.yparts; ++z) {
        float q[4];
        if (on) {
            hy_ldv<4>(p.y + z * p.ystride + w, q);
#pragma unroll
            for (int i = 0; i < 4; ++i) yv[i] += q[i];
        }
    }
    if (p.post_w) {
        float sd = 0.f;
        if (on)
#pragma unroll
            for (int i = 0; i < 4; ++i) { yv[i] *= p.y_mul; sd = fmaf(yv[i], yv[i], sd); }
        sd = hy_block_sum<1024>(sd, red);
        const float r = 1.f / sqrtf(sd / (float)K + p.eps);
        if (on)
#pragma unroll
            for (int i = 0; i < 4; ++i) yv[i] = yv[i] * r * pw[i];
        __syncthreads();          // red again
    }
    float ss = 0.f, h[4];
    if (on) {
        float nx[S][4];
#pragma unroll
        for (int u = 0; u < S; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (S == 1 && !p.mix) nx[0][i] = p.post_w ? xs[0][i] + yv[i] : fmaf(p.y_mul, yv[i], xs[0][i]);
                else {
                    float t = p.mix[u] * xs[0][i];
#pragma unroll
                    for (int s = 1; s < S; ++s) t = fmaf(p.mix[s * S + u], xs[s][i], t);
                    nx[u][i] = fmaf(p.po[u], yv[i], t);
                }
            }
        if (blockIdx.x == 0)
#pragma unroll
            for (int s = 0; s < S; ++s) hy_stv<4>(p.x_out + s * p.xos + w, nx[s]);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            h[i] = (p.pi ? p.pi[0] : 1.f) * nx[0][i];
#pragma unroll
            for (int s = 1; s < S; ++s) h[i] = fmaf(p.pi[s], nx[s][i], h[i]);
            ss = fmaf(h[i], h[i], ss);
        }
    }
    ss = hy_block_sum<1024>(ss, red);
    const float r = 1.f / sqrtf(ss / (float)K + p.eps);
    if (on) {
#pragma unroll
        for (int i = 0; i < 4; ++i) h[i] = h[i] * r * nw[i];
        hy_stv<4>(sh + w, h);
        if (blockIdx.x == 0) hy_stv<4>((T*)p.h_out + w, h);
    }
    __syncthreads();
    auto store = [&](int i, float s0, float s1) {
        const int r0 = row0(i), r1 = row1(r0);
        const bool has1 = r1 < N;
        if constexpr (EPI == HY_EPI_GLU) {
            const int f = (r0 >> 6) * 32 + (r0 & 31);
            if (f < ld_act) hy_st(act + f, hy_glu(s0, has1 ? s1 : 0.f, glu));
        } else if constexpr (EPI == HY_EPI_ACTMUL) {
            hy_st(act + r0, hy_actmul<T>(s0, 0, r0, glu));
            if (has1) hy_st(act + r1, hy_actmul<T>(s1, 0, r1, glu));
        } else {
            hy_put2(C, r0, has1, s0, s1, glu);
        }
    };
    float a0 = 0.f, a1 = 0.f;
    auto take = [&](int set, int q) {
        const int c = q % chunks, k = c * UN * STEP + (kp * 64 + lane) * PE;
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
            const int i = first + q / chunks * slots;
            if (lane == 0) { if constexpr (KS == 1) store(i, s0, s1); else { part[i * KS + kp][0] = s0; part[i * KS + kp][1] = s1; } }
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
    if constexpr (KS > 1) {
        __syncthreads();
        if (tid < mine) {
            const float (*s)[2] = part + tid * KS;
            store(tid, (s[0][0] + s[1][0]) + (s[2][0] + s[3][0]), (s[0][1] + s[1][1]) + (s[2][1] + s[3][1]));
        }
    }
}
