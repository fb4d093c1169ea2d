// gl3_hy_scan_chunk.h — the recurrences with one decay per head and token (HyScanArgs modes 0 - 2: state-space layers, matrix memories with exponential
// gates or a fixed decay) over portions of many tokens, 32 tokens at a time as matrix products.
//
// S_t = a_t S_(t-1) + b_t k_t x_t^T, y_t = S_t^T q_t walked token by token is a chain of n steps that no number of workgroups shortens
// (hy_ssm_scan_kernel: 0.35 - 0.5 us a token at the sizes below).  With L[t][s] = a_(s+1) .. a_t inside a chunk and A_t = a_first .. a_t:
//     y_t = A_t S^T q_t + sum_(s <= t) (q_t . k_s) L[t][s] b_s x_s,        S <- A_last S + sum_s k_s (L[last][s] b_s x_s)^T,
// all products on the float32 matrix cores (v_mfma_f32_16x16x4_f32).  L is made of products, not of quotients of running products or of
// exponentials of summed logarithms: a strong decay underflows to its limit and nothing cancels.
// Workgroup = one head x PC value columns.  Four wavefronts make a chunk (rows to LDS; q . k in three 16 x 16 tiles by three of them while the fourth makes L; the masked
// product) one chunk ahead of four that walk: walker w keeps the N / 4 state rows from w N / 4 on in accumulators, and since register r of a lane is row 4 (lane / 16) + r
// of its tile, they are the second operand of Q S as they stand; it adds its rows' share of Q S and its eight tokens' share of the masked product to y (joined in LDS) and
// updates its rows.  Each SIMD has a maker and a walker, three barriers a chunk, two chunk buffers; the chunk behind travels in the makers' registers.  (One group of four
// wavefronts doing both in turn: five barriers, and one wavefront per SIMD that waits for each of its LDS reads and MFMA chains alone.)
// A token whose x is not finite must not reach the tokens in front of it, and a product with its zero place in the masked matrix would carry it there:
// the matrix cores take zero in its stead, and a chunk that holds one (looked for on the way into LDS) adds its products entry by entry as y is written.
// Keys and queries come finished (hy_scan_prep_kernel); x passes through silu on the way into LDS where the layer asks for it (act & 4).
// Measured for 512 tokens (us), hy_ssm_scan_kernel -> one group of four wavefronts -> this: 128 heads x (128 x 64) 278 -> 80 -> 70, 16 x (128 x 256) 310 -> 53 -> 43, 8 x (256 x 513)
// 430 -> 99 -> 87 (88 tokens: 15.6 -> 13.3 and 26 -> 25); the look for an x that is not finite is 1 - 3 us of them.
#pragma once
#include "gl3_hy_attn_mfma.h"

// workgroup barrier for LDS alone (__syncthreads() also waits for every global load in flight: the next chunk's rows)
__device__ __forceinline__ void hy_lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ hy_acc4 hy_mma4(float a, float b, hy_acc4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Keys and queries of a whole portion in place, as the recurrence takes them: silu (act 1: keys, 2: queries), the multiplier, the turn by the
// position (HyScanRot).  One workgroup per token; the angles are shared by the heads.  (1024 threads: in place, a thread's pairs wait for each other; 88 and 512 tokens of 16 heads
// x 128 5.0 and 8.0 us, 8.9 and 10.6 with 256 threads.)
static __global__ __launch_bounds__(1024) void hy_scan_prep_kernel(float* __restrict__ proj, int ld, int q_off, int k_off, int heads, int N, float q_mul, float k_mul, int act,
                                                                  HyScanRot rot, const int* __restrict__ dyn) {
    extern __shared__ float sc[];          // cosines, sines of rot.dims / 2 angles
    const int half = rot.dims >> 1, pos = dyn[0] + blockIdx.x;
    for (int j = threadIdx.x; j < half; j += 1024) sincosf((float)pos * rot.freq[j], &sc[half + j], &sc[j]);
    __syncthreads();
    float* row = proj + (size_t)blockIdx.x * ld;
    const int pairs = N - half;            // per head: half pairs, then single entries
    for (int i = threadIdx.x; i < 2 * heads * pairs; i += 1024) {
        const int which = i / (heads * pairs), h = i / pairs % heads, j = i % pairs;
        float* r = row + (which ? k_off : q_off) + h * N;
        const float mul = which ? k_mul : q_mul;
        const bool si = act & (which ? 1 : 2);
        if (j < half) {
            const int i0 = rot.interleaved ? 2 * j : j, i1 = rot.interleaved ? 2 * j + 1 : j + half;
            const float u = (si ? hy_silu(r[i0]) : r[i0]) * mul, v = (si ? hy_silu(r[i1]) : r[i1]) * mul;
            r[i0] = u * sc[j] - v * sc[half + j];
            r[i1] = v * sc[j] + u * sc[half + j];
        } else {
            const int d = j + half;
            r[d] = (si ? hy_silu(r[d]) : r[d]) * mul;
        }
    }
}

// floats of one chunk's buffer in LDS (there are two)
__host__ __device__ constexpr int hy_chunk_floats(int N, int PC) { return 2 * 32 * (N + 4) + 32 * (PC + 4) + 32 * 36 + 32 * 33 + 68; }
template <int NT, int PC>          // N = 64 NT states per column, PC value columns
static __global__ __launch_bounds__(512, 2) void hy_scan_chunk_kernel(HyScanArgs a) {
    constexpr int C = 32, N = 64 * NT, QS = N + 4, XS = PC + 4, JC = PC / 16, NV = C * N / 4 / 256, XV = C * PC / 256;
    static_assert(4 * C * PC <= C * QS, "the shares of y end where the query rows do: x and the masked product behind them are still read while the shares are written");
    extern __shared__ __attribute__((aligned(16))) float smem[];
    constexpr int BUF = hy_chunk_floats(N, PC);
    struct Buf {                         // one chunk
        float *K, *Q, *X, *M, *L, *A;    // [C][QS] keys, [C][QS] queries, [C][XS], [C][36] masked, weighted q . k, [C][33], [C] a + [C] b
        int* F;                          // [4] whether a wavefront staged an x that is not finite
        float* Y;                        // [4][C][PC] the wavefronts' shares of y, when the query rows have been read
    };
    auto buffer = [&](int b) {
        Buf r;
        r.K = smem + b * BUF; r.Q = r.K + C * QS; r.X = r.Q + C * QS; r.M = r.X + C * XS; r.L = r.M + C * 36; r.A = r.L + C * 33; r.F = (int*)(r.A + 2 * C); r.Y = r.Q;
        return r;
    };
    const int tid = threadIdx.x & 255, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3), l16 = lane & 15, g = lane >> 4;
    const bool maker = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int P = a.P, n = a.n, Px = P - (a.ones_col ? 1 : 0), head = blockIdx.y, col0 = blockIdx.x * PC, gr = head / (a.heads / a.G), nc = (n + C - 1) / C;
    for (int i = threadIdx.x; i < 2 * 16 * 16; i += 512) buffer(i >> 8).M[((i >> 4) & 15) * 36 + 16 + (i & 15)] = 0.f;          // tokens 0 - 15 see none of 16 - 31
    if (maker) {
        const float* kbase = a.ksrc + a.k_off + (size_t)gr * a.k_hstride;
        const float* qbase = a.qsrc + a.q_off + (size_t)gr * a.q_hstride;
        const float* xbase = a.xsrc + a.x_off + (size_t)head * Px;
        const float na = a.mode == 0 ? -expf(a.A_log[head]) : 0.f, dtb = a.mode == 0 ? a.dt_bias[head] : 0.f, fixed = a.mode == 2 ? a.decay[head] : 0.f;
        const float* pa = a.mode == 0 ? a.dtsrc + a.dt_off + head : a.mode == 1 ? a.ga + head : kbase;          // (mode 2 has no source: any readable place)
        const float* pb = a.mode == 1 ? a.gb + head : pa;
        const int lda = a.mode == 0 ? a.ld_dt : a.mode == 1 ? a.heads : 0;
        hy_acc4 rk[NV], rq[NV];
        float rx[XV], ra, rb;
        auto load = [&](int t0) {          // unconditional (a guarded load is waited for at once); rows past the portion's end repeat the last one
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int i = tid + u * 256, t = min(t0 + i / (N / 4), n - 1), c = 4 * (i % (N / 4));
                rk[u] = *reinterpret_cast<const hy_acc4*>(kbase + (size_t)t * a.ldk + c);
                rq[u] = *reinterpret_cast<const hy_acc4*>(qbase + (size_t)t * a.ldq + c);
            }
#pragma unroll
            for (int u = 0; u < XV; ++u) {
                const int i = tid + u * 256;
                rx[u] = xbase[(size_t)min(t0 + i / PC, n - 1) * a.ldx + min(col0 + i % PC, Px - 1)];
            }
            const int t = min(t0 + (tid & (C - 1)), n - 1);
            ra = pa[(size_t)t * lda]; rb = pb[(size_t)t * lda];
        };
        load(0);
        for (int q = 0; q < nc; ++q) {
            const Buf s = buffer(q & 1);
            const int t0 = q * C;          // tokens past the end: zero rows, a = 1, b = 0
#pragma unroll
            for (int u = 0; u < NV; ++u) {
                const int i = tid + u * 256, t = i / (N / 4), c = 4 * (i % (N / 4));
                const bool live = t0 + t < n;
                hy_acc4 kv, qv;
#pragma unroll
                for (int e = 0; e < 4; ++e) { kv[e] = live ? rk[u][e] : 0.f; qv[e] = live ? rq[u][e] : 0.f; }
                *reinterpret_cast<hy_acc4*>(s.K + t * QS + c) = kv;
                *reinterpret_cast<hy_acc4*>(s.Q + t * QS + c) = qv;
            }
            bool odd = false;
#pragma unroll
            for (int u = 0; u < XV; ++u) {
                const int i = tid + u * 256, p = col0 + i % PC;
                float x = (a.act & 4) ? hy_silu(rx[u]) : rx[u];
                x = t0 + i / PC >= n ? 0.f : p < Px ? x : p < P ? 1.f : 0.f;
                s.X[(i / PC) * XS + i % PC] = x;
                odd |= !(fabsf(x) < INFINITY);
            }
            const bool wodd = __any(odd);
            if (lane == 0) s.F[wave] = wodd;
            if (tid < C) {
                float av = 1.f, bv = 0.f;
                if (t0 + tid < n) {
                    if (a.mode == 0) { bv = hy_softplus(ra + dtb); av = expf(na * bv); }
                    else { av = a.mode == 1 ? ra : fixed; bv = a.mode == 1 ? rb : 1.f; }
                }
                s.A[tid] = av; s.A[C + tid] = bv;
            }
            hy_lds_barrier();
            load(t0 + C);
            hy_acc4 g0, g1;
#pragma unroll
            for (int r = 0; r < 4; ++r) g0[r] = g1[r] = 0.f;
            const int tt = wave == 0 ? 0 : 16, ss = wave == 2 ? 16 : 0;          // wavefronts 0 - 2: tiles (0, 0), (16, 0), (16, 16) of q . k
            if (wave < 3) {
                const float *q = s.Q + (tt + l16) * QS + 4 * g, *k = s.K + (ss + l16) * QS + 4 * g;
#pragma unroll 8
                for (int c = 0; c < N; c += 16) {
                    const float4 qv = *reinterpret_cast<const float4*>(q + c), kv = *reinterpret_cast<const float4*>(k + c);
                    g0 = hy_mma4(qv.x, kv.x, g0); g1 = hy_mma4(qv.y, kv.y, g1);
                    g0 = hy_mma4(qv.z, kv.z, g0); g1 = hy_mma4(qv.w, kv.w, g1);
                }
            } else {                                                              // the fourth: lane s (and s + 32, the same) makes L[0 ..][s]
                int sl = lane & 31;
                asm volatile("" : "+v"(sl));          // (32 comparisons kept from chunk to chunk would spill)
                const float av = s.A[sl];
                float l = 1.f;
#pragma unroll
                for (int t = 0; t < C; ++t) {
                    const float at = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(av), t));
                    l = t > sl ? l * at : l;
                    s.L[t * 33 + sl] = t >= sl ? l : 0.f;
                }
            }
            hy_lds_barrier();
            if (wave < 3) {
                const float bs = s.A[C + ss + l16];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int t = tt + 4 * g + r;
                    s.M[t * 36 + ss + l16] = t >= ss + l16 ? (g0[r] + g1[r]) * (s.L[t * 33 + ss + l16] * bs) : 0.f;          // (chosen: a later key may be infinite)
                }
            }
            hy_lds_barrier();
        }
#pragma unroll
        for (int i = 0; i < 3; ++i) hy_lds_barrier();          // (the walkers' last chunk)
        return;
    }
    float* S = a.state + (size_t)a.dyn[1] * a.slot_stride + (size_t)head * N * P;
    const bool fresh = a.dyn[0] == 0;
    const float dd = (a.mode == 0 && a.Dp) ? a.Dp[head] : 0.f;
    hy_acc4 st[NT][JC];
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < JC; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int nn = (wave * NT + i) * 16 + 4 * g + r, p = col0 + 16 * j + l16;
                st[i][j][r] = (!fresh && p < P) ? S[(size_t)nn * P + p] : 0.f;
            }
#pragma unroll
    for (int i = 0; i < 3; ++i) hy_lds_barrier();              // (the makers' first chunk)
    for (int q = 0; q < nc; ++q) {
        const Buf s = buffer(q & 1);
        const int t0 = q * C;
        hy_acc4 y[2][JC];
        const float a0 = s.A[0];
        const int entries = __builtin_amdgcn_readfirstlane((s.F[0] | s.F[1]) | (s.F[2] | s.F[3]));
#pragma unroll
        for (int u = 0; u < 2; ++u) {
#pragma unroll
            for (int j = 0; j < JC; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) y[u][j][r] = 0.f;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const float4 qv = *reinterpret_cast<const float4*>(s.Q + (16 * u + l16) * QS + (wave * NT + i) * 16 + 4 * g);
                const float q4[4] = {qv.x, qv.y, qv.z, qv.w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < JC; ++j) y[u][j] = hy_mma4(q4[e], st[i][j][e], y[u][j]);
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float at = s.L[(16 * u + 4 * g + r) * 33] * a0;
#pragma unroll
                for (int j = 0; j < JC; ++j) y[u][j][r] *= at;
            }
        }
        hy_lds_barrier();
#pragma unroll
        for (int e = 0; e < 2; ++e) {          // this wavefront's eight tokens s of the masked product
            const int tk = 8 * wave + 4 * e + g;
            const float m0 = s.M[l16 * 36 + tk], m1 = s.M[(16 + l16) * 36 + tk];
#pragma unroll
            for (int j = 0; j < JC; ++j) {
                float x = s.X[tk * XS + 16 * j + l16];
                x = fabsf(x) < INFINITY ? x : 0.f;
                y[0][j] = hy_mma4(m0, x, y[0][j]);
                y[1][j] = hy_mma4(m1, x, y[1][j]);
            }
        }
        const float ac = s.L[(C - 1) * 33] * a0;
#pragma unroll
        for (int i = 0; i < NT; ++i)
#pragma unroll
            for (int j = 0; j < JC; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) st[i][j][r] *= ac;
#pragma unroll
        for (int e = 0; e < 8; ++e) {          // k of the product: lane group g takes token tk (rows 4 apart: other LDS banks)
            const int tk = (e & 3) + 4 * g + 16 * (e >> 2);
            const float w = s.L[(C - 1) * 33 + tk] * s.A[C + tk];
            float x[JC];
#pragma unroll
            for (int j = 0; j < JC; ++j) x[j] = s.X[tk * XS + 16 * j + l16] * w;
#pragma unroll
            for (int i = 0; i < NT; ++i) {
                const float k = s.K[tk * QS + (wave * NT + i) * 16 + l16];
#pragma unroll
                for (int j = 0; j < JC; ++j) st[i][j] = hy_mma4(k, x[j], st[i][j]);
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int j = 0; j < JC; ++j)
#pragma unroll
                for (int r = 0; r < 4; ++r) s.Y[(wave * C + 16 * u + 4 * g + r) * PC + 16 * j + l16] = y[u][j][r];
        hy_lds_barrier();
        float v[XV], xs[XV];
#pragma unroll
        for (int u = 0; u < XV; ++u) {
            const int i = tid + u * 256;
            v[u] = (s.Y[i] + s.Y[C * PC + i]) + (s.Y[2 * C * PC + i] + s.Y[3 * C * PC + i]);
            xs[u] = s.X[(i / PC) * XS + i % PC];
        }
        if (entries)
#pragma unroll
            for (int u = 0; u < XV; ++u) {
                const int t = (tid + u * 256) / PC, c = (tid + u * 256) % PC;
#pragma unroll 1
                for (int sk = 0; sk <= t; ++sk) {
                    const float x = s.X[sk * XS + c];
                    if (!(fabsf(x) < INFINITY)) v[u] = fmaf(s.M[t * 36 + sk], x, v[u]);
                }
            }
#pragma unroll
        for (int u = 0; u < XV; ++u) {
            const int i = tid + u * 256, t = t0 + i / PC, p = col0 + i % PC;
            if (t < n && p < P) a.y[(size_t)t * a.ldy + head * P + p] = fmaf(dd, xs[u], v[u]);
        }
        hy_lds_barrier();
    }
#pragma unroll
    for (int i = 0; i < NT; ++i)
#pragma unroll
        for (int j = 0; j < JC; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int nn = (wave * NT + i) * 16 + 4 * g + r, p = col0 + 16 * j + l16;
                if (p < P) S[(size_t)nn * P + p] = st[i][j][r];
            }
}
