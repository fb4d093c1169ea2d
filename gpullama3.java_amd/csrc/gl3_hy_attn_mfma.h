// gl3_hy_attn_mfma.h — the attention core of the layer-list family for portions of many tokens, its products on the matrix cores
// (many tokens: float32 operands as three bfloat16 planes, the products of at least 2^-16 on v_mfma_f32_32x32x16_bf16, see gl3_hy_gemm.h; a few: v_mfma_f32_32x32x2_f32).
//
// Workgroup = (32 rows of a key / value head, key split): rows are (token, head of the group) pairs, token-major, as in hy_attn_kernel; its four
// wavefronts deal the key tiles of 32 out between them and join their sums in LDS at the end, so that 512 tokens x 32 heads are 512
// workgroups and no wavefront waits for another inside the key loop.  Both products are taken transposed, keys x rows and value columns x
// rows: a lane then holds ONE query row in all of them, the running maximum and sum are its own registers (one exchange with
// lane ^ 32 per tile), and the scores' accumulators ARE the second product's operand: register r of a lane is key 8 (r / 4) + 4 (lane / 32) + r % 4, so a half-wave's
// registers 0 - 7 and 8 - 15 are its eight keys of two MFMA steps, in the order in which it holds the values — nothing is transposed through LDS.
// Keys and values come straight from the cache (each wavefront its own tile): a lane reads its key row 32 bytes at a time (elements 16 c + 8 (lane / 32) .. + 7 of chunk c)
// and DVT consecutive value columns of the keys r (value column DVT m + i is row m of tile i); the values travel under the first product
// and the softmax, the next tile's keys under the second half of the second product (all at once do not fit 256 registers, and a second wavefront
// per SIMD is what covers the waits).  Queries (scaled) stay in LDS as planes; a step's MFMAs stand between the splits of the next step's keys or values, which the vector units
// make under them.  The scores have one chain (a second one was 16 registers spilled and 14 % of the kernel) in two passes: every chunk's small plane products, rounded to their own size,
// then the largest products of all chunks, whose key planes wait in registers.  Each product in turn as its chunk comes rounds six times per 16 entries to the size of the score: relative
// error of a head's output against 64 bits, head size 128, scores of one / of four, 512 tokens behind 1529: 4.5e-7 / 9.7e-7 against 3.5e-7 / 4.7e-7 as it is (float32 MFMAs
// 4.5e-7 / 7.9e-7; 192 entries, scores of four 7.1e-7, 3.2e-7, 5.2e-7), in the same time.
// A value that is not finite must stay with the rows that see its key, and the second product carries it to every row of the tile (p = 0 times infinity).  Nothing in the
// loops below looks for one (values cleaned in the tiles with unseen keys cost 1 and 5 % of the two kernels, right in front of every MFMA 6 - 12 %): sums that hold a
// not-a-number at the end are made once more, key by key on the vector units (hy_attn_again), which costs other inputs the look at the sums: 1 % of the kernel of
// many tokens, of that of few 2 % with 64 and 256 entries and 7 % with 512.  It stands behind the last exchange in LDS, which the loop's last MFMAs run under.  An infinite key
// or query entry has no planes: a row whose sum is not a number has its maximum and sum made again, in front of that exchange (hy_softmax_again), up to the first score that is none in float32
// either.  (Looking at the scores inside the loop: 2 % of the kernel, and 0.1 -> 1.0 - 4.9 ms for 512 tokens with queries or keys that are not numbers, 0.15 this way.)
// What bounds it: at position 0 a wavefront has two tiles on average and waits for memory half of its time (queries, first keys and the gate are asked for as early as they are
// known); behind many positions the splits (11 vector instructions per pair of values).  8 key / value heads x 4, head size 128, 512 tokens (us, float32 MFMAs -> now): at position 0 45 -> 34.5,
// behind 1529 176 -> 140 (launched over and over, caches warm; inside a prompt of 2041 tokens hy_attn_kernel took 131 at position 0, 1795 for the four portions).
#pragma once
#include "gl3_hy_gemm.h"

typedef float hy_acc4 __attribute__((ext_vector_type(4)));
template <int DVT> struct HyVec;
template <> struct HyVec<2> { typedef float2 V; };
template <> struct HyVec<4> { typedef float4 V; };

// The rare second passes: a lane's row, key by key in float32.  A score of k and q (which is multiplied first, as the planes' are).
template <int DK> __device__ __forceinline__ float hy_score(const float* __restrict__ k, const float* __restrict__ q, float qscale) {
    float s = 0.f;
#pragma unroll 4
    for (int d = 0; d < DK; d += 4) {
        const hy_v4f x = *reinterpret_cast<const hy_v4f*>(k + d), y = *reinterpret_cast<const hy_v4f*>(q + d);
#pragma unroll
        for (int e = 0; e < 4; ++e) s = fmaf(x[e], y[e] * qscale, s);
    }
    return s;
}
// Maximum and sum of a row whose sum is not a number: an infinity's planes and their products are none.  A score that is not a number without planes either leaves the row as it is: none.
template <int DK, typename Key>
__device__ __forceinline__ void hy_softmax_again(float& m, float& l, const HyAttnArgs& a, const float* q, float slope, int pr, int nbr, int win, const float* kc, const float* pkc, int vt0, int step,
                                                 int nv, Key key) {
    const int ldk = a.G * DK;
    float mx = -INFINITY, sum = 0.f;
    bool nan = false;
#pragma unroll 1
    for (int pass = 0; pass < 2; ++pass)
#pragma unroll 1
        for (int vt = vt0; vt < nv && !nan; vt += step) {
            int j, last;
            bool pooled;
            key(vt, j, last, pooled);
            last = min(j + 31, last);
#pragma unroll 1
            for (; j <= last && !nan; ++j) {
                if (!(pooled ? j < nbr : (j <= pr && (pr - j < win || j < a.keep)))) continue;
                float s = hy_score<DK>((pooled ? pkc : kc) + (size_t)j * ldk, q, a.scale);
                s = pooled ? s : s - slope * (float)(pr - j);
                if (pass == 0) { mx = fmaxf(mx, s); nan = s != s; }
                else sum += expf(s - (mx > -INFINITY ? mx : 0.f));
            }
        }
    if (!nan) { m = mx; l = sum; }
    if (l != l) m = INFINITY;          // (whoever joins the sums has none left)
}
// The weighted sums of a lane's row over the keys it sees, vt0, vt0 + step ... of the tile list (key(vt): first key, last one, pooled or not): register r of tile i is
// value column DVT (8 (r / 4) + 4 (lane / 32) + r % 4) + i behind col0.  q: the row's query; m: its maximum.
template <int DVT> __device__ __forceinline__ bool hy_attn_nan(const hy_v16f* o) {
    bool nan = false;
#pragma unroll
    for (int i = 0; i < DVT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) nan |= o[i][r] != o[i][r];
    return nan;
}
template <int DK, int DVT, typename Key>
__device__ __forceinline__ void hy_attn_again(hy_v16f* o, const HyAttnArgs& a, const float* q, float qscale, float scale, float m, float slope, int pr, int nbr, int win, const float* kc, const float* vc,
                                              const float* pkc, const float* pvc, int col0, int kh, int vt0, int step, int nv, Key key) {
#pragma unroll
    for (int i = 0; i < DVT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    const int ldk = a.G * DK, ldv = a.G * a.dv;
#pragma unroll 1
    for (int vt = vt0; vt < nv; vt += step) {
        int j, last;
        bool pooled;
        key(vt, j, last, pooled);
        last = min(j + 31, last);
#pragma unroll 1
        for (; j <= last; ++j) {
            if (!(pooled ? j < nbr : (j <= pr && (pr - j < win || j < a.keep)))) continue;
            const float *k = (pooled ? pkc : kc) + (size_t)j * ldk, *v = (pooled ? pvc : vc) + (size_t)j * ldv + col0 + DVT * 4 * kh;
            const float s = hy_score<DK>(k, q, qscale) * scale;
            const float p = expf((pooled ? s : s - slope * (float)(pr - j)) - m);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
#pragma unroll
                for (int i = 0; i < DVT; ++i) o[i][r] = fmaf(p, v[DVT * (8 * (r >> 2) + (r & 3)) + i], o[i][r]);
                __builtin_amdgcn_sched_barrier(0);          // (rarely run: a few loads at a time rather than registers for sixty-four)
            }
        }
    }
}

template <int DKC, int DVT>          // dk = 8 DKC, dv = 32 DVT
static __global__ __launch_bounds__(256, DKC > 16 ? 1 : 2) void hy_attn_mfma_kernel(HyAttnArgs a) {
    constexpr int DK = 8 * DKC, DV = 32 * DVT, CH = DK / 16, QB = 6 * DK + 16, OS = DV + 4;
    typedef typename HyVec<DVT>::V VV;
    __shared__ __attribute__((aligned(16))) uint8_t sQ[32 * QB];          // a row: its three planes
    __shared__ __attribute__((aligned(16))) float sO[32 * OS];
    __shared__ float sml[4][2][32];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r32 = lane & 31, kh = lane >> 5;
    // the LAST row block first: late tokens see the most keys
    const int g = blockIdx.x % a.G, rb = (int)(gridDim.x / a.G) - 1 - (int)(blockIdx.x / a.G), split = blockIdx.z, hpg = a.H / a.G;
    const int rows = a.n * hpg, row0 = rb * 32;
    // queries, then the first keys: both are on their way before the first is waited for
    constexpr int QI = (32 * (DK / 8) + 255) / 256;
    hy_v4f qs[QI][2];
#pragma unroll
    for (int u = 0; u < QI; ++u) {
        const int i = min(tid + 256 * u, 32 * (DK / 8) - 1), p = min(row0 + i / (DK / 8), rows - 1);          // (a row that is not there repeats the last one: its results are not stored)
        const float* src = a.q + (size_t)(p / hpg) * a.ldq + (size_t)(g * hpg + p % hpg) * DK + 8 * (i % (DK / 8));
        qs[u][0] = *reinterpret_cast<const hy_v4f*>(src);
        qs[u][1] = *reinterpret_cast<const hy_v4f*>(src + 4);
    }
    const int pos0 = a.dyn[0];
    const int minpos = pos0 + row0 / hpg, maxpos = pos0 + min(rows - 1, row0 + 31) / hpg;
    const int rho = row0 + r32, pr = rho < rows ? pos0 + rho / hpg : -1;          // this lane's row: position (-1: no such row), head
    const int hr = g * hpg + (rho < rows ? rho % hpg : 0);
    const float slope = a.slope_log2 != 0.f ? exp2f(-a.slope_log2 * (float)(hr + 1) / (float)a.H) : 0.f;
    const float* qrow = a.q + (size_t)(min(rho, rows - 1) / hpg) * a.ldq + (size_t)hr * DK;
    const size_t slot = (size_t)a.dyn[1] * a.slot_stride;
    const float *kc = a.kc + slot + (size_t)g * DK, *vc = a.vc + slot + (size_t)g * DV;
    const int ldk = a.G * DK, ldv = a.G * DV;
    // the list of key tiles: pooled rows, kept first keys, the window from the earliest row's to the latest row's position
    const int win = a.window > 0 ? a.window : 0x3fffffff, P = a.pool;
    const int lo_t = max(0, minpos - win + 1) >> 5, hi_t = maxpos >> 5, nk = min((a.keep + 31) >> 5, lo_t);
    const int nbr = P > 0 ? max(0, pr - win + 1) / P : 0, nb_wg = P > 0 ? max(0, maxpos - win + 1) / P : 0;
    const int np_t = (nb_wg + 31) >> 5, nv = np_t + nk + hi_t - lo_t + 1;
    const float *pkc = P > 0 ? a.pk + slot + (size_t)g * DK : kc, *pvc = P > 0 ? a.pv + slot + (size_t)g * DV : vc;
    auto first_key = [&](int vt) { const int w = vt - np_t; return (vt < np_t ? vt : w < nk ? w : lo_t + w - nk) << 5; };
    hy_v4f kr[CH][2];          // elements 16 c + 8 (lane / 32) .. + 7 of key lane % 32
    auto load_keys = [&](int vt) {          // (rows past the last one repeat it: masked)
        const bool pooled = vt < np_t;
        const char* p = (const char*)(pooled ? pkc : kc);          // uniform base + 32-bit byte offset
        const uint32_t off = ((uint32_t)min(first_key(vt) + r32, pooled ? nb_wg - 1 : maxpos) * (uint32_t)ldk + 8 * kh) * 4;
#pragma unroll
        for (int c = 0; c < CH; ++c) { kr[c][0] = *reinterpret_cast<const hy_v4f*>(p + off + 64 * c); kr[c][1] = *reinterpret_cast<const hy_v4f*>(p + off + 64 * c + 16); }
    };
    hy_v16f o[DVT];
#pragma unroll
    for (int i = 0; i < DVT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    float m = -INFINITY, l = 0.f;
    int vt = split * 4 + wave;
    if (vt < nv) load_keys(vt);
#pragma unroll
    for (int u = 0; u < QI; ++u) {
        const int i = tid + 256 * u, r = i / (DK / 8), c = i % (DK / 8);
        if (i >= 32 * (DK / 8)) continue;
        qs[u][0] *= a.scale; qs[u][1] *= a.scale;
#pragma unroll
        for (int pl = 0; pl < 3; ++pl) {
            hy_v4u d;
#pragma unroll
            for (int e = 0; e < 4; ++e) d[e] = hy_plane<true>(*((float*)&qs[u][e / 2] + e % 2 * 2), *((float*)&qs[u][e / 2] + e % 2 * 2 + 1));
            *reinterpret_cast<hy_v4u*>(sQ + r * QB + pl * 2 * DK + 16 * c) = d;
        }
    }
    __syncthreads();
    // product q of a step: planes PA and PB, the small ones first (those of less than 2^-16 are left out); a step's MFMAs stand between the splits of the next one's operand
    constexpr int PA[6] = {2, 1, 0, 1, 0, 0}, PB[6] = {0, 1, 2, 0, 1, 0};
    for (; vt < nv; vt += 4 * a.nsplit) {
        const bool pooled = vt < np_t;
        const int j0 = first_key(vt), last = pooled ? nb_wg - 1 : maxpos;
        VV vr[16];          // values of keys r, the second half under the softmax
        const char* vb = (const char*)(pooled ? pvc : vc);
        auto load_values = [&](int r0) {
#pragma unroll
            for (int r = r0; r < r0 + 8; ++r) vr[r] = *reinterpret_cast<const VV*>(vb + ((uint32_t)min(j0 + 8 * (r >> 2) + 4 * kh + (r & 3), last) * (uint32_t)ldv + DVT * r32) * 4);
        };
        load_values(0);
        __builtin_amdgcn_sched_barrier(0);
        hy_v16f s0;
#pragma unroll
        for (int r = 0; r < 16; ++r) s0[r] = 0.f;
        {
            hy_v4u k0[CH], ka[2][2];          // largest planes of all chunks, the smaller two of this and the next one
            hy_v8bf qv[3];
            auto cut = [&](auto uc, auto cc) {          // step u of chunk c's split
                constexpr int u = decltype(uc)::value, c = decltype(cc)::value, e = u % 4;
                const uint32_t d = hy_plane<(u < 8)>(*((float*)&kr[c][e / 2] + e % 2 * 2), *((float*)&kr[c][e / 2] + e % 2 * 2 + 1));
                if constexpr (u < 4) k0[c][e] = d; else ka[c & 1][u / 4 - 1][e] = d;
            };
            auto rq = [&](int pl, int c) { return *reinterpret_cast<const hy_v8bf*>(sQ + r32 * QB + pl * 2 * DK + 32 * c + 16 * kh); };
#pragma unroll
            for (int pl = 0; pl < 3; ++pl) qv[pl] = rq(pl, 0);
            hy_static_for<0, 12>([&](auto u) { cut(u, std::integral_constant<int, 0>{}); });
            __builtin_amdgcn_sched_barrier(0);
            hy_static_for<0, CH>([&](auto cc) {
                constexpr int c = decltype(cc)::value;
                hy_static_for<0, 5>([&](auto qc) {
                    constexpr int q = decltype(qc)::value, ka_ = q < 2 ? 0 : q < 4 ? 1 : 2, qb = q == 0 ? 2 : q < 3 ? 1 : 0;
                    hy_mma(s0, __builtin_bit_cast(hy_v8bf, ka_ ? ka[c & 1][ka_ ? ka_ - 1 : 0] : k0[c]), qv[qb]);
                    if constexpr (c + 1 < CH) {
                        if constexpr (q != 1 && q != 3) qv[qb] = rq(qb, c + 1);
                        hy_static_for<q * 12 / 5, (q + 1) * 12 / 5>([&](auto u) { cut(u, std::integral_constant<int, c + 1>{}); });
                    } else if constexpr (q == 0 || q == 2) qv[qb] = rq(0, q == 0 ? 0 : 1);
                    __builtin_amdgcn_sched_barrier(0);
                });
            });
            hy_static_for<0, CH>([&](auto cc) {          // the largest products
                constexpr int c = decltype(cc)::value;
                hy_mma(s0, __builtin_bit_cast(hy_v8bf, k0[c]), qv[c & 1 ? 1 : 2]);
                if constexpr (c + 2 < CH) qv[c & 1 ? 1 : 2] = rq(0, c + 2);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
        load_values(8);
        __builtin_amdgcn_sched_barrier(0);
        float p[16], mx = m;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int j = j0 + 8 * (r >> 2) + 4 * kh + (r & 3);
            const float s = s0[r];
            if (pooled) p[r] = j < nbr ? s : -INFINITY;
            else p[r] = (j <= pr && (pr - j < win || j < a.keep)) ? s - slope * (float)(pr - j) : -INFINITY;
            mx = fmaxf(mx, p[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const bool any = mx > -INFINITY;                         // false: this row has seen no key yet, or none whose score is a number
        const float corr = any ? expf(m - mx) : 1.f, top = any ? mx : 0.f;             // exp(-inf) = 0 the first time
        float ls = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) { p[r] = expf(p[r] - top); ls += p[r]; }
        l = l * corr + ls;
        m = mx;
        hy_v4u pp[2][3], va[2][3];          // weights of keys 0 .. 7 and 8 .. 15 of the lane, a value tile's column
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int u = 0; u < 12; ++u) pp[h][u / 4][u % 4] = u < 8 ? hy_plane<true>(p[8 * h + 2 * (u % 4)], p[8 * h + 2 * (u % 4) + 1]) : hy_plane<false>(p[8 * h + 2 * (u % 4)], p[8 * h + 2 * (u % 4) + 1]);
        auto cut = [&](auto uc, auto tc) {          // step u of item t = (half, value tile)
            constexpr int u = decltype(uc)::value, t = decltype(tc)::value, i = t % DVT, r = 8 * (t / DVT) + 2 * (u % 4);
            va[t & 1][u / 4][u % 4] = hy_plane<(u < 8)>(*((float*)&vr[r] + i), *((float*)&vr[r + 1] + i));
        };
        hy_static_for<0, 12>([&](auto u) { cut(u, std::integral_constant<int, 0>{}); });
#pragma unroll
        for (int i = 0; i < DVT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[i][r] *= corr;
        __builtin_amdgcn_sched_barrier(0);
        hy_static_for<0, 2 * DVT>([&](auto tc) {
            constexpr int t = decltype(tc)::value;
            constexpr std::integral_constant<int, t + 1 < 2 * DVT ? t + 1 : t> nx{};
            if constexpr (t == DVT) {
                if (vt + 4 * a.nsplit < nv) load_keys(vt + 4 * a.nsplit);
                __builtin_amdgcn_sched_barrier(0);
            }
            hy_static_for<0, 6>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                hy_mma(o[t % DVT], __builtin_bit_cast(hy_v8bf, va[t & 1][PA[q]]), __builtin_bit_cast(hy_v8bf, pp[t / DVT][PB[q]]));
                if constexpr (t + 1 < 2 * DVT) hy_static_for<2 * q, 2 * q + 2>([&](auto u) { cut(u, nx); });
                __builtin_amdgcn_sched_barrier(0);
            });
        });
    }
    // the gate's values travel while the wavefronts join
    constexpr int GI = 32 * (DV / 4) / 256;
    float4 gz[GI];
    const bool gated = a.out && a.gate && a.gate_mode != 2;
    if (gated)
#pragma unroll
        for (int u = 0; u < GI; ++u) {
            const int i = tid + 256 * u, q = min(row0 + i / (DV / 4), rows - 1), c = i % (DV / 4);
            gz[u] = *reinterpret_cast<const float4*>(a.gate + (size_t)(q / hpg) * a.ldg + (g * hpg + q % hpg) * DV + 4 * c);
        }
    // join the wavefronts: every lane scales by e^(m - M), the wavefronts add up in LDS one after the other
    l += __shfl_xor(l, 32, 64);
    const auto tile = [&](int t, int& j, int& last, bool& pooled) { pooled = t < np_t; j = first_key(t); last = pooled ? nb_wg - 1 : maxpos; };
    if (__builtin_expect(l != l, 0)) hy_softmax_again<DK>(m, l, a, qrow, slope, pr, nbr, win, kc, pkc, split * 4 + wave, 4 * a.nsplit, nv, tile);
    if (kh == 0) { sml[wave][0][r32] = m; sml[wave][1][r32] = l; }
    __syncthreads();
    const float M = fmaxf(fmaxf(sml[0][0][r32], sml[1][0][r32]), fmaxf(sml[2][0][r32], sml[3][0][r32]));
    const float sc = m > -INFINITY ? expf(m - M) : 0.f;
    if (__builtin_expect(__any(hy_attn_nan<DVT>(o) && pr >= 0 && l == l), 0))
        hy_attn_again<DK, DVT>(o, a, qrow, a.scale, 1.f, m, slope, pr, nbr, win, kc, vc, pkc, pvc, 0, kh, split * 4 + wave, 4 * a.nsplit, nv, tile);
    for (int w = 0; w < 4; ++w) {
        if (wave == w) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                VV* d = reinterpret_cast<VV*>(sO + r32 * OS + DVT * (8 * (r >> 2) + 4 * kh + (r & 3)));
                VV v;
                if (w > 0) v = *d;
                v.x = (w > 0 ? v.x : 0.f) + sc * o[0][r];
                v.y = (w > 0 ? v.y : 0.f) + sc * o[1][r];
                if constexpr (DVT == 4) { v.z = (w > 0 ? v.z : 0.f) + sc * o[2][r]; v.w = (w > 0 ? v.w : 0.f) + sc * o[3][r]; }
                *d = v;
            }
        }
        __syncthreads();
    }
    if (a.out) {          // one split: denominators, gate and the operand's type here (512 tokens x 32 heads of 128: a launch of 10 us, and 16 MB of parts written and read, less)
        __shared__ float sF[32][2];
        if (tid < 32) {
            float L = 0.f;
#pragma unroll
            for (int w = 0; w < 4; ++w) if (sml[w][0][r32] > -INFINITY) L += expf(sml[w][0][r32] - M) * sml[w][1][r32];
            const float z = a.sink_w ? a.sink_w[hr] : 0.f, top = a.sink ? fmaxf(M, z) : M, e = M > -INFINITY ? expf(M - top) : 0.f;
            sF[tid][0] = e;
            sF[tid][1] = e * L + (a.sink ? expf(z - top) : 0.f);
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < GI; ++u) {
            const int i = tid + 256 * u, r = i / (DV / 4), c = i % (DV / 4), q = row0 + r;
            if (q >= rows) continue;
            const int t = q / hpg, h = g * hpg + q % hpg;
            const float4 v4 = *reinterpret_cast<const float4*>(sO + r * OS + 4 * c);
            const float e = sF[r][0], den = sF[r][1];
            float v[4] = {v4.x * e / den, v4.y * e / den, v4.z * e / den, v4.w * e / den};
            if (a.gate && a.gate_mode == 2) {
                const float s = hy_sigmoid(a.gate[(size_t)t * a.ldg + h]);
#pragma unroll
                for (int k = 0; k < 4; ++k) v[k] *= s;
            } else if (a.gate) {
                const float4 z = gz[u];
                v[0] *= hy_sigmoid(z.x); v[1] *= hy_sigmoid(z.y); v[2] *= hy_sigmoid(z.z); v[3] *= hy_sigmoid(z.w);
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) v[k] *= a.out_mul;
            const size_t o = (size_t)t * a.ldo + h * DV + 4 * c;
            if (a.out_f32) hy_stv<4>((float*)a.out + o, v); else hy_stv<4>((bf16_t*)a.out + o, v);
        }
        return;
    }
    for (int i = tid; i < 32 * (DV / 4); i += 256) {
        const int r = i / (DV / 4), c = i % (DV / 4), q = row0 + r;
        if (q >= rows) continue;
        const size_t ob = ((size_t)(q / hpg) * a.H + g * hpg + q % hpg) * a.nsplit + split;
        *reinterpret_cast<float4*>(a.part_acc + ob * DV + 4 * c) = *reinterpret_cast<const float4*>(sO + r * OS + 4 * c);
    }
    if (tid < 32 && pr >= 0) {
        float L = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) if (sml[w][0][r32] > -INFINITY) L += expf(sml[w][0][r32] - M) * sml[w][1][r32];
        const size_t ob = ((size_t)(rho / hpg) * a.H + hr) * a.nsplit + split;
        a.part_ml[2 * ob] = M;
        a.part_ml[2 * ob + 1] = L;
    }
}

// A few tokens (decode): workgroup = (32 rows of a key / value head, key split) with one tile of 32 keys at a time for all its wavefronts (four; eight for long rows): each multiplies
// its share of the entries (queries and keys straight from memory), the shares of the scores meet in LDS, every wavefront makes its share of the
// softmax and the weighted sum of its own value columns.  Same layouts as above; rows that are not there cost MFMAs nobody waits for.  Latent attention's
// cached rows (keys = values) come as kc = vc.  A tile is one round trip to memory and (DK + DV) / 2 MFMAs over the wavefronts, and the tiles of a
// token up to 32 x HY_MAX_SPLITS positions run side by side, where hy_attn_kernel walked tiles of 64 keys with four rows per wavefront (us):
// 32 heads on 512-entry latents 29 - 33 -> 12.4, 8 x 4 heads of 64 7.3 -> 5.8, of 128 behind 2041 positions 13.5 -> 8.2 us.
template <int DK, int DV, int NW = 4>          // NW wavefronts
static __global__ __launch_bounds__(64 * NW, 1) void hy_attn_few_kernel(HyAttnArgs a) {
    constexpr int RQ = DK / NW, KC = RQ / 8, CW = DV >= 32 * NW ? DV / NW : 32, NE = 16 / NW, DVT = CW / 32;
    __shared__ float sS[NW][16][64], sP[16][64], sM[NW][64];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), r32 = lane & 31, kh = lane >> 5;
    const int g = blockIdx.x % a.G, rb = blockIdx.x / a.G, split = blockIdx.z, hpg = a.H / a.G, rows = a.n * hpg, row0 = rb * 32, pos0 = a.dyn[0];
    const int minpos = pos0 + row0 / hpg, maxpos = pos0 + min(rows - 1, row0 + 31) / hpg;
    const int rho = row0 + r32, pr = rho < rows ? pos0 + rho / hpg : -1, hr = g * hpg + (rho < rows ? rho % hpg : 0);
    const float slope = a.slope_log2 != 0.f ? exp2f(-a.slope_log2 * (float)(hr + 1) / (float)a.H) : 0.f;
    const size_t slot = (size_t)a.dyn[1] * a.slot_stride;
    const int ldk = a.G * DK, ldv = a.G * DV, col0 = wave * CW;
    const bool live = col0 < DV;          // (64 value columns are two wavefronts' work)
    const float *kc = a.kc + slot + (size_t)g * DK, *vc = a.vc + slot + (size_t)g * DV;
    const int win = a.window > 0 ? a.window : 0x3fffffff, P = a.pool;
    const int lo_t = max(0, minpos - win + 1) >> 5, hi_t = maxpos >> 5, nk = min((a.keep + 31) >> 5, lo_t);
    const int nbr = P > 0 ? max(0, pr - win + 1) / P : 0, nb_wg = P > 0 ? max(0, maxpos - win + 1) / P : 0;
    const int np_t = (nb_wg + 31) >> 5, nv = np_t + nk + hi_t - lo_t + 1;
    const float *pkc = P > 0 ? a.pk + slot + (size_t)g * DK : kc, *pvc = P > 0 ? a.pv + slot + (size_t)g * DV : vc;
    hy_acc4 qr[KC];
    {
        const int q = min(rho, rows - 1);
        const float* p = a.q + (size_t)(q / hpg) * a.ldq + (size_t)(g * hpg + q % hpg) * DK + wave * RQ + 4 * kh;
#pragma unroll
        for (int c = 0; c < KC; ++c) qr[c] = *reinterpret_cast<const hy_acc4*>(p + 8 * c);
    }
    hy_v16f o[DVT];
#pragma unroll
    for (int i = 0; i < DVT; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
    float m = -INFINITY, l = 0.f;
    for (int vt = split; vt < nv; vt += a.nsplit) {          // (uniform over the workgroup)
        const bool pooled = vt < np_t;
        const int w_ = vt - np_t, j0 = (pooled ? vt : w_ < nk ? w_ : lo_t + w_ - nk) << 5, last = pooled ? nb_wg - 1 : maxpos;
        hy_acc4 kr[KC];
        const float* kp = (pooled ? pkc : kc) + (size_t)min(j0 + r32, last) * ldk + wave * RQ + 4 * kh;
#pragma unroll
        for (int c = 0; c < KC; ++c) kr[c] = *reinterpret_cast<const hy_acc4*>(kp + 8 * c);
        float vr[16][DVT];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float* vp = (pooled ? pvc : vc) + (size_t)min(j0 + 8 * (r >> 2) + 4 * kh + (r & 3), last) * ldv + (live ? col0 : 0) + DVT * r32;
#pragma unroll
            for (int i = 0; i < DVT; ++i) vr[r][i] = vp[i];
        }
        hy_v16f s0, s1;
#pragma unroll
        for (int r = 0; r < 16; ++r) s0[r] = s1[r] = 0.f;
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[c][0], qr[c][0], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[c][1], qr[c][1], s1, 0, 0, 0);
            s0 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[c][2], qr[c][2], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f32_32x32x2f32(kr[c][3], qr[c][3], s1, 0, 0, 0);
        }
        if (vt != split) __syncthreads();
#pragma unroll
        for (int r = 0; r < 16; ++r) sS[wave][r][lane] = s0[r] + s1[r];
        __syncthreads();
        // scores NE wave .. of every lane: a share of the softmax per wavefront (all sixteen in each would be four or eight times the exponentials)
        float p[NE], mx = -INFINITY;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            const int r = NE * wave + e, j = j0 + 8 * (r >> 2) + 4 * kh + (r & 3);
            float s = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w += 2) s += sS[w][r][lane] + sS[w + 1][r][lane];
            s *= a.scale;
            if (pooled) p[e] = j < nbr ? s : -INFINITY;
            else p[e] = (j <= pr && (pr - j < win || j < a.keep)) ? s - slope * (float)(pr - j) : -INFINITY;
            mx = fmaxf(mx, p[e]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        sM[wave][lane] = mx;
        __syncthreads();
        mx = m;
#pragma unroll
        for (int w = 0; w < NW; ++w) mx = fmaxf(mx, sM[w][lane]);
        const bool any = mx > -INFINITY;                         // false: this row has seen no key yet
        const float corr = any ? expf(m - mx) : 1.f;
        float ls = 0.f;
#pragma unroll
        for (int e = 0; e < NE; ++e) {
            p[e] = any ? expf(p[e] - mx) : 0.f;
            ls += p[e];
            sP[NE * wave + e][lane] = p[e];
        }
        l = l * corr + ls;                                       // (this wavefront's share)
        m = mx;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < DVT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[i][r] *= corr;
        if (live) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float pr_ = sP[r][lane];
#pragma unroll
                for (int i = 0; i < DVT; ++i) o[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(vr[r][i], pr_, o[i], 0, 0, 0);
            }
        }
    }
    l += __shfl_xor(l, 32, 64);
    __syncthreads();
    sM[wave][lane] = l;
    __syncthreads();
    l = 0.f;
#pragma unroll
    for (int w = 0; w < NW; ++w) l += sM[w][lane];
    if (pr < 0) return;
    const size_t ob = ((size_t)(rho / hpg) * a.H + hr) * a.nsplit + split;
    if (wave == 0 && kh == 0) { a.part_ml[2 * ob] = m; a.part_ml[2 * ob + 1] = l; }
    if (!live) return;
    float* dst = a.part_acc + ob * DV + col0;
    auto store = [&](const hy_v16f* v) {
#pragma unroll
        for (int r = 0; r < 16; ++r)
#pragma unroll
            for (int i = 0; i < DVT; ++i) dst[DVT * (8 * (r >> 2) + 4 * kh + (r & 3)) + i] = v[i][r];
    };
    const bool nan = hy_attn_nan<DVT>(o);
    if (__builtin_expect(!__any(nan), 1)) store(o);          // (the rare way out of line: 256 entries 9.2 -> 8.6 us, 64 6.1 -> 6.0)
    else if (nan) {
        hy_v16f again[DVT];
        hy_attn_again<DK, DVT>(again, a, a.q + (size_t)(rho / hpg) * a.ldq + (size_t)hr * DK, 1.f, a.scale, m, slope, pr, nbr, win, kc, vc, pkc, pvc, col0, kh, split, a.nsplit, nv,
                               [&](int t, int& j, int& last, bool& pooled) { const int w = t - np_t; pooled = t < np_t; j = (pooled ? t : w < nk ? w : lo_t + w - nk) << 5; last = pooled ? nb_wg - 1 : maxpos; });
        store(again);
    } else store(o);
}
