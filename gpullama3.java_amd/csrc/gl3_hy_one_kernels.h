// gl3_hy_one_kernels.h — the mixers of the layer-list family for ONE token behind few positions, each in one launch.
//
// A token's small launches cost 2 us of boundary and one or two round trips to memory each, whatever they compute; behind a few hundred positions the
// work of all of them fits one workgroup per query head: cache row, queries, scores, softmax, weighted sum, gate.  All float32; longer caches, windows in use and other forms stay with the kernels of many workgroups (gl3_hy_kernels.h, gl3_hy_attn_mfma.h).
#pragma once
#include "gl3_hy_kernels.h"

template <int N> __device__ __forceinline__ float hy_row_ror(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 + N, 0xf, 0xf, false));
}
// over the 16 lanes of a row (rotations by 8, 4, 2, 1: every lane gets the same sum)
__device__ __forceinline__ float hy_row_sum(float v) { v += hy_row_ror<8>(v); v += hy_row_ror<4>(v); v += hy_row_ror<2>(v); return v + hy_row_ror<1>(v); }
__device__ __forceinline__ float hy_row_max(float v) {
    v = fmaxf(v, hy_row_ror<8>(v)); v = fmaxf(v, hy_row_ror<4>(v)); v = fmaxf(v, hy_row_ror<2>(v));
    return fmaxf(v, hy_row_ror<1>(v));
}
__device__ __forceinline__ float hy_dot4(const float4& a, const float4& b, float s) { return fmaf(a.w, b.w, fmaf(a.z, b.z, fmaf(a.y, b.y, fmaf(a.x, b.x, s)))); }
__device__ __forceinline__ void hy_axpy4(float4& o, float p, const float4& v) { o.x = fmaf(p, v.x, o.x); o.y = fmaf(p, v.y, o.y); o.z = fmaf(p, v.z, o.z); o.w = fmaf(p, v.w, o.w); }
__device__ __forceinline__ void hy_mul4(float4& o, float s) { o.x *= s; o.y *= s; o.z *= s; o.w *= s; }

// p[0] + p[ld] + .. + p[(n - 1) ld], eight chains side by side that meet in pairs
__device__ __forceinline__ float hy_sum_rows(const float* p, int ld, int n) {
    float s[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) s[u] = 0.f;
    for (int k = 0; k < n; k += 8)
#pragma unroll
        for (int u = 0; u < 8; ++u)
            if (k + u < n) s[u] += p[(k + u) * ld];
    return ((s[0] + s[1]) + (s[2] + s[3])) + ((s[4] + s[5]) + (s[6] + s[7]));
}
// How the sums of sixteen wavefronts weigh in the result: lane w of 16 brings maximum and denominator of wavefront w and gets e^(m_w - M) / den, with the
// sink's unit in the denominator.
__device__ __forceinline__ float hy_join_weight(float mw, float lw, int sink, float z) {
    float M = hy_row_max(mw);
    if (sink) M = fmaxf(M, z);
    const float e = mw > -INFINITY ? expf(mw - M) : 0.f;
    float den = hy_row_sum(e * lw);
    if (sink) den += expf(z - M);
    return e / den;
}

// ---- attention ------------------------------------------------------------------------------------------------------------------------
// Workgroup = query head, sixteen wavefronts.  Three of them finish the query, the key and the value (bias, norm, weight, turn: as
// hy_attn_prep_kernel; the heads of a group make the same key and value) in LDS; then every wavefront walks its strips of 4 U cached keys, sixteen lanes per key
// (NI pieces of 16 bytes each, DPP rotations add them up), keys and values on their way together, a running maximum and sums per sixteen lanes; the
// token's own key joins from LDS.  One meeting in LDS, then the gated result itself.  Whole steps of one layer, us, with and without (three launches, four with a norm over the whole
// projections): 32 heads of 64 behind 5 positions 92 / 99, 500 88 / 94, 1000 92 / 93, 2000 101 / 96; of 128 behind 5 154 / 161, 500 163 / 164, 1000 169 / 162: the line
// lies at 384 KB of keys and values a head (HY_ATTN_ONE), with few heads as with many (us a layer, one launch / many, just behind it: 2 heads of 64 1000 positions 25.3 / 25.7, 64 heads 34.1 / 33.8; 2 heads of
// 128 500 26.0 / 27.6, 64 heads 45.8 / 45.1; 4 heads of 256 250 28.8 / 33.0).  Splitting longer caches over workgroups behind it gains less than the runs differ.
// Bound: latency (three dependent round trips), further back one CU's reads of the head's cache; the heads of a group read it side by side, which costs
// an idle chip nothing, while four heads in a workgroup would queue their arithmetic.
struct HyAttnOne {
    const float* proj; int q_off, k_off, v_off;
    int H, G, D, V, unit_norm;
    float eps;
    float* kc; float* vc; size_t slot_stride; const int* dyn;
    HyRot rot;
    const float *bias, *qn, *kn;
    int v_from_k;
    float scale, slope_log2;
    int sink; const float* sink_w;
    const float* gate; int gate_mode;
    const float* v_freq; float out_mul;
};
constexpr long HY_ATTN_ONE = 384 * 1024;
template <typename TO, int NI>          // head sizes up to 64 NI
__device__ __forceinline__ void hy_attn_one(const HyAttnOne& a, TO* __restrict__ out, const int h) {
    constexpr int U = 4 / NI, NW = 16, MD = 64 * NI;
    __shared__ __attribute__((aligned(16))) float sQ[MD], sK[MD], sV[MD], sO[NW][MD];
    __shared__ float sML[NW][2], sW[NW], sR[2 * NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, grp = lane >> 4;
    const int g = h / (a.H / a.G), D = a.D, V = a.V, pos = a.dyn[0];
    const size_t slot = (size_t)a.dyn[1] * a.slot_stride;
    float *kc = a.kc + slot + (size_t)g * D, *vc = a.vc + slot + (size_t)g * V;
    const int ldk = a.G * D, ldv = a.G * V;
    // the wavefront's first strip travels from the start
    float4 kr[U][NI], vr[U][NI];
    int base = wave * 4 * U;
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = min(base + 4 * u + grp, pos - 1);
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                const int c = 4 * (l16 + 16 * i);
                kr[u][i] = c < D ? *reinterpret_cast<const float4*>(kc + (size_t)j * ldk + c) : make_float4(0.f, 0.f, 0.f, 0.f);
                vr[u][i] = c < V ? *reinterpret_cast<const float4*>(vc + (size_t)j * ldv + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    };
    if (base < pos) load();
    float rq = 1.f, rk = 1.f;
    if (a.unit_norm == 2) {          // one norm over the whole q and k projections
        float sq = 0.f, sk = 0.f;
        for (int i = tid; i < a.H * D; i += 1024) { const float v = a.proj[a.q_off + i] + (a.bias ? a.bias[a.q_off + i] : 0.f); sq += v * v; }
        for (int i = tid; i < a.G * D; i += 1024) { const float v = a.proj[a.k_off + i] + (a.bias ? a.bias[a.k_off + i] : 0.f); sk += v * v; }
        hy_block_sum2<1024>(sq, sk, sR);
        rq = 1.f / sqrtf(sq / (float)(a.H * D) + a.eps);
        rk = 1.f / sqrtf(sk / (float)(a.G * D) + a.eps);
    }
    if (wave < 3) {
        const bool isq = wave == 0, isk = wave == 1;
        const int col = isq ? a.q_off + h * D : isk || a.v_from_k ? a.k_off + g * D : a.v_off + g * V, len = isq || isk ? D : V;
        const float *src = a.proj + col, *bias = a.bias ? a.bias + col : nullptr;
        float* dst = isq ? sQ : isk ? sK : sV;
        const bool norm = isq || isk ? a.unit_norm == 1 || a.unit_norm == 3 : a.rot.v_norm && !a.v_from_k;
        float r = isq ? rq : isk ? rk : 1.f;
        const float* w = !(isq || isk) ? nullptr : a.unit_norm == 2 ? (isq ? a.qn + h * D : a.kn + g * D) : a.unit_norm == 3 ? (isq ? a.qn : a.kn) : nullptr;
        if (norm) {
            float ss = 0.f;
            for (int d = lane; d < len; d += 64) { const float v = src[d] + (bias ? bias[d] : 0.f); ss += v * v; }
            ss = hy_wave_sum(ss);
            r = 1.f / sqrtf(ss / (float)len + a.eps);
        }
        if (isq || isk) hy_turn_store(dst, src, D, a.rot.qk_dims, a.rot.qk_freq, pos, r, lane, a.rot.interleaved, bias, w);
        else hy_turn_store(dst, src, V, a.rot.v_freq && !a.v_from_k ? V : 0, a.rot.v_freq, pos, r, lane, 0, bias);
    }
    __syncthreads();
    if (h % (a.H / a.G) == 0) {          // the cache's new rows
        if (tid < D) kc[(size_t)pos * ldk + tid] = sK[tid];
        if (tid < V) vc[(size_t)pos * ldv + tid] = sV[tid];
    }
    const float slope = a.slope_log2 != 0.f ? exp2f(-a.slope_log2 * (float)(h + 1) / (float)a.H) : 0.f;
    float4 q[NI], o[NI];
    float m = -INFINITY, l = 0.f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int c = 4 * (l16 + 16 * i);
        q[i] = c < D ? *reinterpret_cast<const float4*>(sQ + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        o[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    // UU keys of every sixteen lanes join the running sums; dist[u] < 0: there is no such key
    auto join = [&](auto uu, const float4 (*k)[NI], const float4 (*v)[NI], const int* dist) {
        constexpr int UU = decltype(uu)::value;
        float s[UU], mx = m;
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            float t = 0.f;
#pragma unroll
            for (int i = 0; i < NI; ++i) t = hy_dot4(k[u][i], q[i], t);
            t = hy_row_sum(t) * a.scale;
            s[u] = dist[u] >= 0 ? t - slope * (float)dist[u] : -INFINITY;
            mx = fmaxf(mx, s[u]);
        }
        const bool any = mx > -INFINITY;
        const float corr = any ? expf(m - mx) : 1.f;
        l *= corr;
        m = mx;
#pragma unroll
        for (int i = 0; i < NI; ++i) hy_mul4(o[i], corr);
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            const float p = dist[u] >= 0 && (any || s[u] != s[u]) ? expf(s[u] - mx) : 0.f;          // (fmaxf passes over a score that is not a number: a key alone must reach l all the same)
            l += p;
            if (dist[u] >= 0)
#pragma unroll
                for (int i = 0; i < NI; ++i) hy_axpy4(o[i], p, v[u][i]);
        }
    };
    while (base < pos) {
        int dist[U];
#pragma unroll
        for (int u = 0; u < U; ++u) { const int j = base + 4 * u + grp; dist[u] = j < pos ? pos - j : -1; }
        join(std::integral_constant<int, U>{}, kr, vr, dist);
        base += NW * 4 * U;
        if (base < pos) load();
    }
    if (wave == NW - 1) {          // the token's own key
        float4 k1[1][NI], v1[1][NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int c = 4 * (l16 + 16 * i);
            k1[0][i] = c < D ? *reinterpret_cast<const float4*>(sK + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            v1[0][i] = c < V ? *reinterpret_cast<const float4*>(sV + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        const int dist[1] = {grp == 0 ? 0 : -1};
        join(std::integral_constant<int, 1>{}, k1, v1, dist);
    }
    // the four keys side by side, then the wavefronts
    float M = fmaxf(m, __shfl_xor(m, 16, 64));
    M = fmaxf(M, __shfl_xor(M, 32, 64));
    const float sc = m > -INFINITY ? expf(m - M) : 0.f;
    l *= sc;
    l += __shfl_xor(l, 16, 64); l += __shfl_xor(l, 32, 64);
    if (lane == 0) { sML[wave][0] = M; sML[wave][1] = l; }
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        float4 x = o[i];
        hy_mul4(x, sc);
        x.x += __shfl_xor(x.x, 16, 64); x.y += __shfl_xor(x.y, 16, 64); x.z += __shfl_xor(x.z, 16, 64); x.w += __shfl_xor(x.w, 16, 64);
        x.x += __shfl_xor(x.x, 32, 64); x.y += __shfl_xor(x.y, 32, 64); x.z += __shfl_xor(x.z, 32, 64); x.w += __shfl_xor(x.w, 32, 64);
        if (grp == 0) *reinterpret_cast<float4*>(&sO[wave][4 * (l16 + 16 * i)]) = x;
    }
    __syncthreads();
    if (tid < NW) sW[tid] = hy_join_weight(sML[tid][0], sML[tid][1], a.sink, a.sink_w ? a.sink_w[h] : 0.f);
    __syncthreads();
    auto column = [&](int c) {
        float v = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) v = fmaf(sW[w], sO[w][c], v);
        return v;
    };
    auto put = [&](int c, float v) {
        if (a.gate) v *= hy_sigmoid(a.gate[a.gate_mode == 2 ? h : h * V + c]);
        hy_st(out + h * V + c, v * a.out_mul);
    };
    if (a.v_freq) {          // turned values: a thread has both entries of a pair
        const int half = V >> 1;
        if (tid < half) {
            float sn, cs;
            sincosf((float)pos * a.v_freq[tid], &sn, &cs);
            const float u = column(tid), v = column(tid + half);
            put(tid, u * cs + v * sn);
            put(tid + half, v * cs - u * sn);
        }
    } else if (tid < V) put(tid, column(tid));
}

template <typename TO, int NI>
static __global__ __launch_bounds__(1024) void hy_attn_one_kernel(HyAttnOne a, TO* __restrict__ out) { hy_attn_one<TO, NI>(a, out, blockIdx.x); }

// ---- latent attention -------------------------------------------------------------------------------------------------------------------
// Workgroup = one head, sixteen wavefronts: the token's cached row (norm, weight, turned part), the query carried into the latent's space (the head's rows of the
// key expansion read once, sixteen bytes a lane, their first pieces on the way before anything else), the scores and the weighted sum over the cached rows
// (a wavefront takes four rows at a time, 64 lanes to a row), the join in LDS and the value expansion with its gate.
// It replaces five launches: cache row 3.6 us, query 2.9, attention 12.6 (7.2 for 256 entries), join 4.6 - 8.6, expansion 4.9 - 6.0.
// Bound: one CU's share of the expansions (2 x 131 KB a head of 64 on 512-entry latents) and, further back, the cached rows, which every head reads.  Whole steps, us,
// with and without: 512 entries, three layers, behind 5 positions 171 / 188, 250 178 / 191, 500 193 / 200; 256 entries, two layers, 5 205 / 217, 180 208 / 221, 400 215 / 223:
// the line is hy_latent_one_line's, at most HY_LATENT_ONE_POS.
struct HyLatentOne {
    const float* q; int D, P;                                // the head's query: D + P entries, the last P turn by the position
    const float* src; int R0; const float* lat_norm;         // the token's raw row (R0 + P entries); null: the cache holds the token's row already
    float eps;
    float* cc; size_t slot_stride; const int* dyn;
    const double* freq; float mscale;
    const float *wk, *wvT;                                   // [H][D + P][R], [H][R][V]
    int R, V;
    float scale; int sink; const float* sink_w;
    const float* gate; int gate_mode;
};
constexpr int HY_LATENT_ONE = 512, HY_LATENT_ONE_POS = 640;
template <typename TO>
static __global__ __launch_bounds__(1024) void hy_latent_one_kernel(HyLatentOne a, TO* __restrict__ out) {
    constexpr int NW = 16, U = 4;
    __shared__ __attribute__((aligned(16))) float sC[HY_LATENT_ONE], sQ[1024], sA[HY_LATENT_ONE], sO[NW * HY_LATENT_ONE];
    __shared__ float sML[NW][2], sW[NW], sR[NW];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int h = blockIdx.x, R = a.R, V = a.V, De = a.D + a.P, pos = a.dyn[0], half = a.P >> 1;
    float* cc = a.cc + (size_t)a.dyn[1] * a.slot_stride;
    // key expansion: column piece kc4 of the rows kg, kg + nkg ..
    const int rc = R >> 2, nkg = 1024 / rc, kg = tid / rc, kc4 = tid - kg * rc;
    const float* wk = a.wk + (size_t)h * De * R + 4 * kc4;
    float4 w8[8];
    auto load_w = [&](const float* w, int ld, int g0, int step, int n) {
#pragma unroll
        for (int u = 0; u < 8; ++u) w8[u] = *reinterpret_cast<const float4*>(w + (size_t)min(g0 + u * step, n - 1) * ld);
    };
    if (kg < nkg) load_w(wk, R, kg, nkg, De);
    // the wavefront's first cached rows
    const int last = a.src ? pos : pos + 1;                  // rows the cache holds
    float4 kr[U][2];
    int base = wave * U;
    auto load = [&]() {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int c = 4 * (lane + 64 * i);
                kr[u][i] = c < R ? *reinterpret_cast<const float4*>(cc + (size_t)min(base + u, last - 1) * R + c) : make_float4(0.f, 0.f, 0.f, 0.f);
            }
    };
    if (base < last) load();
    for (int d = tid; d < De; d += 1024) {
        const float* q = a.q + (size_t)h * De;
        const int i = d - a.D;
        float v = q[d];
        if (i >= 0) {
            const int j = i < half ? i : i - half;
            const float w = q[a.D + (i < half ? i + half : j)];
            float sn, cs;
            hy_sincos_pos(pos, a.freq[j], a.mscale, &sn, &cs);
            v = i < half ? v * cs - w * sn : v * cs + w * sn;
        }
        sQ[d] = v;
    }
    if (a.src) {
        float x = tid < a.R0 ? a.src[tid] : 0.f;             // (R0 <= 512)
        const float ss = hy_block_sum<1024>(x * x, sR), s = 1.f / sqrtf(ss / (float)a.R0 + a.eps);
        if (tid < a.R0) x = x * s * a.lat_norm[tid];
        else if (tid < R) {
            const int i = tid - a.R0, j = i < half ? i : i - half;
            const float u = a.src[tid], w = a.src[a.R0 + (i < half ? i + half : j)];
            float sn, cs;
            hy_sincos_pos(pos, a.freq[j], a.mscale, &sn, &cs);
            x = i < half ? u * cs - w * sn : u * cs + w * sn;
        }
        if (tid < R) {
            sC[tid] = x;
            if (h == 0) cc[(size_t)pos * R + tid] = x;
        }
    }
    __syncthreads();
    if (kg < nkg) {
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int d0 = kg; d0 < De; d0 += 8 * nkg) {
            if (d0 > kg) load_w(wk, R, d0, nkg, De);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (d0 + u * nkg < De) hy_axpy4(s, sQ[d0 + u * nkg], w8[u]);
        }
        *reinterpret_cast<float4*>(sO + kg * R + 4 * kc4) = s;
    }
    __syncthreads();
    for (int c = tid; c < R; c += 1024) {
        sA[c] = hy_sum_rows(sO + c, R, nkg);
    }
    __syncthreads();
    float4 q[2], o[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = 4 * (lane + 64 * i);
        q[i] = c < R ? *reinterpret_cast<const float4*>(sA + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        o[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    float m = -INFINITY, l = 0.f;
    auto join = [&](auto uu, const float4 (*k)[2], int n) {          // n of the UU rows are there
        constexpr int UU = decltype(uu)::value;
        float s[UU], mx = m;
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            float t = hy_row_sum(hy_dot4(k[u][1], q[1], hy_dot4(k[u][0], q[0], 0.f)));
            t += __shfl_xor(t, 16, 64); t += __shfl_xor(t, 32, 64);
            s[u] = u < n ? t * a.scale : -INFINITY;
            mx = fmaxf(mx, s[u]);
        }
        const bool any = mx > -INFINITY;
        const float corr = any ? expf(m - mx) : 1.f;
        l *= corr;
        m = mx;
        hy_mul4(o[0], corr); hy_mul4(o[1], corr);
#pragma unroll
        for (int u = 0; u < UU; ++u) {
            if (u >= n) break;
            const float p = any || s[u] != s[u] ? expf(s[u] - mx) : 0.f;
            l += p;
            hy_axpy4(o[0], p, k[u][0]); hy_axpy4(o[1], p, k[u][1]);
        }
    };
    while (base < last) {
        join(std::integral_constant<int, U>{}, kr, min(U, last - base));
        base += NW * U;
        if (base < last) load();
    }
    if (a.src && wave == NW - 1) {                           // the token's own row
        float4 k1[1][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int c = 4 * (lane + 64 * i);
            k1[0][i] = c < R ? *reinterpret_cast<const float4*>(sC + c) : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        join(std::integral_constant<int, 1>{}, k1, 1);
    }
    // value expansion: column piece vc4 of the entries vg, vg + nvg ..; the first pieces travel under the join
    const int vcn = V >> 2, nvg = 1024 / vcn, vg = tid / vcn, vc4 = tid - vg * vcn;
    const float* wv = a.wvT + (size_t)h * R * V + 4 * vc4;
    if (vg < nvg) load_w(wv, V, vg, nvg, R);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int c = 4 * (lane + 64 * i);
        if (c < R) *reinterpret_cast<float4*>(sO + wave * R + c) = o[i];
    }
    if (lane == 0) { sML[wave][0] = m; sML[wave][1] = l; }
    __syncthreads();
    if (tid < NW) sW[tid] = hy_join_weight(sML[tid][0], sML[tid][1], a.sink, a.sink_w ? a.sink_w[h] : 0.f);
    __syncthreads();
    for (int c = tid; c < R; c += 1024) {
        float s = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) s = fmaf(sW[w], sO[w * R + c], s);
        sA[c] = s;
    }
    __syncthreads();
    if (vg < nvg) {
        float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int r0 = vg; r0 < R; r0 += 8 * nvg) {
            if (r0 > vg) load_w(wv, V, r0, nvg, R);
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (r0 + u * nvg < R) hy_axpy4(s, sA[r0 + u * nvg], w8[u]);
        }
        *reinterpret_cast<float4*>(sO + vg * V + 4 * vc4) = s;          // (nvg V <= 4096 floats)
    }
    __syncthreads();
    for (int c = tid; c < V; c += 1024) {
        float s = hy_sum_rows(sO + c, V, nvg);
        if (a.gate) s *= hy_sigmoid(a.gate[a.gate_mode == 2 ? h : h * V + c]);
        hy_st(out + h * V + c, s);
    }
}

// ---- matrix memories ----------------------------------------------------------------------------------------------------------------------
// Workgroup = one head: the gates of a memory with exponential gating (hy_mem_gates_kernel's arithmetic for one token), the step of the state (hy_scan_one_kernel's:
// every element read and written once, QN rows of 64 CB NB columns a wavefront on their way at once) and what leaves the
// head (hy_mem_out_kernel's norm and gate).  It replaces two launches, three with exponential gates.  Bound: one CU reads and writes the head's state,
// so it is taken while that is small (HY_SCAN_OUT); one norm over the heads side by side needs them all and stays apart.  Whole steps, us, with and without: retention of 16 x
// 64 x 128 and mLSTM 8 x 128 x 257 144 / 149; retention 16 x 128 x 256 equal; with mLSTM 8 x 256 x 513 too 313 / 291.
struct HyScanOut {
    HyScanArgs s;                                            // mode 1 (exponential gates) and 2 (fixed decay), ga / gb / y unused
    int i_off, f_off; const float* gbias; float cap; float* m;          // mode 1: raw gates in the projection row, running maximum of the slot
    const float* gate; int gate_act;                         // gate null: none; 1 sigmoid, else silu
    const float* w; int w_stride; float eps, out_mul;
};
constexpr int HY_SCAN_OUT = 40 * 1024;                       // state elements a head
constexpr int HY_SCAN_OUT_P = 1024;                          // value columns a head
template <typename TO, int QN>
__device__ __forceinline__ void hy_scan_out(const HyScanOut& b, TO* __restrict__ out, const int head) {
    constexpr int CB = 16 / QN, NB = QN == 4 ? 1 : 3, NW = 16;          // NB times 64 CB columns at once
    __shared__ float sK[16 * QN], sQ[16 * QN], sY[NW][64 * CB * NB], sP[HY_SCAN_OUT_P], red[NW];
    const HyScanArgs& a = b.s;
    const int N = a.N, P = a.P, V = P - (a.ones_col ? 1 : 0), tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), pos = a.dyn[0];
    const bool fresh = pos == 0;
    const float *kb = a.ksrc + a.k_off + (size_t)head * a.k_hstride, *qb = a.qsrc + a.q_off + (size_t)head * a.q_hstride;
    float* S = a.state + (size_t)a.dyn[1] * a.slot_stride + (size_t)head * N * P;
    const int half = a.rot.dims >> 1, n0 = wave * QN;
    float s[NB][CB][QN];
    auto load = [&](int p0) {
#pragma unroll
        for (int k = 0; k < NB; ++k)
            if (k == 0 || p0 + 64 * CB * k < P)
#pragma unroll
                for (int c = 0; c < CB; ++c)
#pragma unroll
                    for (int u = 0; u < QN; ++u) s[k][c][u] = S[(size_t)min(n0 + u, N - 1) * P + min(p0 + 64 * (CB * k + c) + lane, P - 1)];
    };
    load(0);
    for (int i = tid; i < 2 * N; i += 1024) {
        const bool q = i >= N;
        const int n = q ? i - N : i;
        const bool si = a.act & (q ? 2 : 1);
        const float mul = q ? a.q_mul : a.k_mul;
        const float* src = q ? qb : kb;
        float v = (si ? hy_silu(src[n]) : src[n]) * mul;
        if (n < a.rot.dims) {          // the other entry of the pair, and which of the two this is
            const int j = a.rot.interleaved ? n >> 1 : n < half ? n : n - half, o = a.rot.interleaved ? n ^ 1 : n < half ? n + half : n - half;
            const bool first = a.rot.interleaved ? !(n & 1) : n < half;
            const float w = (si ? hy_silu(src[o]) : src[o]) * mul;
            float sn, cs;
            sincosf((float)pos * a.rot.freq[j], &sn, &cs);
            v = first ? v * cs - w * sn : v * cs + w * sn;
        }
        (q ? sQ : sK)[n] = v;
    }
    float av, bv = 1.f, ge = 0.f;
    if (a.mode == 1) {
        float* mp = b.m + (size_t)a.dyn[1] * a.slot_stride + head;
        const float mprev = fresh ? 0.f : *mp;
        const float zi = a.ksrc[b.i_off + head] + (b.gbias ? b.gbias[b.i_off + head] : 0.f), zf = a.ksrc[b.f_off + head] + (b.gbias ? b.gbias[b.f_off + head] : 0.f);
        const float gi = b.cap * tanhf(zi / b.cap), fr = b.cap * tanhf(zf / b.cap), gf = fminf(fr, 0.f) - log1pf(expf(-fabsf(fr)));
        const float mt = fmaxf(gf + mprev, gi);
        av = expf(gf + mprev - mt); bv = expf(gi - mt); ge = expf(-mt);
        __syncthreads();               // every thread has read the running maximum
        if (tid == 0) *mp = mt;
    } else av = a.decay[head];
    __syncthreads();
    for (int p0 = 0; p0 < P; p0 += 64 * CB * NB) {
        if (p0 > 0) load(p0);
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            if (k > 0 && p0 + 64 * CB * k >= P) break;
#pragma unroll
            for (int c = 0; c < CB; ++c) {
                const int p = p0 + 64 * (CB * k + c) + lane;
                float x = 0.f, y = 0.f;
                if (p < V) { x = a.xsrc[a.x_off + (size_t)head * V + p]; if (a.act & 4) x = hy_silu(x); }
                else if (p < P) x = 1.f;
                const float bx = bv * x;
#pragma unroll
                for (int u = 0; u < QN; ++u) {
                    if (n0 + u >= N) break;
                    const float v = fmaf(av, fresh ? 0.f : s[k][c][u], sK[n0 + u] * bx);
                    y = fmaf(v, sQ[n0 + u], y);
                    if (p < P) S[(size_t)(n0 + u) * P + p] = v;
                }
                sY[wave][64 * (CB * k + c) + lane] = y;
            }
        }
        __syncthreads();
        for (int c = tid; c < 64 * CB * NB && p0 + c < P; c += 1024) {
            float v = 0.f;
#pragma unroll
            for (int w = 0; w < NW; ++w) v += sY[w][c];
            sP[p0 + c] = v;
        }
        __syncthreads();
    }
    // P <= 1024: a column per thread
    const float inv = a.mode == 1 ? 1.f / (fmaxf(fabsf(sP[V]), ge) + 1e-6f) : 1.f;
    const float o = tid < V ? sP[tid] * inv : 0.f;
    const float gz = tid < V && b.gate ? b.gate[head * V + tid] : 0.f, w = tid < V && b.w ? b.w[head * b.w_stride + tid] : 1.f;
    const float r = 1.f / sqrtf(hy_block_sum<1024>(o * o, red) / (float)V + b.eps);
    const float act = !b.gate ? 1.f : b.gate_act == 1 ? hy_sigmoid(gz) : hy_silu(gz);
    if (tid < V) hy_st(out + head * V + tid, o * r * w * act * b.out_mul);
}
template <typename TO, int QN>
static __global__ __launch_bounds__(1024) void hy_scan_out_kernel(HyScanOut b, TO* __restrict__ out) { hy_scan_out<TO, QN>(b, out, blockIdx.x); }

// Attention and a matrix memory side by side on one input: the heads of both are workgroups of one launch (one after the other the second waits for the first's
// last head and for a launch, on a chip that is idle but for some dozens of CUs).
template <typename TO, int NI, int QN>
static __global__ __launch_bounds__(1024) void hy_pair_one_kernel(HyAttnOne a, TO* __restrict__ out_a, HyScanOut b, TO* __restrict__ out_b) {
    if ((int)blockIdx.x < a.H) hy_attn_one<TO, NI>(a, out_a, blockIdx.x);
    else hy_scan_out<TO, QN>(b, out_b, (int)blockIdx.x - a.H);
}
