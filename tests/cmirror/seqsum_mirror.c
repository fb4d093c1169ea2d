/* CPU mirror of gpullama3.java_amd/csrc/gl3_seqsum.h (exact_seqsum_lds, replay_events; 4-element segments): the same predictor, trial, composition, replay
 * and verification steps in plain C, with the kernel's own places: prefixes and hard lists per wavefront's span of segments (place, before), the check of the
 * borders between spans, passes of 61 events in which every lane runs its own five adds and results move one lane up, steps rounded up to groups of four.
 * tests/test_seqsum_mirror.py runs it without a GPU.  Thread t of the kernel = loop index t here, the 64 lanes of the replaying wavefront = arrays; the
 * predictor's wavefront scan is a plain prefix sum (it is order-insensitive by design, the integer prefix is exact mod 2^32).
 *   gcc -O2 -ffp-contract=off -fno-fast-math seqsum_mirror.c -o seqsum_mirror -lm ; ./seqsum_mirror <trials> <seed>
 * exit status 0 = every trial bit-identical to the sequential chain. */
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>

static inline uint32_t f2u(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
static inline float u2f(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
static inline int imin(int a, int b) { return a < b ? a : b; }
static inline int imax(int a, int b) { return a > b ? a : b; }
static float naive(const float* x, int n, int sq, float start) {
    volatile float s = start;
    for (int i = 0; i < n; ++i) { volatile float p = sq ? x[i] * x[i] : x[i]; s = s + p; }
    return s;
}

#define SS_T 256
#define SS_EVENTS 61
#define MAXSEG 1280
static long g_fallback = 0, g_hard = 0, g_calls = 0, g_passes[8];

static uint32_t ep_x[MAXSEG], ep_y[MAXSEG];             /* prefix inside the segment's span, exponent | hard << 31 */
static int hl[MAXSEG];                                  /* hard segments of a span from the span's own place on */
static uint32_t w_nd[4]; static int w_cnt[4], w_bad[4];

/* replay_events: x is padded with four zeros */
static void replay(const float* x, int nseg, int S, int sq, float* base_, int* fail_) {
    float base = *base_; int fail = *fail_;
    const int c0n = w_cnt[0], c1n = c0n + w_cnt[1], c2n = c1n + w_cnt[2], nhard = c2n + w_cnt[3];
    const int o1 = S - c0n, o2 = S - (c1n - c0n), o3 = S - (c2n - c1n);
#define PLACE(j) ((j) + ((j) >= c0n ? o1 : 0) + ((j) >= c1n ? o2 : 0) + ((j) >= c2n ? o3 : 0))
#define BEFORE(s) (((s) >= S ? w_nd[0] : 0u) + ((s) >= 2 * S ? w_nd[1] : 0u) + ((s) >= 3 * S ? w_nd[2] : 0u))
    for (int lane = 1; lane < 4; ++lane) {
        if (lane * S >= nseg) continue;
        const uint32_t el = ep_y[lane * S - 1], er = ep_y[lane * S];
        if (!((el | er) >> 31) && el != er) fail = 1;
    }
    int passes = 0;
    for (int k0 = 0; k0 <= nhard; k0 += SS_EVENTS, ++passes) {
        float sqv[64][4], runadd[64], t2[64], made[64]; uint32_t er[64];
        for (int lane = 0; lane < 64; ++lane) {
            const int j = k0 + lane, pj = PLACE(imin(j, nhard - 1)), pp = PLACE(imin(imax(j - 1, 0), nhard - 1));
            if (pj < 0 || pj >= nseg || pp < 0 || pp >= nseg) { printf("place out of range\n"); exit(2); }
            const int h = j < nhard ? hl[pj] : nseg, ph = j > 0 ? hl[pp] : -1;
            for (int q = 0; q < 4; ++q) { volatile float v = x[4 * h + q]; v = sq ? v * v : v; sqv[lane][q] = j >= nhard || lane >= SS_EVENTS ? 0.f : v; }
            const int run = j <= nhard && h - 1 > ph && lane < SS_EVENTS;
            const uint32_t R = ep_x[imax(h - 1, 0)] + BEFORE(h - 1) - (ep_x[imax(ph, 0)] + BEFORE(ph));
            er[lane] = run ? ep_y[imin(ph + 1, nseg - 1)] & 0x7FFFFFFFu : 0u;
            runadd[lane] = run ? (float)R * u2f((er[lane] - 23u) << 23) : 0.f;
        }
        const int nev = imin(SS_EVENTS, 1 + ((imin(SS_EVENTS, nhard + 1 - k0) + 2) & ~3));
#define TERMS(dst, l, in) do { volatile float t_ = (in); t_ = t_ + runadd[l]; for (int q = 0; q < 4; ++q) t_ = t_ + sqv[l][q]; dst = t_; } while (0)
        for (int l = 0; l < 64; ++l) { TERMS(t2[l], l, base); made[l] = t2[l]; }
        for (int k = 1; k < nev; k += 4)
            for (int u = 0; u < 4; ++u) {
                float in[64];
                for (int l = 0; l < 64; ++l) in[l] = l ? t2[l - 1] : 0.f;
                for (int l = 0; l < 64; ++l) { TERMS(t2[l], l, in[l]); if (l == k + u) made[l] = t2[l]; }
            }
        for (int l = 0; l < 64; ++l)
            if (er[l]) {
                const float in = l ? made[l - 1] : base;
                volatile float after = in + runadd[l];
                if ((f2u(in) >> 23) != er[l] || (f2u(after) >> 23) != er[l]) fail = 1;
            }
        base = t2[nev - 1];
    }
    ++g_passes[imin(passes, 7)];
    *base_ = base; *fail_ = fail;
}

/* n % 4 == 0, n <= 5120, x padded with four zeros; start: the running sum in front of x[0] */
static float exact_sum(const float* x, int n, int sq, float start) {
    const int nseg = n >> 2, spt = (nseg + SS_T - 1) / SS_T;
    static float a[SS_T][5][4], qs[SS_T][5], qt[SS_T], w_tot[4], incl[SS_T];
    ++g_calls;
    for (int t = 0; t < SS_T; ++t) {
        qt[t] = 0.f;
        for (int i = 0; i < spt; ++i) {
            const float* p = x + 4 * imin(t * spt + i, nseg);
            for (int k = 0; k < 4; ++k) a[t][i][k] = sq ? p[k] * p[k] : p[k];
            qs[t][i] = (a[t][i][0] + a[t][i][1]) + (a[t][i][2] + a[t][i][3]);
            qt[t] += qs[t][i];
        }
        incl[t] = t % 64 ? incl[t - 1] + qt[t] : qt[t];
        if (t % 64 == 63) w_tot[t / 64] = incl[t];
    }
    for (int w = 0; w < 4; ++w) {
        uint32_t prefix = 0, prev = 0x80000000u; int count = 0, bad = 0;
        for (int t = 64 * w; t < 64 * w + 64; ++t) {
            const int seg0 = t * spt;
            volatile float P = start + (incl[t] - qt[t]);
            for (int v = 0; v < w; ++v) P = P + w_tot[v];
            for (int i = 0; i < spt; ++i) {
                const uint32_t rb = f2u(P) & ~1u, e = rb >> 23;
                const float R0 = u2f(rb), R1 = u2f(rb | 1u), margin = u2f((e - 10u) << 23);
                volatile float E0 = R0, E1 = R1;
                for (int k = 0; k < 4; ++k) { E0 = E0 + a[t][i][k]; E1 = E1 + a[t][i][k]; }
                volatile float D0 = E0 - R0, D1 = E1 - R1, lo = R0 - margin, hi = E0 + margin;
                const uint32_t leaves = (f2u(E0) ^ rb) | (f2u(E1) ^ rb) | (f2u(lo) ^ rb) | (f2u(hi) ^ rb);
                const int easy = (D0 == D1) & (leaves < 1u << 23) & (e - 41u < 209u) & (seg0 + i > 0) & (seg0 + i < nseg);
                const uint32_t ev = easy ? e : e | 0x80000000u;
                if (easy) { volatile float q = D0 * u2f((277u - e) << 23); prefix += (uint32_t)q; }
                bad |= !((prev | ev) >> 31) && prev != ev;
                prev = ev;
                if (seg0 + i < nseg) {
                    ep_x[seg0 + i] = prefix; ep_y[seg0 + i] = ev;
                    if (!easy) hl[64 * spt * w + count++] = seg0 + i;
                }
                P = P + qs[t][i];
            }
        }
        w_nd[w] = prefix; w_cnt[w] = count; w_bad[w] = bad;
    }
    float base = start; int fail = 0;
    replay(x, nseg, 64 * spt, sq, &base, &fail);
    g_hard += w_cnt[0] + w_cnt[1] + w_cnt[2] + w_cnt[3];
    if (fail | w_bad[0] | w_bad[1] | w_bad[2] | w_bad[3]) { ++g_fallback; return naive(x, n, sq, start); }
    return base;
}

static float rnd01(void) { return (float)rand() / (float)RAND_MAX; }

int main(int argc, char** argv) {
    const int trials = argc > 1 ? atoi(argv[1]) : 12000;
    srand(argc > 2 ? atoi(argv[2]) : 12345);
    static float x[5124];
    float carried = 0.f;                                                                     /* sums of long vectors go on from the chunk before */
    long bad = 0;
    for (int trial = 0; trial < trials; ++trial) {
        const int kind = trial % 12;
        int n = (trial % 7 == 0) ? 2048 : (trial % 7 == 1) ? 2560 : (trial % 7 == 2) ? 5120 : (trial % 7 == 3) ? 4000 : 4096;
        if (kind == 11) n = 4 * (256 + rand() % 1024);
        for (int i = 0; i < n; ++i) {
            float v;
            switch (kind) {
            case 0: v = (rnd01() - 0.5f) * 2.f; break;
            case 1: { float u1 = rnd01() + 1e-9f, u2 = rnd01(); v = sqrtf(-2.f * logf(u1)) * cosf(6.2831853f * u2) * 0.02f; } break;
            case 2: v = (float)(rand() % 8); break;                                  /* exact ties everywhere */
            case 3: v = ldexpf(1.f, rand() % 12 - 6); break;
            case 4: v = (rand() % 50 == 0) ? 100.f * rnd01() : 1e-3f * rnd01(); break;
            case 5: v = 1.0f; break;
            case 6: v = (i < 5) ? 1e-12f : rnd01(); break;
            case 7: v = (i % 97 == 0) ? 0.f : (float)(rand() % 3) * 0.5f; break;
            case 8: v = ldexpf(rnd01(), rand() % 40 - 20); break;                    /* wide dynamic range */
            case 9: v = (i == n / 2) ? 3000.f : rnd01() * 0.01f; break;              /* one giant element */
            case 10: v = (float)(1 + rand() % 4) * 0.25f; break;
            default: v = rnd01() * 3.f; break;
            }
            x[i] = v;
        }
        if (kind == 3 && trial % 24 == 3) for (int i = 0; i < n; ++i) x[i] = 0.f;
        if (kind == 10 && trial % 5 == 0) { for (int i = 0; i < n; ++i) x[i] = 2.f; x[0] = 5000.f; for (int i = 0; i < trial / 12 % 250; ++i) x[4 * (1 + rand() % (n / 4 - 1))] = 1.f; }          /* up to five passes of ties */
        for (int i = 0; i < 4; ++i) x[n + i] = 0.f;
        const int sq = trial / 12 % 3 != 1;
        if (!sq) for (int i = 0; i < n; ++i) x[i] = fabsf(x[i]);
        const float start = trial / 12 % 3 == 0 ? 0.f : carried;
        const float ref = naive(x, n, sq, start), got = exact_sum(x, n, sq, start);
        if (f2u(ref) != f2u(got)) { if (bad < 5) printf("MISMATCH trial %d kind %d n %d squares %d start %.9g: ref %.9g got %.9g\n", trial, kind, n, sq, start, ref, got); ++bad; }
        carried = ref < 1e30f ? ref * (trial % 5 ? 1.f : 1e-6f) : 0.f;
    }
    printf("trials %d mismatches %ld fallbacks %ld hard/call %.1f calls with 1 .. 6 passes", trials, bad, g_fallback, (double)g_hard / (double)g_calls);
    for (int p = 1; p < 7; ++p) printf(" %ld", g_passes[p]);
    printf("\n");
    return bad != 0;
}
