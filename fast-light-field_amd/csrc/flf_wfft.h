// Mixed-radix FFTs in LDS (radices 2..6, 8..10, 12 and a last prime), by one
// wave, several waves or a workgroup per sequence.
//
// One 64-lane wave transforms one sequence held in LDS (element stride es).
// Stockham passes as in flf_fft.h, but each pass is executed by the wave
// alone: all lanes read their butterflies' inputs into registers, the wave
// synchronises (LDS operations of one wave complete in order; the barrier
// stops the compiler from moving accesses across it), then writes the
// outputs in place.  Twiddles come from a table tw[m] = exp(-2 pi i m / L)
// (computed on the host in double precision), so no transcendental is
// evaluated per butterfly.
#pragma once
#include "flf_common.h"
#include "flf_fft.h"

namespace flf {

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Values of a pass that the compiler is not to reason about: the indices of
// every radix would otherwise be computed ahead of the loop over the passes
// and held in registers (60 to 100 more in the workgroup-level passes).
__device__ __forceinline__ void opaque_lane_length(int& lane, int& L) {
    L = __builtin_amdgcn_readfirstlane(L);
    asm volatile("" : "+v"(lane), "+s"(L));
}

// q = n / d and r = n % d for 0 <= n < 2^22 and d >= 1, from the float
// reciprocal rd = 1/d of the pass (one correction step makes it exact:
// n * rd is within 0.5 of n / d).
__device__ __forceinline__ int div_small(int n, int d, float rd, int& r) {
    int q = (int)((float)n * rd);
    r = n - q * d;
    if (r < 0) { --q; r += d; } else if (r >= d) { ++q; r -= d; }
    return q;
}

// a[t] *= w^t for t = 1..R-1, w = tw[idx] (conjugated for the inverse): running
// products, restarted from the table at every fourth power (at most 2
// roundings).
template <int R>
__device__ __forceinline__ void twiddle_powers(float2* a, const float2* __restrict__ tw, int idx, bool inv) {
    float2 w1 = tw[idx];
    if (inv) w1.y = -w1.y;
    float2 w = w1;
#pragma unroll
    for (int t = 1; t < R; ++t) {
        if (t > 1 && (t & 3) == 0) {
            w = tw[t * idx];
            if (inv) w.y = -w.y;
        } else if (t > 1) {
            w = cmul(w, w1);
        }
        a[t] = cmul(a[t], w);
    }
}

// NT lanes on one sequence: 64 (one wave), or several waves, which then meet at
// workgroup barriers (every sequence of the workgroup runs the same plan).
template <int NT>
__device__ __forceinline__ void seq_sync() {
    if constexpr (NT == 64) wave_sync();
    else __syncthreads();
}

template <int R, int LMAX, int NT, bool OPAQUE>
__device__ __forceinline__ void wave_pass(float2* buf, int es, int L, int Ns, const float2* __restrict__ tw,
                                          bool inv, int lane) {
    // (one wave, 5-smooth plans up to 1024: the registers do not limit its
    // kernels, held indices are 6 % faster)
    if constexpr (OPAQUE) opaque_lane_length(lane, L);
    constexpr int MAXQ = (LMAX / R + NT - 1) / NT;
    const int M = L / R;
    const int tstep = L / (Ns * R);
    const float rNs = 1.0f / (float)Ns;
    const float sign = inv ? 1.f : -1.f;
    float2 v[MAXQ][R];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
        const int j = lane + NT * q;
        if (j < M) {
            int k;
            div_small(j, Ns, rNs, k);
            float2 a[FLF_RADIX_MAX];
#pragma unroll
            for (int t = 0; t < R; ++t) a[t] = buf[(j + t * M) * es];
            if (k != 0) twiddle_powers<R>(a, tw, k * tstep, inv);
            dft_small<R>(a, sign);
#pragma unroll
            for (int t = 0; t < R; ++t) v[q][t] = a[t];
        }
    }
    seq_sync<NT>();
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
        const int j = lane + NT * q;
        if (j < M) {
            int k;
            const int o = div_small(j, Ns, rNs, k) * Ns * R + k;   // recomputed: fewer live registers
#pragma unroll
            for (int t = 0; t < R; ++t) buf[(o + t * Ns) * es] = v[q][t];
        }
    }
    seq_sync<NT>();
}

// Butterfly j of the last pass of an odd prime radix P (5 < P <= FLF_PRIME_MAX;
// M = Ns = L / P): y_q = sum_t x[j + t M] W^(j t) W_P^(t q), W = tw[1], W_P =
// W^M, the table tw[m] = exp(-2 pi i m / L) (conjugated for the inverse).  y_q
// goes to dst[j + q M], the positions the inputs held in src.  The powers of
// W^j are running products, re-read from the table every 8 steps (at most 7
// roundings).  With a_t the twiddled inputs and (c, s) = W_P^(t q), outputs q and
// P - q share their sums over the pairs (t, P - t),
//   y = a_0 + sum c (a_t + a_(P-t)) +- i sum s (a_t - a_(P-t)),
// 4 real operations and one table read (the same for every lane) per pair and
// q, where the sum over all t took 10 and two running products per t and q.
__device__ __forceinline__ void prime_butterfly(const float2* src, float2* dst, int es, int j, int M, int P,
                                                const float2* __restrict__ tw, bool inv) {
    constexpr int H = FLF_PRIME_MAX / 2;
    const int h = P / 2;
    const float2 a0 = src[j * es];
    float2 sp[H], df[H], y0 = a0;
    {
        float2 w1 = tw[j], wP = tw[j * P];                     // W^j, W^(j P)
        if (inv) { w1.y = -w1.y; wP.y = -wP.y; }
        float2 w = w1;
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            if (t <= h) {
                if ((t & 7) == 0) {                            // exact table value W^(j t), j t < L
                    w = tw[j * t];
                    if (inv) w.y = -w.y;
                }
                const float2 x = cmul(src[(j + t * M) * es], w);
                const float2 y = cmul(src[(j + (P - t) * M) * es], cmul(wP, cconj(w)));
                sp[t - 1] = cadd(x, y);
                df[t - 1] = csub(x, y);
                w = cmul(w, w1);
            }
        }
    }
#pragma unroll
    for (int t = 1; t <= H; ++t)
        if (t <= h) y0 = cadd(y0, sp[t - 1]);
    dst[j * es] = y0;
    for (int q = 1; q <= h; ++q) {
        float2 c = a0, d = make_float2(0.f, 0.f);
        int m = 0;                                             // t q mod P
#pragma unroll
        for (int t = 1; t <= H; ++t) {
            if (t <= h) {
                m += q;
                if (m >= P) m -= P;
                const float2 w = tw[m * M];
                c.x += sp[t - 1].x * w.x;
                c.y += sp[t - 1].y * w.x;
                d.x += df[t - 1].x * w.y;
                d.y += df[t - 1].y * w.y;
            }
        }
        if (inv) { d.x = -d.x; d.y = -d.y; }
        dst[(j + q * M) * es] = make_float2(c.x - d.y, c.y + d.x);
        dst[(j + (P - q) * M) * es] = make_float2(c.x + d.y, c.y - d.x);
    }
}

// Last pass of a prime radix in place: each lane takes its butterflies one at
// a time, whose outputs lie where its inputs did.
template <int NT>
__device__ __forceinline__ void wave_pass_prime(float2* buf, int es, int L, int P, const float2* __restrict__ tw,
                                                bool inv, int lane) {
    opaque_lane_length(lane, L);
    const int M = L / P;
    for (int j = lane; j < M; j += NT) prime_butterfly(buf, buf, es, j, M, P, tw, inv);
    seq_sync<NT>();
}

// In-place transform of one sequence by NT lanes (inv: unnormalised inverse).
// PRIME: the plan may end with an odd prime radix above 5 (kernels for lenslet
// pitches such as 7, 13, 19 are compiled separately, so that the prime pass's
// registers do not lower the occupancy of the 5-smooth kernels).
template <int LMAX, bool PRIME = false, int NT = 64>
__device__ __forceinline__ void wave_fft(float2* buf, int es, const RadixPlan& rp, const float2* __restrict__ tw,
                                         bool inv, int lane) {
    constexpr bool OPQ = PRIME || NT > 64 || LMAX > 1024;
    int Ns = 1;
    for (int p = 0; p < rp.n; ++p) {
        const int R = rp.r[p];
        switch (R) {
            case 12: wave_pass<12, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 10: wave_pass<10, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 9: wave_pass<9, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 8: wave_pass<8, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 6: wave_pass<6, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 4: wave_pass<4, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 2: wave_pass<2, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 3: wave_pass<3, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            case 5: wave_pass<5, LMAX, NT, OPQ>(buf, es, rp.L, Ns, tw, inv, lane); break;
            default:
                if constexpr (PRIME) wave_pass_prime<NT>(buf, es, rp.L, R, tw, inv, lane);   // last pass
                break;
        }
        Ns *= R;
    }
}

// Out-of-place forms for transforms longer than the register-held passes
// cover (grids above 2048 points): each pass reads one LDS buffer and writes
// the other, and a lane takes its butterflies one at a time, so no register
// array grows with the length.  Contiguous sequences (element stride 1).
template <int R>
__device__ __forceinline__ void wave_pass_oop(const float2* src, float2* dst, int L, int Ns,
                                              const float2* __restrict__ tw, bool inv, int lane) {
    opaque_lane_length(lane, L);
    const int M = L / R;
    const int tstep = L / (Ns * R);
    const float rNs = 1.0f / (float)Ns;
    const float sign = inv ? 1.f : -1.f;
    for (int j = lane; j < M; j += 64) {
        int k;
        const int g = div_small(j, Ns, rNs, k);
        float2 a[FLF_RADIX_MAX];
#pragma unroll
        for (int t = 0; t < R; ++t) a[t] = src[j + t * M];
        if (k != 0) twiddle_powers<R>(a, tw, k * tstep, inv);
        dft_small<R>(a, sign);
        const int o = g * Ns * R + k;
#pragma unroll
        for (int t = 0; t < R; ++t) dst[o + t * Ns] = a[t];
    }
    wave_sync();
}

// The prime last pass out of place.
__device__ __forceinline__ void wave_pass_prime_oop(const float2* src, float2* dst, int L, int P,
                                                    const float2* __restrict__ tw, bool inv, int lane) {
    const int M = L / P;
    for (int j = lane; j < M; j += 64) prime_butterfly(src, dst, 1, j, M, P, tw, inv);
    wave_sync();
}

// Whole transform between buffers a and b (length rp.L each); returns the
// buffer that holds the result (a after an even number of passes).
template <bool PRIME>
__device__ float2* wave_fft_pp(float2* a, float2* b, const RadixPlan& rp, const float2* __restrict__ tw, bool inv,
                               int lane) {
    int Ns = 1;
    float2* src = a;
    float2* dst = b;
    for (int p = 0; p < rp.n; ++p) {
        const int R = rp.r[p];
        switch (R) {
            case 12: wave_pass_oop<12>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 10: wave_pass_oop<10>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 9: wave_pass_oop<9>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 8: wave_pass_oop<8>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 6: wave_pass_oop<6>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 4: wave_pass_oop<4>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 2: wave_pass_oop<2>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 3: wave_pass_oop<3>(src, dst, rp.L, Ns, tw, inv, lane); break;
            case 5: wave_pass_oop<5>(src, dst, rp.L, Ns, tw, inv, lane); break;
            default:
                if constexpr (PRIME) wave_pass_prime_oop(src, dst, rp.L, R, tw, inv, lane);   // last pass
                break;
        }
        Ns *= R;
        float2* t = src;
        src = dst;
        dst = t;
    }
    return src;
}

// NS sequences per call (sequence s at buf + s * ss, element stride es),
// nseq <= NS of them present: the butterflies of all sequences share the
// wave's lanes, which a single short sequence fills only partly.
template <int R, int LMAX, int NS>
__device__ __forceinline__ void wave_pass_ns(float2* buf, int es, int ss, int nseq, int L, int Ns,
                                             const float2* __restrict__ tw, bool inv, int lane) {
    constexpr int MAXQ = (NS * (LMAX / R) + 63) / 64;
    const int M = L / R;
    const int tot = nseq * M;
    const int tstep = L / (Ns * R);
    const float rNs = 1.0f / (float)Ns, rM = 1.0f / (float)M;
    const float sign = inv ? 1.f : -1.f;
    float2 v[MAXQ][R];
    int ov[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
        const int j = lane + 64 * q;
        if (j < tot) {
            int jj, k;
            const int sq = div_small(j, M, rM, jj);
            const int g = div_small(jj, Ns, rNs, k);
            ov[q] = sq * ss + (g * Ns * R + k) * es;
            const float2* b = buf + sq * ss;
            float2 a[FLF_RADIX_MAX];
#pragma unroll
            for (int t = 0; t < R; ++t) a[t] = b[(jj + t * M) * es];
            if (k != 0) twiddle_powers<R>(a, tw, k * tstep, inv);
            dft_small<R>(a, sign);
#pragma unroll
            for (int t = 0; t < R; ++t) v[q][t] = a[t];
        }
    }
    wave_sync();
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
        const int j = lane + 64 * q;
        if (j < tot) {
            const int o = ov[q];
#pragma unroll
            for (int t = 0; t < R; ++t) buf[o + t * Ns * es] = v[q][t];
        }
    }
    wave_sync();
}

// Radices 2..5 only (plans from make_radix_plan without the wide set): the
// composite radices' code raised the small FFT's registers and slowed it.
template <int LMAX, int NS>
__device__ void wave_fft_ns(float2* buf, int es, int ss, int nseq, const RadixPlan& rp, const float2* __restrict__ tw,
                            bool inv, int lane) {
    int Ns = 1;
    for (int p = 0; p < rp.n; ++p) {
        const int R = rp.r[p];
        switch (R) {
            case 4: wave_pass_ns<4, LMAX, NS>(buf, es, ss, nseq, rp.L, Ns, tw, inv, lane); break;
            case 2: wave_pass_ns<2, LMAX, NS>(buf, es, ss, nseq, rp.L, Ns, tw, inv, lane); break;
            case 3: wave_pass_ns<3, LMAX, NS>(buf, es, ss, nseq, rp.L, Ns, tw, inv, lane); break;
            default: wave_pass_ns<5, LMAX, NS>(buf, es, ss, nseq, rp.L, Ns, tw, inv, lane); break;
        }
        Ns *= R;
    }
}

// One pass of nseq sequences of length L by the whole workgroup (NTH threads):
// element e of sequence q is buf[q * ss + e * es], butterflies dealt to the
// threads with the sequence (by_seq) or the butterfly of a sequence fastest.
// FIRST: inputs from ld(sequence, element) instead (Ns = 1, buf only written).
// Twiddles: powers of one table entry, restarted from the table at every fourth
// (at most 2 roundings).
template <int R, int MAXB, int NTH, bool FIRST, class Ld>
__device__ __forceinline__ void wg_pass(float2* buf, int es, int ss, int nseq, bool by_seq, int L, int Ns,
                                        const float2* __restrict__ tw, Ld ld) {
    int tid = threadIdx.x;
    opaque_lane_length(tid, L);
    constexpr int MAXQ = (MAXB / R + NTH - 1) / NTH;   // MAXB: most nseq * L
    const int M = L / R, total = nseq * M, d = by_seq ? nseq : M;
    const float rd = 1.0f / (float)d, rNs = 1.0f / (float)Ns;
    const int tstep = L / (Ns * R);
    float2 v[MAXQ][R];
    int o[MAXQ];
#pragma unroll
    for (int q = 0; q < MAXQ; ++q) {
        const int idx = tid + q * NTH;
        if (idx < total) {
            int lo, k = 0;
            const int hi = div_small(idx, d, rd, lo);
            const int seq = by_seq ? lo : hi, j = by_seq ? hi : lo;
            if constexpr (FIRST) {
                o[q] = seq * ss + j * R * es;
                ld(v[q], seq, j, M);
            } else {
                const int g = div_small(j, Ns, rNs, k);
                o[q] = seq * ss + (g * Ns * R + k) * es;
                const float2* b = buf + seq * ss + j * es;
#pragma unroll
                for (int t = 0; t < R; ++t) v[q][t] = b[t * M * es];
                if (Ns > 1) {
                    const float2 w1 = tw[k * tstep];
                    float2 w = w1;
#pragma unroll
                    for (int t = 1; t < R; ++t) {
                        if (t > 1) w = (t & 3) == 0 ? tw[t * k * tstep] : cmul(w, w1);
                        v[q][t] = cmul(v[q][t], w);
                    }
                }
            }
            dft_small<R>(v[q], -1.f);
        }
    }
    if constexpr (!FIRST) __syncthreads();
#pragma unroll
    for (int q = 0; q < MAXQ; ++q)
        if (tid + q * NTH < total) {
#pragma unroll
            for (int t = 0; t < R; ++t) buf[o[q] + t * Ns * es] = v[q][t];
        }
    __syncthreads();
}
struct NoLoad {
    template <int R>
    __device__ void operator()(float2 (&)[R], int, int, int) const {}
};
template <int MAXB, int NTH, bool FIRST, class Ld>
__device__ __forceinline__ void wg_pass_any(int R, float2* buf, int es, int ss, int nseq, bool by_seq, int L, int Ns,
                                            const float2* __restrict__ tw, Ld ld) {
    switch (R) {
        case 12: wg_pass<12, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 10: wg_pass<10, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 9: wg_pass<9, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 8: wg_pass<8, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 6: wg_pass<6, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 5: wg_pass<5, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 4: wg_pass<4, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 3: wg_pass<3, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        case 2: wg_pass<2, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;
        default: wg_pass<1, MAXB, NTH, FIRST>(buf, es, ss, nseq, by_seq, L, Ns, tw, ld); break;   // L = 1
    }
}

}  // namespace flf
