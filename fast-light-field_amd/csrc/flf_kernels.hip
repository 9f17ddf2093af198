// HIP kernels for the light-field projector and Richardson-Lucy loop (gfx950).
//
// Data flow of one projection (forward: volume -> image, backward: image ->
// volume), for each Fourier grid group g (planes sharing (fY, fX)):
//   k_small_fft    S[p][t][off][k0][k1]  = FFT_r(src[b::N, a::N])   (half plane)
//   k_mac          A[...][k0][k1]        = sum over 225 offsets of S * spectra
//   k_ifft_cols    T[...][y][k1]         = column inverse FFT, rows y < Y kept
//   k_ifft_rows_*  real rows, 'same' crop folded into A as a phase, summed over
//                  groups (forward) or written / RL-updated per plane (backward)
// and once per PSF set: k_psf_rows + k_psf_cols (pruned 2-D FFT of each
// quadrant PSF) and k_spec_pack (gather into the MAC's orbit-major layout).
#include <algorithm>
#include <type_traits>
#include <vector>

#include "flf_common.h"
#include "flf_fft.h"
#include "flf_kernels.h"
#include "flf_wfft.h"

using namespace flf;

namespace {

constexpr int FFT_THREADS = 512;
constexpr int FFT_MAXB = 16;

__device__ __forceinline__ int centred_res(int k, int r) {
    // Centred representative of residue k in Z_r, with r/2 (r even) -> 0.
    if (2 * k < r) return k;
    if (2 * k > r) return k - r;
    return 0;
}

}  // namespace

// ---------------------------------------------------------------------------
// Small FFTs of the lenslet-subsampled source (py_light_field.cpp:1001-1027):
// S_{b,a} = FFT_r(src[b::N, a::N] zero-padded to rY x rX), half spectrum.
// grid (N*N, T, nsrc), block 64 * sfft_waves.  Rows are real, so two rows are
// transformed as one complex sequence, in those two rows' storage (2 (rX/2+1)
// >= rX entries; one spare row at the end), and separated afterwards; then
// the columns of the half spectrum.  Every pass is done by the whole
// workgroup (wg_pass: two passes of radix 8 to 12 at most lengths from 64 to
// 120, the first straight from memory): shared out by waves, two sequences
// filled 40 to 50 of 64 lanes and took 3 passes of radix 2 to 5.  The r x
// (r/2+1) spectrum takes 60 KB of LDS at r = 120, so two workgroups share a CU.
// Bound: latency (the strided pixel loads, barriers), vector instructions for
// half of the time: 42k per workgroup before at r = 110, 17k now.  1455^2 x 41
// planes: 8 frames 5.05 -> 3.73 ms, one frame 700 -> 540 us.
// ---------------------------------------------------------------------------
// Variants by the longer reduced length (see small_fft_variant).
enum SmallFFT { SFFT_64, SFFT_128, SFFT_256 };
constexpr int sfft_len(SmallFFT v) { return v == SFFT_64 ? 64 : v == SFFT_128 ? 128 : 256; }
constexpr int sfft_waves(SmallFFT v) { return v == SFFT_64 ? 4 : 12; }

// Workgroup id -> work index such that the workgroups of one XCD take a
// contiguous range: the dispatcher deals consecutive workgroup ids of a grid
// row to the 8 XCDs in turn, so ids with one value of (id mod 8) share an
// XCD and its L2.  Neighbouring work items (adjacent residues, adjacent
// lenslet offsets) write neighbouring bytes, which then combine in one L2.
// A bijection on [0, n): the last n mod 8 ids map to themselves.
#ifndef FLF_XCD_REMAP
#define FLF_XCD_REMAP 1
#endif
__device__ __forceinline__ int xcd_block(int bid, int n) {
#if FLF_XCD_REMAP
    const int q = n >> 3;
    return bid < 8 * q ? (bid & 7) * q + (bid >> 3) : bid;
#else
    (void)n;
    return bid;
#endif
}
// Grouped launches: the grid groups of one projection in one dispatch.  A
// flattened block index b falls in group g for start[g] <= b < start[g + 1];
// the group is found with static indices only (selects on kernel-argument
// values); its arguments are then read from the kernel arguments with g as
// a scalar index.
struct GroupPick {
    int g, rem, n, nch, nr;                       // n: blocks of the group (start[g + 1] - start[g])
};
__device__ __forceinline__ GroupPick pick_group(const GroupedGrid& gg, int b) {
    GroupPick p{0, b, gg.start[1], gg.nchunks[0], gg.nranges[0]};
    int s0 = 0;
#pragma unroll
    for (int k = 1; k < FLF_MAX_GROUPS; ++k)
        if (k < gg.ngroups && b >= gg.start[k]) {
            p.g = k;
            s0 = gg.start[k];
            p.n = gg.start[k + 1] - gg.start[k];
            p.nch = gg.nchunks[k];
            p.nr = gg.nranges[k];
        }
    p.rem = b - s0;
    return p;
}

// Maximum over the wave's 64 lanes, in every lane.
__device__ __forceinline__ float wave_max(float x) {
#define FLF_DPP_MAX(ctrl) \
    x = fmaxf(x, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), ctrl, 0xf, 0xf, true)))
    FLF_DPP_MAX(0xB1);                            // quad_perm: lane ^ 1
    FLF_DPP_MAX(0x4E);                            // quad_perm: lane ^ 2
    FLF_DPP_MAX(0x124);                           // row_ror 4
    FLF_DPP_MAX(0x128);                           // row_ror 8
#undef FLF_DPP_MAX
    x = fmaxf(x, __shfl_xor(x, 16));
    return fmaxf(x, __shfl_xor(x, 32));
}
// Zero the MAC scales' maxima for the next projection (the last kernel of a
// projection does, after the MAC has read them).
__device__ __forceinline__ void reset_smax(float* smax, int n) {
    if (blockIdx.x == 0 && blockIdx.y == 0 && blockIdx.z == 0)
        for (int i = threadIdx.x; i < n; i += blockDim.x) smax[i] = 0.f;
}

// One (lenslet offset, frame, source plane) of a grid group; src0/src2/
// tsplit: the source buffers of the call.
template <SmallFFT V>
__device__ __forceinline__ void small_fft_body(const SmallFFTArgs& a, const float* src0, const float* src2,
                                               int tsplit, int off, int t, int z) {
    constexpr int RMAX = sfft_len(V), SFFT_WAVES = sfft_waves(V);
    extern __shared__ float2 lds[];
    const int N = a.N;
    const int b = off / N, aa = off % N;
    const int rY = a.rpY.L, rX = a.rpX.L, rXh = rX / 2 + 1;
    float2* H = lds;                              // [rY + 1][rXh]
    float2* twY = H + (rY + 1) * rXh;             // [rY]
    float2* twX = twY + rY;                       // [rX]
    float2* phY = twX + rX;                       // [rY]
    float2* phX = phY + rY;                       // [rX]
    unsigned* wgmax = reinterpret_cast<unsigned*>(phX + rX);
    if (threadIdx.x == 0) *wgmax = 0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int i = threadIdx.x; i < rY; i += blockDim.x) twY[i] = a.twY[i];
    for (int i = threadIdx.x; i < rX; i += blockDim.x) twX[i] = a.twX[i];
    const bool second = src2 && t >= tsplit;      // two-source calls: frames from two buffers
    const float* src = (second ? src2 : src0) + a.src_off[z] + (long long)(second ? t - tsplit : t) * a.src_tstride;
    // frame t's valid region (frames of one batch may be smaller than the plan)
    const int Yv = a.fdims ? a.fdims[t].x : a.Y, Xv = a.fdims ? a.fdims[t].y : a.X;
    const int Ys = max(0, (Yv - b + N - 1) / N);
    const int Xs = max(0, (Xv - aa + N - 1) / N);
    // Sub-sampling phases of this offset: exp(-2 pi i b kt0 / fY) and
    // exp(-2 pi i a kt1 / fX), kt the centred residue (0 for r/2).
    for (int i = threadIdx.x; i < rY + rX; i += blockDim.x) {
        const bool isY = i < rY;
        const int k = isY ? i : i - rY;
        const int r = isY ? rY : rX;
        const int f = isY ? a.fY : a.fX;
        const int kt = (2 * k < r) ? k : ((2 * k > r) ? k - r : 0);
        const int m = ((isY ? b : aa) * kt) % f;
        float sn, cs;
        sincospif(-2.0f * (float)m / (float)f, &sn, &cs);
        (isY ? phY : phX)[k] = make_float2(cs, sn);
    }
    if constexpr (V == SFFT_256) {
        for (int i = Ys * rXh + threadIdx.x; i < rY * rXh; i += blockDim.x) H[i] = make_float2(0.f, 0.f);
        __syncthreads();
        for (int q = wv; 4 * q < Ys; q += SFFT_WAVES) {
            const int y0 = 4 * q;
            const int np = (y0 + 2 < Ys) ? 2 : 1;      // row pairs in this group of four rows
            float2* P = H + (long long)y0 * rXh;      // pair s at P + 2 s rXh
            // All loads of the group's four rows are issued before any is used.
            constexpr int XC = RMAX / 64;              // 64-lane column chunks per row
            float v[2][XC][2];
#pragma unroll
            for (int sq = 0; sq < 2; ++sq) {
                const int ya = y0 + 2 * sq, yb = ya + 1;
                const float* r0 = src + (long long)(b + N * ya) * a.src_pitch + aa;
                const float* r1 = src + (long long)(b + N * yb) * a.src_pitch + aa;
#pragma unroll
                for (int c = 0; c < XC; ++c) {
                    const int x = lane + 64 * c;
                    const bool in = sq < np && x < Xs;
                    v[sq][c][0] = in ? r0[N * x] : 0.f;
                    v[sq][c][1] = (in && yb < Ys) ? r1[N * x] : 0.f;
                }
            }
#pragma unroll
            for (int sq = 0; sq < 2; ++sq)
#pragma unroll
                for (int c = 0; c < XC; ++c) {
                    const int x = lane + 64 * c;
                    if (sq < np && x < rX) P[2 * sq * rXh + x] = make_float2(v[sq][c][0], v[sq][c][1]);
                }
            wave_sync();
            wave_fft_ns<RMAX, 2>(P, 1, 2 * rXh, np, a.rpX, twX, false, lane);
            // Separate: row ya = (Z + Zc)/2, row yb = (Z - Zc)/(2i), Zc = conj Z(-k);
            // all reads before the in-place writes.
            float2 ev[2][2], od[2][2];
#pragma unroll
            for (int sq = 0; sq < 2; ++sq)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int k = lane + 64 * m;
                    if (sq < np && k < rXh) {
                        const float2* Z = P + 2 * sq * rXh;
                        const float2 zk = Z[k];
                        const float2 zc = cconj(Z[(rX - k) % rX]);
                        ev[sq][m] = make_float2(0.5f * (zk.x + zc.x), 0.5f * (zk.y + zc.y));
                        od[sq][m] = make_float2(0.5f * (zk.y - zc.y), -0.5f * (zk.x - zc.x));
                    }
                }
            wave_sync();
#pragma unroll
            for (int sq = 0; sq < 2; ++sq)
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const int k = lane + 64 * m;
                    if (sq < np && k < rXh) {
                        const int ya = y0 + 2 * sq;
                        H[ya * rXh + k] = ev[sq][m];
                        H[(ya + 1) * rXh + k] = (ya + 1 < Ys) ? od[sq][m] : make_float2(0.f, 0.f);
                    }
                }
            wave_sync();
        }
        __syncthreads();
        for (int c = 2 * wv; c < rXh; c += 2 * SFFT_WAVES)
            wave_fft_ns<RMAX, 2>(H + c, rXh, 1, min(2, rXh - c), a.rpY, twY, false, lane);
        __syncthreads();
    } else {
        // Every pass by the whole workgroup.  Rows: sequence q is the row pair
        // (2 q, 2 q + 1) as one complex sequence, stored in the pair's rows of H;
        // the first pass loads it from memory.
        constexpr int NTH = 64 * SFFT_WAVES, MAXB = (RMAX / 2 + 1) * RMAX;
        const int np = (Ys + 1) / 2;
        for (int i = 2 * np * rXh + threadIdx.x; i < rY * rXh; i += NTH) H[i] = make_float2(0.f, 0.f);
        const float* r0 = src + (long long)b * a.src_pitch + aa;
        const int rp = N * a.src_pitch;           // (row offsets within a plane: 32 bits)
        auto load = [&](auto& v, int q, int j, int M) {
            constexpr int R = sizeof(v) / sizeof(v[0]);
            const float* ra = r0 + 2 * q * rp + N * j;
            const bool two = 2 * q + 1 < Ys;
#pragma unroll
            for (int t = 0; t < R; ++t) {
                const bool in = j + t * M < Xs;
                const int x = in ? N * t * M : 0;
                v[t].x = in ? ra[x] : 0.f;
                v[t].y = in && two ? ra[x + rp] : 0.f;
            }
        };
        if (np > 0) {
            wg_pass_any<MAXB, NTH, true>(a.rpX.n ? a.rpX.r[0] : 1, H, 1, 2 * rXh, np, false, rX, 1, twX, load);
            int Ns = a.rpX.n ? a.rpX.r[0] : 1;
            for (int p = 1; p < a.rpX.n; ++p) {
                wg_pass_any<MAXB, NTH, false>(a.rpX.r[p], H, 1, 2 * rXh, np, false, rX, Ns, twX, NoLoad());
                Ns *= a.rpX.r[p];
            }
        }
        // Separate: row ya = (Z + Zc)/2, row yb = (Z - Zc)/(2i), Zc = conj Z(-k);
        // all reads before the in-place writes.
        {
            constexpr int MQ = (RMAX / 2 * (RMAX / 2 + 1) + NTH - 1) / NTH;
            const float rrx = 1.0f / (float)rXh;
            float2 ev[MQ], od[MQ];
#pragma unroll
            for (int m = 0; m < MQ; ++m) {
                const int i = threadIdx.x + m * NTH;
                if (i < np * rXh) {
                    int k;
                    const int q = div_small(i, rXh, rrx, k);
                    const float2* Z = H + 2 * q * rXh;
                    const float2 zk = Z[k], zc = cconj(Z[k == 0 ? 0 : rX - k]);
                    ev[m] = make_float2(0.5f * (zk.x + zc.x), 0.5f * (zk.y + zc.y));
                    od[m] = make_float2(0.5f * (zk.y - zc.y), -0.5f * (zk.x - zc.x));
                    if (2 * q + 1 >= Ys) od[m] = make_float2(0.f, 0.f);
                }
            }
            __syncthreads();
#pragma unroll
            for (int m = 0; m < MQ; ++m) {
                const int i = threadIdx.x + m * NTH;
                if (i < np * rXh) {
                    int k;
                    const int q = div_small(i, rXh, rrx, k);
                    H[2 * q * rXh + k] = ev[m];
                    H[(2 * q + 1) * rXh + k] = od[m];
                }
            }
            __syncthreads();
        }
        int Ns = 1;
        for (int p = 0; p < a.rpY.n; ++p) {
            wg_pass_any<MAXB, NTH, false>(a.rpY.r[p], H, rXh, 1, rXh, true, rY, Ns, twY, NoLoad());
            Ns *= a.rpY.r[p];
        }
    }
    // Orbit-ordered, phase-folded output S[chunk][off][j] for the first NH
    // residues of each chunk's residue list (the MAC reads one contiguous
    // block per chunk), by the table sidx: H row and column, conjugated where
    // only the negated residue is in the half plane (its phases are conjugates
    // too).  All of a thread's table loads are in flight before the first is used.
    float2* S = a.S + a.S_off[z] + (long long)t * a.S_tstride + off * a.NH;
    const int NH = a.NH, lg = NH == 4 ? 2 : 1, step = N * N * NH;
    const int total = a.nchunks * NH;
    float mx = 0.f;                               // largest component written
    constexpr int OU = 8;
    for (int i0 = threadIdx.x; i0 < total; i0 += OU * blockDim.x) {
        unsigned sx[OU];
#pragma unroll
        for (int u = 0; u < OU; ++u) sx[u] = a.sidx[min(i0 + u * (int)blockDim.x, total - 1)];
#pragma unroll
        for (int u = 0; u < OU; ++u) {
            const int i = i0 + u * (int)blockDim.x;
            if (i < total) {
                const int k1 = sx[u] & 0xff, k0 = (sx[u] >> 8) & 0xff;
                float2 v = cmul(H[k0 * rXh + k1], cmul(phY[k0], phX[k1]));
                if (sx[u] >> 31) v.y = -v.y;
                S[(long long)(i >> lg) * step + (i & (NH - 1))] = v;
                mx = fmaxf(mx, fmaxf(fabsf(v.x), fabsf(v.y)));   // (NaN does not count: it scales to NaN)
            }
        }
    }
    // The plane's and frame's largest component, for the MAC's scales: one
    // atomic per workgroup, spread over FLF_SMAX_WAYS words (atomics on one
    // word follow each other at about 25 ns: 225 took 6 us).
    mx = wave_max(mx);
    if (lane == 0) atomicMax(wgmax, __builtin_bit_cast(unsigned, mx));
    __syncthreads();
    if (threadIdx.x == 0)
        atomicMax(reinterpret_cast<unsigned*>(a.smax + ((long long)z * a.smax_zstride + t) * FLF_SMAX_WAYS) + off % FLF_SMAX_WAYS,
                  *wgmax);
}

template <SmallFFT V>
__global__ __launch_bounds__(64 * sfft_waves(V)) void k_small_fft(SmallFFTArgs a) {
    small_fft_body<V>(a, a.src, a.src2, a.tsplit, xcd_block(blockIdx.x, a.N * a.N), blockIdx.y, blockIdx.z);
}
// grid (N*N, T, sum over groups of their source planes): z flattened over
// (group, plane).
template <SmallFFT V>
__global__ __launch_bounds__(64 * sfft_waves(V)) void k_small_fft_grouped(SmallFFTGrouped ga) {
    const GroupPick p = pick_group(ga.gg, blockIdx.z);
    const SmallFFTArgs& a = ga.a[p.g];
    small_fft_body<V>(a, a.src, a.src2, a.tsplit, xcd_block(blockIdx.x, a.N * a.N), blockIdx.y, p.rem);
}

// ---------------------------------------------------------------------------
// PSF spectra, stage 1: row FFTs of the s2 non-zero rows of each quadrant PSF
// (zero padded to fX), half plane kept.  (py_light_field.cpp:757-812 computes
// the same pruned 2-D transform column-first on the full plane.)
// grid (ceil(s2/RB), nu); LDS RB*fX float2.
// ---------------------------------------------------------------------------
template <bool PRIME>
__global__ __launch_bounds__(FFT_THREADS) void k_psf_rows(PsfRowArgs a) {
    extern __shared__ float2 sh[];
    const int u = blockIdx.y;
    const int y0 = blockIdx.x * a.RB;
    const int nrows = min(a.RB, a.s2 - y0);
    const int fX = a.rpX.L, rfX = fX / 2 + 1, s2 = a.s2, h = a.h;
    const int bu = a.u_bu[u], au = a.u_au[u];
    const bool tr = bu > au;   // Q[a][b] for a > b is stored as the transpose of Q[b][a]
    const float* Q = a.Q + ((long long)(tr ? au : bu) * h + (tr ? bu : au)) * s2 * s2;
    for (int i = threadIdx.x; i < nrows * fX; i += blockDim.x) {
        int r = i / fX, x = i - r * fX;
        int y = y0 + r;
        float v = 0.f;
        if (x < s2) v = tr ? Q[(long long)x * s2 + y] : Q[(long long)y * s2 + x];
        sh[i] = make_float2(v, 0.f);
    }
    __syncthreads();
    lds_fft<FFT_MAXB, PRIME>(sh, a.rpX, nrows, 1, fX, -1.f);
    float2* out = a.tmp + (long long)u * s2 * rfX;
    for (int i = threadIdx.x; i < nrows * rfX; i += blockDim.x) {
        int r = i / rfX, k1 = i - r * rfX;
        out[(long long)(y0 + r) * rfX + k1] = sh[r * fX + k1];
    }
}

// ---------------------------------------------------------------------------
// PSF spectra, stage 2: column FFTs (length fY, input rows >= s2 are zero).
// grid (ceil(rfX/CB), nu); LDS CB*fY float2 (column-major).
// ---------------------------------------------------------------------------
template <bool PRIME>
__global__ __launch_bounds__(FFT_THREADS) void k_psf_cols(PsfColArgs a) {
    extern __shared__ float2 sh[];
    const int u = blockIdx.y;
    const int fY = a.rpY.L, rfX = a.rfX, s2 = a.s2;
    const int c0 = blockIdx.x * a.CB;
    const int ncol = min(a.CB, rfX - c0);
    const float2* in = a.tmp + (long long)u * s2 * rfX;
    for (int i = threadIdx.x; i < fY * a.CB; i += blockDim.x) {
        int y = i / a.CB, c = i - y * a.CB;
        float2 v = make_float2(0.f, 0.f);
        if (y < s2 && c < ncol) v = in[(long long)y * rfX + c0 + c];
        sh[c * fY + y] = v;
    }
    __syncthreads();
    lds_fft<FFT_MAXB, PRIME>(sh, a.rpY, a.CB, 1, fY, -1.f);
    float2* out = a.spec + (long long)u * fY * rfX;
    for (int i = threadIdx.x; i < fY * a.CB; i += blockDim.x) {
        int y = i / a.CB, c = i - y * a.CB;
        if (c < ncol) out[(long long)y * rfX + c0 + c] = sh[c * fY + y];
    }
}

// ---------------------------------------------------------------------------
// Gather the natural-layout spectra of one plane into the orbit-major layout
// of the MAC, each value pre-multiplied by w^(bu*m2 + au*n2) and rho^{-1/2},
// w = exp(-2 pi i / (2N)) (m2, n2: half-unit aliases; see k_mac), and split
// into two fp16 numbers:
//   G[chunk][plane][kg][hi, lo][item][8 halves]
// One 16-byte unit (item, kg) holds the (Re, Im) of 4 spectrum values: the 4
// slots of stored spectrum u = kg (square grids), or the 2 slots of u = 2 kg
// and 2 kg + 1 (non-square; zeros past the last u).  Values are scaled by a
// power of two per (item, plane) so that the item's largest component lies in
// [2^14, 2^15): hi + lo then holds 23 of its 24 significant bits (measured
// against 64 bits at k_mac).  The imaginary parts of items whose first slot
// lies on a negated residue are negated (see k_mac).  E[chunk][plane][item]
// [slot] is the factor of the item's outputs: outer phase, 'same'-crop shift
// and the inverse of the scale; psi[chunk][plane][residue][5] the flip factors.
// grid (ceil(FLF_CHUNK_MAX / PACK_ITEMS), nchunks), block 256: PACK_ITEMS
// items x 8 lanes over the spectra, the float values held in LDS between the
// search for the largest and the split (each value read from memory once).
// ---------------------------------------------------------------------------
constexpr int PACK_ITEMS = 32;
__device__ __forceinline__ unsigned pack_half2(float a, float b) {
    const _Float16 x = (_Float16)a, y = (_Float16)b;
    return (unsigned)__builtin_bit_cast(unsigned short, x) | ((unsigned)__builtin_bit_cast(unsigned short, y) << 16);
}
// What fp16 rounding leaves of x (exact: x has 24 significant bits, the
// rounded value 11 of them or x is below the fp16 range's bottom).
__device__ __forceinline__ float half_rest(float x) { return x - (float)(_Float16)x; }
// 2^e as a float (e clamped to [-120, 120]).
__device__ __forceinline__ float exp2_int(int e) {
    e = e < -120 ? -120 : (e > 120 ? 120 : e);
    return __builtin_bit_cast(float, (unsigned)(127 + e) << 23);
}
// Power of two that brings the magnitude m into [2^top, 2^(top+1)); 1 for
// zero, infinity and NaN (which then reach the results unscaled).
__device__ __forceinline__ int scale_exp(float m, int top) {
    const unsigned b = __builtin_bit_cast(unsigned, m) & 0x7fffffffu;
    const int ex = (int)(b >> 23);
    const int e = min(max(top + 127 - ex, -120), 120);       // (a denormal m: 120)
    return b == 0 || ex == 255 ? 0 : e;
}

__global__ __launch_bounds__(256) void k_spec_pack(SpecPackArgs a) {
    extern __shared__ float2 pk[];                   // [nu][PACK_ITEMS][slots], then the lanes' maxima [8][PACK_ITEMS]
    float* mx = reinterpret_cast<float*>(pk + a.nu * PACK_ITEMS * a.slots);
    const int cidx = blockIdx.y;
    const ChunkDesc* ch = a.chunks + cidx;
    const int n_items = ch->n_items;
    const int i0 = blockIdx.x * PACK_ITEMS;
    if (i0 >= n_items) return;
    const int il = threadIdx.x & (PACK_ITEMS - 1), ug = threadIdx.x / PACK_ITEMS;
    const int i = min(i0 + il, n_items - 1);         // lanes past the end repeat the last item, unwritten
    const bool valid = i0 + il < n_items;
    const long long item_base = ch->item_base;
    const ItemDesc it = a.items[item_base + i];
    const int slots = a.slots, NH = slots, N = a.N;
    const int sig = a.s2 - 2 + N;
    const int m2 = it.m2[0], n2 = it.n2[0];
    // rho_i^{-1/2}: the phase ratio of the two uses reading slot i, the same
    // for all output slots of the item (exponents in 1/(4N) turns).
    int rho[4];
    rho[0] = sig * (m2 + n2);
    rho[1] = sig * (n2 - m2);
    rho[2] = sig * (m2 + n2);
    rho[3] = sig * (m2 - n2);
    const bool neg = it.res[0] >= NH;
    float m = 0.f;
    for (int u = ug; u < a.nu; u += 8) {
        const int bu = a.u_bu[u], au = a.u_au[u];
        const float2* spec = a.spec + (long long)u * a.fY * a.rfX;
        for (int j = 0; j < slots; ++j) {
            const long long e = 2LL * ((long long)bu * it.m2[j] + (long long)au * it.n2[j]) - rho[j];
            float2 v = cmul(spec[it.pos[j]], phase_frac(e, 4 * N));
            if (neg) v.y = -v.y;
            m = fmaxf(m, fmaxf(fabsf(v.x), fabsf(v.y)));
            pk[(u * PACK_ITEMS + il) * slots + j] = v;
        }
    }
    mx[ug * PACK_ITEMS + il] = m;
    __syncthreads();
    for (int q = 0; q < 8; ++q) m = fmaxf(m, mx[q * PACK_ITEMS + il]);
    const int ea = scale_exp(m, 14);
    const float s = exp2_int(ea);
    uint4* G = a.G + (item_base * a.nP + (long long)a.p * n_items) * a.kg * 2;
    for (int g = ug; g < a.kg; g += 8) {
        unsigned h[4], l[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int u = slots == 4 ? g : 2 * g + (q >> 1), j = slots == 4 ? q : (q & 1);
            float2 v = u < a.nu ? pk[(u * PACK_ITEMS + il) * slots + j] : make_float2(0.f, 0.f);
            v.x *= s;
            v.y *= s;
            h[q] = pack_half2(v.x, v.y);
            l[q] = pack_half2(half_rest(v.x), half_rest(v.y));
        }
        if (valid) {
            G[(2LL * g + 0) * n_items + i] = make_uint4(h[0], h[1], h[2], h[3]);
            G[(2LL * g + 1) * n_items + i] = make_uint4(l[0], l[1], l[2], l[3]);
        }
    }
    if (blockIdx.x == 0 && threadIdx.x < NH) {
        // flip factors of the chunk's residues: exp(-2 pi i (s2-1) kt / f), as
        // [residue][1, row flip, column flip, both, 0]
        float2 w[2];
        for (int ax = 0; ax < 2; ++ax) {
            const int k = ax == 0 ? ch->res0[threadIdx.x] : ch->res1[threadIdx.x];
            const int f = ax == 0 ? a.fY : a.fX, r = f / N;
            w[ax] = phase_frac((long long)(a.s2 - 1) * centred_res(k, r), f);
        }
        float2* o = a.psi + (((long long)cidx * a.nP + a.p) * NH + threadIdx.x) * 5;
        o[0] = make_float2(1.f, 0.f);
        o[1] = w[0];
        o[2] = w[1];
        o[3] = cmul(w[0], w[1]);
        o[4] = make_float2(0.f, 0.f);
    }
    if (ug < slots && valid) {
        const int j = ug;
        const int c2 = (a.s2 - 1) / 2;
        const int outer = j == 0 ? sig * (m2 + n2) : j == 1 ? sig * (n2 - m2) : j == 2 ? sig * (n2 + m2) : sig * (m2 - n2);
        const int k0 = it.pos[j] / a.rfX, k1 = it.pos[j] - k0 * a.rfX;
        // exp(+2 pi i c2 (k0/fY + k1/fX)): c2 < f / 2 and k < f <= FLF_MAX_FOURIER, 32-bit products
        float fr = (float)((c2 * k0) % a.fY) / (float)a.fY + (float)((c2 * k1) % a.fX) / (float)a.fX;
        fr -= rintf(fr);
        float sn, cs;
        sincospif(2.0f * fr, &sn, &cs);
        const float2 v = cmul(phase_frac_i(outer, 4 * N), make_float2(cs, sn));
        const float is = exp2_int(-ea);
        a.E[(item_base * a.nP + (long long)a.p * n_items + i) * slots + j] = make_float2(v.x * is, v.y * is);
    }
}

// ---------------------------------------------------------------------------
// The multiply-accumulate over the N*N lenslet offsets.
//
// For an item with base alias (m2, n2) (half units) and output slots P0..P3,
// every output accumulates
//   A_j = w4^(outer_j) * sum_u sum_i [ P_{j,i,u} Re g_i + M_{j,i,u} Im g_i ]
// with g_i the stored spectrum value of slot i (pre-multiplied by
// w2^(bu m2_i + au n2_i) and rho_i^{-1/2}), w4 = exp(-2 pi i/(4N)),
// outer = sig*(m2+n2), sig*(n2-m2), sig*(n2+m2), sig*(m2-n2), sig = s2-2+N.
// P and M combine the small-FFT values s of the two uses reading slot i at
// output j, s = S_{b,a}(kappa) exp(-2 pi i (beta_b kt0/fY + alpha_a kt1/fX)),
// beta = b (b <= N/2) or b + s2 - 1 (row-flipped offsets), likewise alpha:
// P = s_plain + s_conj, M = i (s_plain - s_conj).
// This is the accumulation of py_light_field.cpp:303-341, 1029-1087 with the
// mirror multipliers of projector.py:137-151 and the 'same' crop
// (projector.py:792-796) folded into phases.
//
// As a matrix product.  The pair type of source slot i at output slot j is
// pt = i XOR j, so for the items of one residue class (their slots lie on the
// same residues res_j) and one output slot j
//   out_j[item][(f, c)] = sum_{(u, i, r)} A[item][(u, i, r)] B_j[(u, i, r)][(f, c)]
// with A the item's stored values (r = Re, Im), shared by every slot, and B_j
// the P (r = Re) and M (r = Im) components c of frame f at residue res_j, pair
// type i XOR j.  S(-k) = conj S(k) makes the table of a negated residue
// (P*, -M*): such outputs take the table of the positive residue with the
// sign of M flipped and are conjugated afterwards, so only the first NH
// residues of an orbit have tables.  M also changes sign for odd j and
// pt >= 2 (the alias order of the transposed slots).
//
// Matrix cores.  v_mfma_f32_16x16x32_f16: 16 items x 16 columns (NS slots x
// 8 / NS frames x (Re, Im)), K = 32 = 4 spectra of a square grid.  Both
// operands are fp32 numbers split into two fp16 ones (hi + lo: 23 of 24
// significant bits, after a power-of-two scale per item and per frame), and all
// four products hi*hi, lo*hi, hi*lo, lo*lo are taken with fp32 accumulation;
// the three small ones are summed apart, so an accumulator is rounded 5 times
// per 4 spectra where an fp32 FMA chain rounds 32 times.  Relative L2 error of
// whole projections against 64 bits, this kernel / the fp32 FMA kernel it
// replaced: 1455^2 x 41 planes forward 1.06e-7 / 1.04e-7, backward 1.63e-7 /
// 1.66e-7; RL at 2048^2 3.28e-7 / 3.25e-7, 997 x 1171 (Nnum 13) 2.74e-7 /
// 3.00e-7, 1273 x 1463 (Nnum 19) 6.43e-7 / 6.34e-7.
//
// One workgroup: one chunk, 8 waves, one tile (<= 32 items of a class) per
// wave; a plane range's planes in turn.  Per plane the table of P and M goes
// to LDS once (read as 16-byte B operands, conflict free) while the previous
// plane's products run; the stored spectra are streamed from memory straight
// into the A operands, RING K steps ahead.  Bound: HBM up to 4 frames (1455^2 x
// 41 planes, one frame: forward 3.16 ms for 17.8 GB = 5.6 TB/s, a plain read
// of such runs reaches 6.2; the FMA kernel 4.07 ms), matrix and vector issue
// at 8 (forward 13.3 -> 4.4 ms, backward 17.0 -> 5.5 ms).
// ---------------------------------------------------------------------------
namespace {

// Use types (order of the per-spectrum use table): 0 id, 1 both flips,
// 2 row flip, 3 column flip, 4..7 the same for the transposed PSF.
// The two uses that read the same slot of an item always pair a plain and a
// conjugated read; their pair types (plain, conj) are
//   quad:  0 (id, both)  1 (row, col)  2 (Tid, Tboth)  3 (Tcol, Trow)
//   pair:  0 (id, both)  1 (row, col)
// (the planner's pair table lists their source offsets).

typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4f mfma_f16(v4u a, v4u b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}

}  // namespace

constexpr int MAC_THREADS = 64 * FLF_CHUNK_TILES;

// Shapes of a MAC workgroup.  NS output slots share the 16 columns of a
// matrix instruction, so it takes FB = 8 / NS frames: few frames with NS = 1
// would leave most columns empty.
template <int SLOTS, int NS>
struct MacShape {
    static constexpr int NH = SLOTS;              // residues with tables (the rest by conjugation)
    static constexpr int NPT = SLOTS;             // pair types
    static constexpr int UPG = SLOTS == 4 ? 1 : 2;   // spectra per 16-byte unit
    static constexpr int FB = FLF_MAC_FB / NS;
    static constexpr int COLS = 2 * FB;           // table columns per (residue, unit)
    // Waves per SIMD: 4 (two workgroups per CU) where the tables leave LDS and
    // the accumulators registers for it, else 2 with more loads in flight each.
    static constexpr int WAVES = NS == SLOTS ? 4 : 2;
    static constexpr int RING = WAVES == 4 ? 2 : 3;   // K steps of A operands in flight per wave
    static constexpr int KB = WAVES == 4 ? 10 : 9;    // K steps per table batch, a multiple of RING
    static constexpr int NF = SLOTS / NS;         // B operands (groups of NS slots) per K step
    // 16-byte units of one residue's table; the pad puts the residues that one
    // operand read touches (NS > 1) on different banks
    static constexpr int RS = 4 * KB * COLS + (NS > 1 ? COLS : 0);
    static constexpr int TAB = NH * RS;           // units of one half (hi or lo) of a table
    static constexpr int NT = (KB * 4 * UPG * NPT * FB + MAC_THREADS - 1) / MAC_THREADS;   // entries per thread
    static constexpr int E = FLF_CHUNK_TILES * FLF_TILE * SLOTS;                              // output factors
    static constexpr int HM = (FLF_MAX_N + 1) / 2, PAIRS = (SLOTS == 4 ? HM * (HM + 1) / 2 : HM * HM) * NPT;   // the most
    // two tables (the one in use and the next), the output factors of every
    // wave's tile, the items' bins, the pair list, the inverse scales of two
    // planes, every wave's flip factors
    static constexpr size_t LDS = (size_t)4 * TAB * 16 + (size_t)E * 8 + (size_t)FLF_CHUNK_MAX * 8 + (size_t)PAIRS * 4 + (size_t)2 * FB * 4 +
                                  (size_t)FLF_CHUNK_TILES * 5 * NH * 8;
};

// The value of lane ^ 1.
__device__ __forceinline__ float lane_xor1(float x) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0xB1, 0xf, 0xf, true));
}

// One workgroup: chunk cidx, plane range `range` of nranges, frame block
// fblock.  PER_PLANE: store each plane's accumulator (back projection);
// otherwise the planes of the range are summed (forward projection).
template <int SLOTS, int NS, bool PER_PLANE>
__device__ __forceinline__ void mac_body(const MacArgs& a, int cidx, int range, int nranges, int fblock) {
    using M = MacShape<SLOTS, NS>;
    constexpr int NH = M::NH, NPT = M::NPT, UPG = M::UPG, FB = M::FB, NF = M::NF, NT = M::NT, MAC_KB = M::KB, MAC_RING = M::RING;
    extern __shared__ uint4 mac_lds[];
    char* T = reinterpret_cast<char*>(mac_lds);                   // [2 stages][hi, lo][residue][unit][column], 16 bytes each
    float2* Es = reinterpret_cast<float2*>(T + 4 * M::TAB * 16);
    ushort4* wpos = reinterpret_cast<ushort4*>(Es + M::E);        // [item]: GridTables::wpos
    unsigned* prs = reinterpret_cast<unsigned*>(wpos + FLF_CHUNK_MAX);   // [spectrum][pair type]: GridTables::pairs, 16 bits each
    float* inv = reinterpret_cast<float*>(prs + M::PAIRS);        // [2 planes][frame]
    float2* psis = reinterpret_cast<float2*>(inv + 2 * FB);       // [wave][NH][5], see k_spec_pack

    const ChunkDesc* ch = a.chunks + cidx;
    const long long item_base = ch->item_base;
    const int n_items = __builtin_amdgcn_readfirstlane(ch->n_items);
    const int n_tiles = __builtin_amdgcn_readfirstlane(ch->n_tiles);
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int col = lane & 15, kq = lane >> 4;    // operand column / row, K group
    const int jj = col / M::COLS;                 // this lane's output column: slot jj + NS t of operand t,
    const int f = (col % M::COLS) >> 1, c = col & 1;              // frame, component
    const int NN = a.N * a.N;
    const int t0 = fblock * FB;
    const int nf = min(FB, a.T - t0);             // frames of this block
    const int nu = a.nu, KG = a.kg;
    const int nkr = (KG + 3) / 4;                 // K steps with data
    const int nks = (nkr + MAC_RING - 1) / MAC_RING * MAC_RING;   // a multiple of the ring (zeros in the table)
    const int nbatch = (nks + MAC_KB - 1) / MAC_KB;               // table batches per plane

    // This wave's tile (waves without one repeat tile 0 and store nothing).
    const bool active = wv < n_tiles;
    const TileDesc td = a.tiles[ch->tile_base + (active ? wv : 0)];
    const int start = __builtin_amdgcn_readfirstlane(td.start);
    const int count = __builtin_amdgcn_readfirstlane(td.count);
    // Per operand t, for this lane's slot j = jj + NS t (wave-uniform for NS = 1):
    int tb[NF];                                   // byte offset of its table unit, K step 0
    bool cj[NF];                                  // it lies on a negated residue
    unsigned mlo[NF], mhi[NF];                    // sign of M for pair types 0, 1 and 2, 3
    const bool cj0 = (int)td.res[0] >= NH;
#pragma unroll
    for (int t = 0; t < NF; ++t) {
        int q = __builtin_amdgcn_readfirstlane((int)td.res[NS * t]);
#pragma unroll
        for (int s = 1; s < NS; ++s) q = jj == s ? __builtin_amdgcn_readfirstlane((int)td.res[NS * t + s]) : q;
        cj[t] = q >= NH;
        tb[t] = ((cj[t] ? q - NH : q) * M::RS + kq * M::COLS + 2 * f + c) * 16;
        mlo[t] = cj[t] != cj0 ? 0x80000000u : 0u;
        mhi[t] = mlo[t] ^ (SLOTS == 4 && ((jj + NS * t) & 1) ? 0x80000000u : 0u);
    }
    // A operand rows: lane l holds item l % 16 of each 16-item half of the
    // tile (rows past the tile repeat its last item; their results are unused)
    // and unit l / 16 of the K step, as byte offsets; in the last step with
    // data, units past the last one repeat it (against zeros in the table).
    unsigned ao[2], al[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = start + min(16 * h + col, count - 1);
        ao[h] = (unsigned)(kq * 2 * n_items + row) * 16;
        al[h] = (unsigned)(min(kq, KG - 1 - 4 * (nkr - 1)) * 2 * n_items + row) * 16;
    }

    // Planes of this workgroup: an even share of the group's nP planes for
    // nranges plane ranges (nranges = nP gives one plane per workgroup).
    const int pb = (int)(((long long)range * a.nP) / nranges);
    const int pe = (int)(((long long)(range + 1) * a.nP) / nranges);
    auto next_plane = [&](int p) {
        while (p < pe && !a.enable.on(p)) ++p;
        return p;
    };

    const char* Gc = reinterpret_cast<const char*>(a.G) + item_base * a.nP * KG * 32;
    const long long gplane = (long long)KG * n_items * 32;
    auto load_a = [&](v4u (&q)[4], int p, int ks) {
        const int k = min(ks, nkr - 1);
        const char* b = Gc + p * gplane + (long long)k * n_items * 128;
        const bool last = k == nkr - 1;
        const unsigned o0 = last ? al[0] : ao[0], o1 = last ? al[1] : ao[1];
        q[0] = *reinterpret_cast<const v4u*>(b + o0);
        q[1] = *reinterpret_cast<const v4u*>(b + n_items * 16 + o0);
        q[2] = *reinterpret_cast<const v4u*>(b + o1);
        q[3] = *reinterpret_cast<const v4u*>(b + n_items * 16 + o1);
    };

    // ---- the table, one stage = (plane, batch of K steps) ----
    // Thread's entries: q = tid + 512 k -> pair type, frame, spectrum.
    // (from an opaque copy of the thread id at each use, so that what follows
    // from it is not kept in registers across the plane loop)
    constexpr int ESTEP = MAC_THREADS / (NPT * FB);
    struct Entry {
        int pt, f, u;
    };
    auto entry = [&]() {
        int t = tid;
        asm volatile("" : "+v"(t));
        return Entry{t & (NPT - 1), (t / NPT) & (FB - 1), t / (NPT * FB)};
    };
    float2* psi = psis + wv * 5 * NH;
    auto use_of = [&](int b, int ul, int pt) {    // the entry's plain and conjugated use (past the last spectrum: zeros)
        const int u = b * (MAC_KB * 4 * UPG) + ul;
        const unsigned w = prs[min(u, nu - 1) * NPT + pt];
        return u < nu && ul < MAC_KB * 4 * UPG ? make_int2(w & 0xffff, w >> 16) : make_int2(4, 4);
    };
    v4f sp[NT][NH / 2], sc[NT][NH / 2];           // small-FFT values of the plain and conjugated use, all residues
    float2 ps;                                    // flip factor of lane < 5 NH
    v4f smx[FLF_SMAX_WAYS / 4];                   // largest small-FFT components of the entry's frame
    auto fetch = [&](int p, int b) {
        const char* sb = reinterpret_cast<const char*>(a.S + p * a.S_pstride + (long long)t0 * a.S_tstride +
                                                       (long long)cidx * NN * NH);
        const Entry en = entry();
        const int fc = min(en.f, nf - 1);
        const unsigned fo = (unsigned)(fc * a.S_tstride * 8);
        ps = a.psi[((long long)cidx * a.nP + p) * 5 * NH + min(lane, 5 * NH - 1)];
        const v4f* sm = reinterpret_cast<const v4f*>(a.smax + ((long long)p * a.smax_pstride + t0 + fc) * FLF_SMAX_WAYS);
#pragma unroll
        for (int i = 0; i < FLF_SMAX_WAYS / 4; ++i) smx[i] = sm[i];
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int2 pr = use_of(b, en.u + k * ESTEP, en.pt);
            const v4f* x = reinterpret_cast<const v4f*>(sb + (fo + (unsigned)(pr.x & ~7) * NH));
            const v4f* y = reinterpret_cast<const v4f*>(sb + (fo + (unsigned)(pr.y & ~7) * NH));
#pragma unroll
            for (int r = 0; r < NH / 2; ++r) {
                sp[k][r] = x[r];
                sc[k][r] = y[r];
            }
        }
    };
    // The thread's entries of the table of stage st (a plane of parity par).
    // The frame's scale brings the largest small-FFT component of the plane
    // into [2^13, 2^14): P and M components, at most 2^1.5 times as large,
    // stay within fp16, and values down to 2^-17 of the largest keep all 23
    // bits of the split.
    auto convert = [&](int b, int st, int par) {
        const Entry en = entry();
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < FLF_SMAX_WAYS / 4; ++i) m = fmaxf(fmaxf(m, fmaxf(smx[i][0], smx[i][1])), fmaxf(smx[i][2], smx[i][3]));
        const int e = scale_exp(m, 13);
        const float s = exp2_int(e);
        if (tid < NPT * FB && en.pt == 0) inv[par * FB + en.f] = exp2_int(-e);
        if (lane < 5 * NH) psi[lane] = ps;
        wave_sync();
        // dword (residue, unit, column, pair type) of the table's halves
        unsigned* hi = reinterpret_cast<unsigned*>(T + st * (2 * M::TAB * 16));
        unsigned* lo = hi + 4 * M::TAB;
#pragma unroll
        for (int k = 0; k < NT; ++k) {
            const int ul = en.u + k * ESTEP;
            if ((NT * ESTEP == MAC_KB * 4 * UPG || ul < MAC_KB * 4 * UPG) && en.f < nf) {
                const int2 pr = use_of(b, ul, en.pt);
                const int d0 = ((ul / UPG) * M::COLS + 2 * en.f) * 4 + (SLOTS == 4 ? en.pt : 2 * (ul & 1) + en.pt);
#pragma unroll
                for (int r = 0; r < NH; ++r) {
                    const v4f vp = sp[k][r / 2], vc = sc[k][r / 2];
                    const float2 x = cmul(r & 1 ? make_float2(vp.z, vp.w) : make_float2(vp.x, vp.y), psi[5 * r + (pr.x & 7)]);
                    const float2 y = cmul(r & 1 ? make_float2(vc.z, vc.w) : make_float2(vc.x, vc.y), psi[5 * r + (pr.y & 7)]);
                    const float2 P = cadd(x, y);
                    const float2 d = csub(x, y);                               // M = i d = (-d.y, d.x)
                    const float p0 = P.x * s, p1 = P.y * s, m0 = -d.y * s, m1 = d.x * s;
                    const int o = r * (4 * M::RS) + d0;
                    hi[o] = pack_half2(p0, m0);
                    hi[o + 4] = pack_half2(p1, m1);
                    lo[o] = pack_half2(half_rest(p0), half_rest(m0));
                    lo[o + 4] = pack_half2(half_rest(p1), half_rest(m1));
                }
            }
            __builtin_amdgcn_sched_barrier(0);    // one entry's values live at a time
        }
    };

    v4f tot[2][NF], acc[2][NF];
#pragma unroll
    for (int rt = 0; rt < 2; ++rt)
#pragma unroll
        for (int t = 0; t < NF; ++t) tot[rt][t] = acc[rt][t] = v4f{0.f, 0.f, 0.f, 0.f};

    // Store v[rt][t] (component c of frame f, slot jj + NS t) at A + slice *
    // A_pstride.  The accumulators lie chunk by chunk, a chunk's bins by
    // column (GridTables::wpos), the block's frames interleaved: a workgroup
    // writes one contiguous run, which L2 holds together.  (In the natural
    // order of the grid a chunk's bins lie rX columns apart; the neighbours
    // of an 8-byte bin came from other workgroups, after L2 had evicted its
    // line: 49 million write requests per 1455^2 x 41-plane back projection
    // where 7 million lines hold the data.)  Of a lane pair (re, im) the even
    // lane writes row r's bin and the odd lane row r + 1's.  The positions come
    // from LDS: a load from memory here would wait for every A operand in
    // flight, which under load takes as long as a plane.
    auto store = [&](const v4f (&v)[2][NF], int slice) {
        // uniform base, 32-bit lane offsets
        char* A = reinterpret_cast<char*>(a.A + (long long)t0 * a.A_tstride + (long long)slice * a.A_pstride +
                                          item_base * SLOTS * nf);
        const unsigned fo = 8 * f, bs = 8 * nf;
        int z = 0;
        asm volatile("" : "+v"(z));               // (the rows' addresses are not kept across the plane loop)
        const int k4 = 4 * kq + c + z;
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int i = 16 * rt + k4 + 2 * h;
                const unsigned short* ws = reinterpret_cast<const unsigned short*>(wpos + start + min(i, count - 1)) + jj;
                const bool in = active && f < nf && i < count;
#pragma unroll
                for (int t = 0; t < NF; ++t) {
                    const unsigned w = ws[NS * t];
                    const float got = lane_xor1(c ? v[rt][t][2 * h] : v[rt][t][2 * h + 1]);
                    const float2 o = c ? make_float2(got, v[rt][t][2 * h + 1]) : make_float2(v[rt][t][2 * h], got);
                    if (in && w != 0xffff) *reinterpret_cast<float2*>(A + (fo + bs * w)) = o;
                }
                __builtin_amdgcn_sched_barrier(0);        // one row pair's addresses live at a time
            }
    };

    // Products of one K step: the B operand of slot j is its residue's unit with
    // the dwords (pair types) in the order i XOR j.
    auto products = [&](const v4u (&q)[4], const char* tk) {
#pragma unroll
        for (int t = 0; t < NF; ++t) {
            v4u b[2];
            b[0] = *reinterpret_cast<const v4u*>(tk + tb[t]);
            b[1] = *reinterpret_cast<const v4u*>(tk + tb[t] + M::TAB * 16);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                v4u d = b[h];
                if constexpr (SLOTS == 4) {
                    d[0] ^= mlo[t];
                    d[1] ^= mlo[t];
                    d[2] ^= mhi[t];
                    d[3] ^= mhi[t];
                } else {
#pragma unroll
                    for (int i = 0; i < 4; ++i) d[i] ^= mlo[t];
                }
                if constexpr (NS == 1) {
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[h][i] = d[i ^ t];
                } else {
                    const bool odd = jj & 1;      // bit 0 of the slot by lane, bit 1 by lane (NS = 4) or operand
                    v4u e;
#pragma unroll
                    for (int i = 0; i < 4; ++i) e[i] = odd ? d[i ^ 1] : d[i];
#pragma unroll
                    for (int i = 0; i < 4; ++i) b[h][i] = NS == 4 ? (jj & 2 ? e[i ^ 2] : e[i]) : e[i ^ (2 * t)];
                }
            }
            // hi*hi into the accumulators; the small products lo*hi + hi*lo +
            // lo*lo on their own first, one fp32 addition for all of them
            const v4f zero = v4f{0.f, 0.f, 0.f, 0.f};
            v4f x0 = mfma_f16(q[1], b[0], zero), x1 = mfma_f16(q[3], b[0], zero);
            acc[0][t] = mfma_f16(q[0], b[0], acc[0][t]);
            acc[1][t] = mfma_f16(q[2], b[0], acc[1][t]);
            x0 = mfma_f16(q[0], b[1], x0);
            x1 = mfma_f16(q[2], b[1], x1);
            x0 = mfma_f16(q[1], b[1], x0);
            x1 = mfma_f16(q[3], b[1], x1);
            acc[0][t] += x0;
            acc[1][t] += x1;
        }
    };

    int p = next_plane(pb);
    if (p >= pe && PER_PLANE) return;
    v4u ring[MAC_RING][4];
    if (p < pe)
#pragma unroll
        for (int d = 0; d < MAC_RING; ++d) load_a(ring[d], p, d);
    if (tid < n_items) wpos[tid] = a.wpos[item_base + tid];
    for (int i = tid; i < nu * NPT; i += MAC_THREADS) {
        const int2 w = a.pairs[i];
        prs[i] = (unsigned)w.x | (unsigned)w.y << 16;
    }
    __syncthreads();
    if (p >= pe) {                                // no plane enabled: a sum of zeros
        store(tot, range);
        return;
    }
    fetch(p, 0);
    convert(0, 0, 0);

    float2* Ew = Es + wv * FLF_TILE * SLOTS;      // this wave's output factors
    int b = 0, st = 0, par = 0;
    while (true) {
        // Every wave's part of this stage's table is written, and every wave is
        // done with the previous stage's, which convert() below overwrites.
        __syncthreads();
        const bool lastb = b + 1 == nbatch;
        const int pa = next_plane(p + 1);
        const int pl = pa < pe ? pa : p;          // plane of the loads past this one's last step
        const int pn = lastb ? pa : p, bn = lastb ? 0 : b + 1;
        const bool more = pn < pe;
        // The next stage's small-FFT values and this plane's output factors are
        // in flight during this stage's products.  No branch surrounds a load
        // here (past the last stage they load something in bounds, unused), so
        // that the compiler's waits leave the newer loads in flight.
        fetch(more ? pn : p, bn);
        const v4u ev = reinterpret_cast<const v4u*>(a.E + (item_base * a.nP + (long long)p * n_items + start) *
                                                              SLOTS)[min(lane, count * SLOTS / 2 - 1)];
        const int kse = min((b + 1) * MAC_KB, nks);
        const char* tk = T + st * (2 * M::TAB * 16);
        int k0 = b * MAC_KB;
        do {                                      // (at least one turn: no path around the loads)
#pragma unroll
            for (int d = 0; d < MAC_RING; ++d) {
                // step ks uses slot ks % MAC_RING; past the last step the slots
                // take the next plane's first steps
                const int ks = k0 + d;
                products(ring[d], tk + d * (4 * M::COLS * 16));
                const bool in = ks + MAC_RING < nks;
                load_a(ring[d], in ? p : pl, in ? ks + MAC_RING : d);
                if constexpr (M::WAVES == 4) __builtin_amdgcn_sched_barrier(0);   // one step's operands live at a time
            }
            k0 += MAC_RING;
            tk += MAC_RING * 4 * M::COLS * 16;
        } while (k0 < kse);
        // Epilogue of the plane.  Lane l holds D[item 4 (l / 16) + r][column
        // l % 16]; the other component of its frame is in lane l ^ 1.
        if (lastb) {
            if (lane < FLF_TILE * SLOTS / 2) reinterpret_cast<v4u*>(Ew)[lane] = ev;
            wave_sync();
            int z = 0;
            asm volatile("" : "+v"(z));           // (the rows' addresses are not kept across the plane loop)
            const float is = inv[par * FB + min(f, nf - 1)];
            float q1[NF], q2[NF];
#pragma unroll
            for (int t = 0; t < NF; ++t) {
                const float sg = cj[t] ? -1.f : 1.f;
                q1[t] = c ? sg * is : is;         // times own component x factor.x
                q2[t] = c ? is : -sg * is;        // times other component x factor.y
            }
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int i = min(16 * rt + 4 * kq + r + z, count - 1);
#pragma unroll
                    for (int t = 0; t < NF; ++t) {
                        const float2 e = Ew[i * SLOTS + jj + NS * t];
                        const float mine = acc[rt][t][r];
                        const float other = lane_xor1(mine);
                        const float v = fmaf(q1[t], mine * e.x, q2[t] * (other * e.y));
                        if constexpr (PER_PLANE) acc[rt][t][r] = v;
                        else tot[rt][t][r] += v;
                    }
                    __builtin_amdgcn_sched_barrier(0);    // one row's factors live at a time
                }
            if constexpr (PER_PLANE) store(acc, p);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt)
#pragma unroll
                for (int t = 0; t < NF; ++t) acc[rt][t] = v4f{0.f, 0.f, 0.f, 0.f};
        }
        if (!more) break;
        par = lastb ? par ^ 1 : par;
        st ^= 1;
        convert(bn, st, par);
        p = pn;
        b = bn;
    }
    if constexpr (!PER_PLANE) store(tot, range);
}

// Block id w in [0, R * nfb) -> frame block and the rest r in [0, R):
// frame blocks in super-blocks of S (the last one possibly shorter), and
// within a super-block the frame block fastest.  S = nfb: all frame blocks of
// an r consecutive; S = 1: frame block slowest.
__device__ __forceinline__ void split_frames(int w, int R, int nfb, int S, int& fblock, int& r) {
    S = (S <= 0 || S > nfb) ? nfb : S;
    const int sb = w / (S * R);
    const int sc = min(S, nfb - sb * S);
    const int rem = w - sb * S * R;
    fblock = sb * S + rem % sc;
    r = rem / sc;
}

template <int SLOTS, int NS, bool PER_PLANE>
__global__ __launch_bounds__(MAC_THREADS) __attribute__((amdgpu_waves_per_eu(MacShape<SLOTS, NS>::WAVES)))
void k_mac(MacArgs a) {
    // grid x = chunk x frame block, frame blocks of a chunk consecutive (in
    // super-blocks of a.fgroup): after the XCD remap they share one XCD's L2
    // for the spectra they all read
    constexpr int FB = MacShape<SLOTS, NS>::FB;
    const int nfb = (a.T + FB - 1) / FB;
    const int w = xcd_block(blockIdx.x, gridDim.x);
    int fblock, cidx;
    split_frames(w, gridDim.x / nfb, nfb, a.fgroup, fblock, cidx);
    mac_body<SLOTS, NS, PER_PLANE>(a, cidx, blockIdx.y, gridDim.y, fblock);
}

// All active grid groups of one projection: grid x flattened over (group,
// plane range, chunk, frame block), frame block fastest.  Each group's range
// starts at a multiple of 8 (padded with idle workgroups), and the XCD remap
// applies within the group: every XCD then takes an eighth of every group,
// whose workgroups cost about the same, where one remap over the whole grid
// would give some XCDs only a cheap group's workgroups and leave them idle
// early.  After the remap the frame blocks of one (chunk, plane range) are
// consecutive ids of one XCD, dispatched together: they read the same
// stored spectra at about the same time, which the XCD's L2 then serves
// once from HBM for all of them.  fgroup < nfb dispatches them in
// super-blocks of fgroup instead, so that more chunks run side by side
// (their scattered accumulator stores then combine in L2 more often).
template <int SLOTS, int NS, bool PER_PLANE>
__global__ __launch_bounds__(MAC_THREADS) __attribute__((amdgpu_waves_per_eu(MacShape<SLOTS, NS>::WAVES)))
void k_mac_grouped(MacGrouped ga) {
    const GroupPick p = pick_group(ga.gg, blockIdx.x);
    const int w = xcd_block(p.rem, p.n);
    const int R = p.nch * p.nr;
    if (w >= R * ga.nfb) return;                  // padding
    int fblock, r;
    split_frames(w, R, ga.nfb, ga.a[p.g].fgroup, fblock, r);
    mac_body<SLOTS, NS, PER_PLANE>(ga.a[p.g], r % p.nch, r / p.nch, p.nr, fblock);
}

// ---------------------------------------------------------------------------
// Inverse transform, stage 1: column inverse FFTs (length fY) of the half
// plane, keeping output rows y < Yout.  The input is the sum of nsum partial
// accumulators A_sstride apart (the forward projection's plane ranges), in
// the MAC's order: bin (k0, k1) of frame f at A[colidx * nf + f], where the
// bins of one orbit that fall on one column are consecutive.  A column is
// read in the order k0 = y0 + m rY, m fastest (colidx is laid out in it), so
// that neighbouring lanes read neighbouring bins.  The output holds rows
// [y][k1][frame of the block].
// A workgroup takes CB columns: CB / nf columns k1 of nf frames, or CB of the
// nf frames of one column.  grid (column blocks, planes x frame blocks),
// COL_LANES lanes per column; LDS CB*fY + fY (twiddles).
// ---------------------------------------------------------------------------
struct ColBlocks {
    int fc, kc, nfg;                 // frames and columns per workgroup, frame groups
    __host__ __device__ ColBlocks(int nf, int CB)
        : fc(nf < CB ? nf : CB), kc(nf < CB ? CB / nf : 1), nfg((nf + fc - 1) / fc) {}
    __host__ __device__ int count(int rfX) const { return (rfX + kc - 1) / kc * nfg; }
};
// Lanes per column: two waves (registers for half the butterflies each), one
// where the transform runs out of place.  Bound: the LDS passes' latency.  The
// columns of a workgroup fill LDS, so waves in flight come from the lanes per
// column and overlap of one workgroup's loads with another's passes from two
// workgroups per CU: 4 columns of 2 waves (the plan's default) against 8 of
// one took 8 frames of 1455^2 x 41 planes from 4.62 to 2.85 ms (6.8 GB; 4
// columns of one wave 3.40, 8 of two 4.04), one frame 603 -> 388 us.  XCD
// neighbours share the 128-byte lines that 4 columns or frames split.
template <bool BIG>
constexpr int COL_LANES = BIG ? 64 : 128;
template <bool PRIME, bool BIG>
__device__ __forceinline__ void ifft_cols_body(const IfftColArgs& a, int colblk, int batch) {
    extern __shared__ float2 lds[];
    const int fY = a.rpY.L, CB = a.CB;
    const int nfb = (a.T + a.FB - 1) / a.FB;
    const int plane = batch / nfb, t0 = (batch - plane * nfb) * a.FB;
    const int nf = min(a.FB, a.T - t0);
    const ColBlocks cb(nf, CB);
    const int f0 = colblk % cb.nfg * cb.fc, k10 = colblk / cb.nfg * cb.kc;
    if (k10 >= a.rfX) return;                           // (a block of fewer frames has fewer column blocks)
    const int fn = min(cb.fc, nf - f0);
    const int ncol = fn * min(cb.kc, a.rfX - k10);
    const int cs = ifft_col_stride(fY, CB);
    float2* C = lds;                 // [CB][cs], column kk * fn + frame
    float2* C2 = C + CB * cs;        // BIG: [CB][cs], the second buffer of the out-of-place passes
    float2* tw = BIG ? C2 + CB * cs : C2;   // [fY]
    const float2* in = a.A + ((long long)plane * a.T + t0) * a.A_bstride + f0;
    const int* idx = a.colidx + (long long)k10 * fY;
    for (int i = threadIdx.x; i < fY; i += blockDim.x) tw[i] = a.twY[i];
    // Thread -> frame fl and every nslot-th of the columns' entries (kk, y0, m),
    // stepped without divisions.
    const int tid = threadIdx.x, nslot = blockDim.x / fn;
    const int slot = tid / fn, fl = tid - slot * fn;
    if (slot < nslot) {
        constexpr int B = 8;                    // loads in flight per thread
        const int N = a.N, rY = a.rY, Q = fY * (ncol / fn);
        const int sm = nslot % N, sy = nslot / N % rY, sk = nslot / N / rY;
        int m = slot % N, y0 = slot / N % rY, kk = slot / N / rY;
        for (int q0 = slot; q0 < Q; q0 += nslot * B) {
            float2 v[B];
            int src[B];
#pragma unroll
            for (int u = 0; u < B; ++u) src[u] = idx[min(q0 + u * nslot, Q - 1)] * nf + fl;
#pragma unroll
            for (int u = 0; u < B; ++u) v[u] = in[src[u]];
            for (int q = 1; q < a.nsum; ++q) {     // partial accumulators, fixed order
#pragma unroll
                for (int u = 0; u < B; ++u) v[u] = cadd(v[u], in[src[u] + q * a.A_sstride]);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (q0 + u * nslot < Q) C[(kk * fn + fl) * cs + y0 + m * rY] = v[u];
                m += sm;
                y0 += sy;
                kk += sk;
                if (m >= N) { m -= N; ++y0; }
                if (y0 >= rY) { y0 -= rY; ++kk; }
            }
        }
    }
    __syncthreads();
    constexpr int NT = COL_LANES<BIG>;
    const int lane = tid & (NT - 1), col = tid / NT;
    if constexpr (BIG) {
        if (col < ncol) wave_fft_pp<PRIME>(C + col * cs, C2 + col * cs, a.rpY, tw, true, lane);
        __syncthreads();
    } else {
        wave_fft<2048, PRIME, NT>(C + col * cs, 1, a.rpY, tw, true, lane);   // (columns past ncol: not stored)
    }
    const float2* Res = (BIG && (a.rpY.n & 1)) ? C2 : C;   // after an odd pass count: the second buffer
    float2* out = a.out + ((long long)plane * a.T + t0) * a.out_bstride + (long long)k10 * nf + f0;
    const int rowst = a.rfX * nf;
    const int cc = tid % CB;                    // blockDim = NT * CB: fixed column, every NT-th row
    if (cc < ncol) {
        const int kk = cc / fn;
        const float2* R = Res + cc * cs;
        out += kk * nf + cc - kk * fn;
        for (int y = tid / CB; y < a.Yout; y += NT) out[(long long)y * rowst] = R[y];
    }
}
template <bool PRIME, bool BIG>
__global__ __launch_bounds__(8 * COL_LANES<BIG>) void k_ifft_cols(IfftColArgs a) {
    ifft_cols_body<PRIME, BIG>(a, xcd_block(blockIdx.x, gridDim.x), blockIdx.y);
}
// All active grid groups: grid x flattened over (group, batch, column
// block), nchunks[g] = column blocks of group g; one CB for every group.
template <bool PRIME>
__global__ __launch_bounds__(8 * COL_LANES<false>) void k_ifft_cols_grouped(IfftColGrouped ga) {
    const GroupPick p = pick_group(ga.gg, blockIdx.x);
    const int b = xcd_block(p.rem, p.n);
    ifft_cols_body<PRIME, false>(ga.a[p.g], b % p.nch, b / p.nch);
}

// c2r of one row by NT lanes (one wave, or a workgroup).  row: rfX = L/2+1 half-spectrum values rs apart (global);
// buf: LDS work area (L/2 entries for even L, L for odd L; BIG, for L above
// 2048: buf2 is a second such area for the out-of-place passes).  For even L the
// length-L/2 complex transform of Z[k] = E[k] + i O[k],
//   E = X[k] + conj(X[L/2-k]),  O = (X[k] - conj(X[L/2-k])) exp(+2 pi i k/L),
// gives x[2m] = Re z[m], x[2m+1] = Im z[m]; odd L uses the Hermitian
// extension and a full-length transform.  The imaginary parts of X[0] and
// X[L/2] are dropped, as a c2r transform does.  Returns with the result in
// buf (interleaved real samples for even L, real parts for odd L).
template <bool PRIME, bool BIG, bool ODD, int NT = 64>
__device__ __forceinline__ float2* wave_c2r(float2* buf, float2* buf2, const float2* __restrict__ row, int L,
                                            const RadixPlan& rph, const float2* twh,
                                            const RadixPlan& rpf, const float2* twf, int lane, int rs) {
    // Loads are issued C2R_BATCH per lane at a time, so that their latencies
    // overlap instead of adding up.
    constexpr int B = NT == 64 ? 8 : 4, LE = NT == 64 ? 1024 : 2048;   // (LE: longest half-length transform)
    if (!ODD || (L & 1) == 0) {
        const int L2 = L / 2;
        for (int k0 = lane; k0 < L2; k0 += NT * B) {
            float2 xs[B], xrs[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int k = k0 + NT * u;
                if (k < L2) {
                    xs[u] = row[k * rs];
                    xrs[u] = row[(L2 - k) * rs];
                }
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int k = k0 + NT * u;
                if (k < L2) {
                    float2 x = xs[u];
                    float2 xr = cconj(xrs[u]);
                    if (k == 0) { x.y = 0.f; xr.y = 0.f; }
                    const float2 E = cadd(x, xr);
                    const float2 d = csub(x, xr);
                    const float2 w = cconj(twf[k]);          // exp(+2 pi i k / L)
                    const float2 O = cmul(d, w);
                    buf[k] = make_float2(E.x - O.y, E.y + O.x);  // E + i O
                }
            }
        }
        seq_sync<NT>();
        if constexpr (BIG) return wave_fft_pp<PRIME>(buf, buf2, rph, twh, true, lane);
        wave_fft<LE, PRIME, NT>(buf, 1, rph, twh, true, lane);
        return buf;
    } else {
        const int rfX = L / 2 + 1;
        for (int k0 = lane; k0 < L; k0 += NT * B) {
            float2 vs[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int k = k0 + NT * u;
                if (k < L) vs[u] = k < rfX ? row[k * rs] : cconj(row[(L - k) * rs]);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int k = k0 + NT * u;
                if (k < L) {
                    float2 v = vs[u];
                    if (k == 0) v.y = 0.f;
                    buf[k] = v;
                }
            }
        }
        seq_sync<NT>();
        if constexpr (BIG) return wave_fft_pp<PRIME>(buf, buf2, rpf, twf, true, lane);
        wave_fft<2 * LE, PRIME, NT>(buf, 1, rpf, twf, true, lane);
        return buf;
    }
}

// The same transform of a row that lies in buf already (rfX values, natural
// order), in place: a lane takes both values of a pair (k, L/2 - k), whose
// results E + i O and conj(E) + i conj(O) replace them.  twd: the length-L
// table for the pre-twiddle (global memory, even L); tab: the table of the
// transform itself (LDS).
template <bool PRIME, bool ODD>
__device__ __forceinline__ void wave_c2r_in_place(float2* buf, int L, const RadixPlan& rph, const RadixPlan& rpf,
                                                  const float2* __restrict__ twd, const float2* tab, int lane) {
    if (!ODD || (L & 1) == 0) {
        const int L2 = L / 2;
        for (int k = lane; 2 * k <= L2; k += 64) {
            float2 x = buf[k], xr = cconj(buf[L2 - k]);
            if (k == 0) { x.y = 0.f; xr.y = 0.f; }
            const float2 E = cadd(x, xr), O = cmul(csub(x, xr), cconj(twd[k]));
            buf[k] = make_float2(E.x - O.y, E.y + O.x);                        // E + i O
            if (2 * k < L2 && k > 0) buf[L2 - k] = make_float2(E.x + O.y, O.x - E.y);   // conj(E) + i conj(O)
        }
        wave_sync();
        wave_fft<1024, PRIME>(buf, 1, rph, tab, true, lane);
    } else {
        for (int k = lane; 2 * k < L; k += 64) {
            if (k == 0) buf[0].y = 0.f;
            else buf[L - k] = cconj(buf[k]);
        }
        wave_sync();
        wave_fft<2048, PRIME>(buf, 1, rpf, tab, true, lane);
    }
}

__device__ __forceinline__ float c2r_sample(const float2* buf, int L, int x) {
    if ((L & 1) == 0) {
        const float2 v = buf[x >> 1];
        return (x & 1) ? v.y : v.x;
    }
    return buf[x].x;
}

// Rows per workgroup of the row transforms that read rows from memory directly
// (one frame, or rows longer than 2048; one wave each).
constexpr int ROWS_PER_WG = 4;
// Wave w of frame block tb (8 frames) -> output row and frame, frames fastest.
struct RowFrame {
    int y, t;
};
__device__ __forceinline__ RowFrame row_frame(int w, int tb, int T) {
    const int n = min(8, T - 8 * tb), y = w / n;
    return {y, 8 * tb + w - y * n};
}

// Several frames: rows staged through LDS.  The frames of a block lie
// interleaved, so a wave that reads its own row takes 8 of every 8 n bytes
// (n frames) and each of its loads touches 64 lines.  Here a workgroup of
// ROW_WAVES waves takes ROW_WAVES / n rows of the n frames of a block, one
// contiguous run of memory, and spreads it over the waves' LDS buffers.
// Bound: memory and the passes' latency.  8 frames of 1455^2 x 41 planes, stored
// (6 GB) / with the update (11.6 GB): 3.55 / 6.65 -> 2.29 / 3.08 ms (2.42 / 4.52
// from rows apart, as one frame has them; that order costs the column
// transform its runs).  Even lengths alone: 75 registers instead of 127 (odd
// lengths take full-length transforms), 6 waves per SIMD instead of 4.
constexpr int ROW_WAVES = 8;
struct RowSet {
    int t0, n, y0, rows;          // frames t0 .. t0 + n - 1, rows y0 .. y0 + rows - 1
};
__device__ __forceinline__ RowSet row_set(int blk, int tb, int T, int Y) {
    RowSet r;
    r.t0 = 8 * tb;
    r.n = min(8, T - r.t0);
    const int R = ROW_WAVES / r.n;
    r.y0 = blk * R;
    r.rows = min(R, Y - r.y0);    // <= 0: past the end (a block of fewer frames has fewer workgroups)
    return r;
}
// Buffer stride (float2): the values of one k and the n frames fall on
// distinct banks, with the 32 / n neighbours that a half wave writes along.
__host__ __device__ inline int row_stage_stride(int wbuf, int n) {
    const int want = 32 / n % 32, len = wbuf + 1;
    return len + ((want - len) % 32 + 32) % 32;
}
// src: the run's first value; element q = ((row, k), frame) goes to the buffer
// of wave row * n + frame, entry k.
__device__ __forceinline__ void stage_rows(float2* buf, int bs, const float2* __restrict__ src, const RowSet& r, int rfX) {
    constexpr int B = 8;                        // loads in flight per thread
    const int total = r.rows * rfX * r.n;
    const float rn = 1.0f / (float)r.n, rrf = 1.0f / (float)rfX;
    for (int i0 = threadIdx.x; i0 < total; i0 += (int)blockDim.x * B) {
        float2 v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = src[min(i0 + u * (int)blockDim.x, total - 1)];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int i = i0 + u * (int)blockDim.x;
            int f, k;
            const int row = div_small(div_small(i, r.n, rn, f), rfX, rrf, k);
            if (i < total) buf[(row * r.n + f) * bs + k] = v[u];
        }
    }
}
__device__ __forceinline__ void stage_table(float2* tab, int L, const float2* __restrict__ twh, const float2* __restrict__ twf) {
    const int n = (L & 1) ? L : L / 2;
    const float2* t = (L & 1) ? twf : twh;
    for (int i = threadIdx.x; i < n; i += blockDim.x) tab[i] = t[i];
}

template <int XPL, int NT>
__device__ __forceinline__ void store_row_sum(const IfftRowSumArgs& a, const float* acc, int y, int t, int lane) {
    const int Yv = a.fdims ? a.fdims[t].x : a.Y, Xv = a.fdims ? a.fdims[t].y : a.X;
    const long long ro = (long long)t * a.img_tstride + (long long)y * a.X;
    if (a.img) {
#pragma unroll
        for (int q = 0; q < XPL; ++q) {
            const int x = lane + NT * q;
            if (x < a.X) a.img[ro + x] = (y < Yv && x < Xv) ? acc[q] : 0.f;
        }
    }
    if (a.ratio) {
        // standard RL's error image im / HX (lfdeconv.py:191) with IEEE
        // division: 0/0 gives NaN and x/0 inf, as in numpy
#pragma unroll
        for (int q = 0; q < XPL; ++q) {
            const int x = lane + NT * q;
            if (x < a.X) a.ratio[ro + x] = (y < Yv && x < Xv) ? a.im[ro + x] / acc[q] : 0.f;
        }
    }
}

// Forward projection, stage 2: per output row, c2r each grid group's row and
// sum the groups in a fixed order.  One workgroup of ROW_SUM_LANES per (row,
// frame), the frames of a block of 8 fastest (they are interleaved in memory);
// grid (Y * min(8, T), ceil(T / 8)).  Bound: latency (the groups follow each
// other, each a load, 3 or 4 passes and the samples), so a row gets 4 waves:
// one wave per row, 4 rows per workgroup, held 200 registers and left 300 rows
// on 75 CUs (300^2 x 11 planes 41 -> 30 us, 150^2 x 2 16.4 -> 10.9, 2048^2, rows
// longer than 2048 then out of place, 211 -> 72; 1455^2 67 either way; with a
// prime pass, whose few butterflies fill a third of the lanes, 103 -> 130 us at
// 1273 x 1463, Nnum 19, 0.2 % of a projection).
constexpr int ROW_SUM_LANES = 256;
template <bool PRIME, bool ODD>
__global__ __launch_bounds__(ROW_SUM_LANES) void k_ifft_rows_sum(IfftRowSumArgs a) {
    extern __shared__ float2 lds[];
    reset_smax(a.smax, a.nsmax);
    const int lane = threadIdx.x;
    const RowFrame rf = row_frame(blockIdx.x, blockIdx.y, a.T);
    const int y = rf.y, t = rf.t;
    if (y >= a.Y) return;                       // (a block of fewer frames has fewer workgroups)
    float2* twf = lds;                          // [maxfX]
    float2* twh = twf + a.maxfX;                // [maxfX/2 + 1]
    float2* buf = twh + a.maxfX / 2 + 1;        // [wbuf]
    constexpr int XPL = 4096 / ROW_SUM_LANES;   // output samples per lane (X <= 4096)
    float acc[XPL];
#pragma unroll
    for (int q = 0; q < XPL; ++q) acc[q] = 0.f;
    for (int g = 0; g < a.ngroups; ++g) {
        const IfftRowGroup& G = a.grp[g];
        if (!G.active) continue;
        const int L = G.rp.L;
        __syncthreads();
        for (int i = lane; i < L; i += ROW_SUM_LANES) twf[i] = G.twf[i];
        if ((L & 1) == 0)
            for (int i = lane; i < L / 2; i += ROW_SUM_LANES) twh[i] = G.twh[i];
        const int b0 = t / G.FB * G.FB, nf = min(G.FB, a.T - b0);
        const float2* row = G.T + (long long)b0 * G.tstride + (long long)y * G.rfX * nf + (t - b0);
        __syncthreads();
        wave_c2r<PRIME, false, ODD, ROW_SUM_LANES>(buf, nullptr, row, L, G.rph, twh, G.rp, twf, lane, nf);
        const float sc = G.scale;
#pragma unroll
        for (int q = 0; q < XPL; ++q) {
            const int x = lane + ROW_SUM_LANES * q;
            if (x < a.X) acc[q] += c2r_sample(buf, L, x) * sc;
        }
    }
    store_row_sum<XPL, ROW_SUM_LANES>(a, acc, y, t, lane);
}

// The same for several frames, rows staged through LDS (see stage_rows);
// grid (ceil(Y / (ROW_WAVES / n)), ceil(T / 8)), a wave per row and frame.
template <bool PRIME, bool ODD>
__global__ __launch_bounds__(64 * ROW_WAVES) void k_ifft_rows_sum_staged(IfftRowSumArgs a) {
    extern __shared__ float2 lds[];
    reset_smax(a.smax, a.nsmax);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const RowSet r = row_set(blockIdx.x, blockIdx.y, a.T, a.Y);
    if (r.rows <= 0) return;
    const int bs = row_stage_stride(a.wbuf, r.n);
    float2* tab = lds;                          // [wbuf]
    float2* bufs = lds + a.wbuf;                // [ROW_WAVES][bs]
    float2* buf = bufs + wv * bs;
    const int row = wv / r.n, y = r.y0 + row, t = r.t0 + wv - row * r.n;
    const bool busy = row < r.rows;
    constexpr int XPL = 2048 / 64;
    float acc[XPL];
#pragma unroll
    for (int q = 0; q < XPL; ++q) acc[q] = 0.f;
    for (int g = 0; g < a.ngroups; ++g) {
        const IfftRowGroup& G = a.grp[g];
        if (!G.active) continue;
        const int L = G.rp.L;
        __syncthreads();
        stage_table(tab, L, G.twh, G.twf);
        stage_rows(bufs, bs, G.T + (long long)r.t0 * G.tstride + (long long)r.y0 * G.rfX * r.n, r, G.rfX);
        __syncthreads();
        if (busy) {
            wave_c2r_in_place<PRIME, ODD>(buf, L, G.rph, G.rp, G.twf, tab, lane);
            const float sc = G.scale;
#pragma unroll
            for (int q = 0; q < XPL; ++q) {
                const int x = lane + 64 * q;
                if (x < a.X) acc[q] += c2r_sample(buf, L, x) * sc;
            }
        }
    }
    if (busy) store_row_sum<XPL, 64>(a, acc, y, t, lane);
}

// One row's samples to the volume: stored, or the Richardson-Lucy update.  Two
// samples per lane and step, as they lie in buf for even lengths (rows of an
// odd X start on 4-byte boundaries; 8-byte accesses need no more).
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));
__device__ __forceinline__ float rl_update(int mode, float v, float xo, float hd, bool trust) {
    if (mode == 0) return v;
    float xn;
    if (mode == 1) {
        xn = xo * (hd / v);
    } else {
        xn = xo * v;
        if (trust) xn = xn / hd;
    }
    return __builtin_isnan(xn) ? 0.f : xn;
}
__device__ __forceinline__ void update_row(const IfftRowPlaneArgs& a, const float2* buf, const RowPlaneDesc& pd, int z,
                                           int t, int y, int lane) {
    const int L = pd.rp.L, X2 = a.X / 2;
    const float sc = pd.scale;
    const long long o = (((long long)z * a.T + t) * a.Y + y) * a.X;
    const int Yv = a.fdims ? a.fdims[t].x : a.Y, Xv = a.fdims ? a.fdims[t].y : a.X;
    float* vol = a.vol + o;
    const bool tr = a.mode == 2 && a.trust;
    const float* hs = a.mode == 1 ? a.Htf + o : tr ? a.trust + ((long long)z * a.Y + y) * a.X : nullptr;
    constexpr int B = 4;                        // pairs in flight per lane
    for (int k0 = lane; k0 < X2; k0 += 64 * B) {
        f2u xo[B], hd[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int x = 2 * min(k0 + 64 * u, X2 - 1);
            xo[u] = a.mode != 0 ? *(const f2u*)(vol + x) : f2u{0.f, 0.f};
            hd[u] = hs ? *(const f2u*)(hs + x) : f2u{1.f, 1.f};
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int k = k0 + 64 * u, x = 2 * k;
            if (k < X2) {
                float2 v = (L & 1) ? make_float2(buf[x].x, buf[x + 1].x) : buf[k];
                f2u r;
                r.x = y < Yv && x < Xv ? rl_update(a.mode, v.x * sc, xo[u].x, hd[u].x, tr) : 0.f;
                r.y = y < Yv && x + 1 < Xv ? rl_update(a.mode, v.y * sc, xo[u].y, hd[u].y, tr) : 0.f;
                *(f2u*)(vol + x) = r;
            }
        }
    }
    if ((a.X & 1) && lane == 0) {
        const int x = a.X - 1;
        const float xo = a.mode != 0 ? vol[x] : 0.f, hd = hs ? hs[x] : 1.f;
        vol[x] = y < Yv && x < Xv ? rl_update(a.mode, c2r_sample(buf, L, x) * sc, xo, hd, tr) : 0.f;
    }
}

// Backward projection, stage 2: per (row, frame, plane) c2r; then either store
// the plane, or apply the Richardson-Lucy update in place
// (lfdeconv.py:112-126 Prevedel: X *= Htf / v;  lfdeconv.py:151-164 standard:
// X *= v [/ trust]; NaN -> 0 after the update).  One wave per (row, frame),
// the frames of a block of 8 fastest (they are interleaved in memory);
// grid (ceil(Y * min(8, T) / ROWS_PER_WG), ceil(T / 8), nplanes), block 64 * ROWS_PER_WG.  Twiddles of every grid group are
// read from global memory (they stay in the caches).
template <bool PRIME, bool BIG, bool ODD>
__global__ __launch_bounds__(64 * ROWS_PER_WG) void k_ifft_rows_plane(IfftRowPlaneArgs a) {
    extern __shared__ float2 lds[];
    reset_smax(a.smax, a.nsmax);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const RowFrame rf = row_frame(blockIdx.x * ROWS_PER_WG + wv, blockIdx.y, a.T);
    const int y = rf.y, t = rf.t;
    const int z = a.plane_ids[blockIdx.z];      // kernel argument (scalar load)
    const RowPlaneDesc& pd = a.pd[z];           // read in place (no private copy)
    const int L = pd.rp.L;
    float2* buf = lds + wv * (BIG ? 2 : 1) * a.wbuf;
    if (y >= a.Y) return;                       // no block-level barrier below
    const int FB = pd.slots == 4 ? a.FB4 : a.FB2;
    const int b0 = t / FB * FB, nf = min(FB, a.T - b0);
    const float2* row = a.Tbuf + pd.T_off + (long long)b0 * pd.T_tstride + (long long)y * pd.rfX * nf + (t - b0);
    const float2* res = wave_c2r<PRIME, BIG, ODD>(buf, buf + a.wbuf, row, L, pd.rph, pd.twh, pd.rp, pd.twf, lane, nf);
    update_row(a, res, pd, z, t, y, lane);
}

// The same for several frames, rows staged through LDS (see stage_rows);
// grid (ceil(Y / (ROW_WAVES / n)), ceil(T / 8), nplanes), a wave per row and frame.
template <bool PRIME, bool ODD>
__global__ __launch_bounds__(64 * ROW_WAVES) __attribute__((amdgpu_waves_per_eu(PRIME || ODD ? 4 : 6)))
void k_ifft_rows_plane_staged(IfftRowPlaneArgs a) {
    extern __shared__ float2 lds[];
    reset_smax(a.smax, a.nsmax);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const RowSet r = row_set(blockIdx.x, blockIdx.y, a.T, a.Y);
    if (r.rows <= 0) return;
    const int z = a.plane_ids[blockIdx.z];
    const RowPlaneDesc& pd = a.pd[z];
    const int L = pd.rp.L, bs = row_stage_stride(a.wbuf, r.n);
    float2* tab = lds;                          // [wbuf]
    float2* bufs = lds + a.wbuf;                // [ROW_WAVES][bs]
    stage_table(tab, L, pd.twh, pd.twf);
    stage_rows(bufs, bs, a.Tbuf + pd.T_off + (long long)r.t0 * pd.T_tstride + (long long)r.y0 * pd.rfX * r.n, r, pd.rfX);
    __syncthreads();
    const int row = wv / r.n;
    if (row >= r.rows) return;                  // no block-level barrier below
    float2* buf = bufs + wv * bs;
    wave_c2r_in_place<PRIME, ODD>(buf, L, pd.rph, pd.rp, pd.twf, tab, lane);
    update_row(a, buf, pd, z, r.t0 + wv - row * r.n, r.y0 + row, lane);
}

// ---------------------------------------------------------------------------
// Data-fit sums in FP64: per frame sum((img-im)^2) and sum(im^2).  Two stages
// with a fixed reduction order (deterministic).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_fit_partial(const float* img, const float* im, long long n_per_frame,
                                                     int im_frames, double* part, int nblk) {
    __shared__ double sd[256], si[256];
    const int t = blockIdx.y;
    const float* a = img + (long long)t * n_per_frame;
    const float* b = im + (long long)(t % im_frames) * n_per_frame;
    double d2 = 0.0, i2 = 0.0;
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n_per_frame;
         i += (long long)nblk * blockDim.x) {
        double d = (double)a[i] - (double)b[i];
        d2 += d * d;
        i2 += (double)b[i] * (double)b[i];
    }
    sd[threadIdx.x] = d2;
    si[threadIdx.x] = i2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) { sd[threadIdx.x] += sd[threadIdx.x + s]; si[threadIdx.x] += si[threadIdx.x + s]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[((long long)t * nblk + blockIdx.x) * 2 + 0] = sd[0];
        part[((long long)t * nblk + blockIdx.x) * 2 + 1] = si[0];
    }
}

__global__ __launch_bounds__(256) void k_fit_final(const double* part, int nblk, double* out) {
    __shared__ double sd[256], si[256];
    const int t = blockIdx.x;
    double d2 = 0.0, i2 = 0.0;
    for (int i = threadIdx.x; i < nblk; i += blockDim.x) {
        d2 += part[((long long)t * nblk + i) * 2 + 0];
        i2 += part[((long long)t * nblk + i) * 2 + 1];
    }
    sd[threadIdx.x] = d2;
    si[threadIdx.x] = i2;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) { sd[threadIdx.x] += sd[threadIdx.x + s]; si[threadIdx.x] += si[threadIdx.x + s]; }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[t * 2 + 0] = sd[0];
        out[t * 2 + 1] = si[0];
    }
}

// Prevedel update with a precomputed denominator (lfdeconv.py:112-126):
// X *= Htf / v, NaN -> 0, the same arithmetic as k_ifft_rows_plane mode 1.
// Used for the first plain iterate from a uniform start, X1 = Htf / Ht(H 1),
// whose denominator does not depend on the image (one slab per plane serves
// every frame: v_frames = 1).  ratio: X = Htf / v (the same update of X = 1,
// without reading X).  grid (x blocks, nz * T slabs), block RL_SCALE_THREADS;
// each thread takes RL_SCALE_E pixels RL_SCALE_THREADS apart, all loads in
// flight before the first use (indices clamped into the slab).
constexpr int RL_SCALE_THREADS = 256, RL_SCALE_E = 16;
__global__ __launch_bounds__(RL_SCALE_THREADS) void k_rl_scale(float* X, const float* Htf, const float* v, int T,
                                                               long long npix, int v_frames, int ratio) {
    const int slab = blockIdx.y;
    const int z = slab / T, t = slab - z * T;
    const long long o = (long long)slab * npix;
    const float* vs = v + ((long long)z * v_frames + (v_frames == 1 ? 0 : t)) * npix;
    constexpr long long CH = (long long)RL_SCALE_THREADS * RL_SCALE_E;
    for (long long b0 = (long long)blockIdx.x * CH + threadIdx.x; b0 < npix; b0 += (long long)gridDim.x * CH) {
        float h[RL_SCALE_E], d[RL_SCALE_E], x[RL_SCALE_E];
#pragma unroll
        for (int e = 0; e < RL_SCALE_E; ++e) {
            const long long i = min(b0 + (long long)e * RL_SCALE_THREADS, npix - 1);
            h[e] = Htf[o + i];
            d[e] = vs[i];
            x[e] = ratio ? 1.f : X[o + i];
        }
#pragma unroll
        for (int e = 0; e < RL_SCALE_E; ++e) {
            const long long i = b0 + (long long)e * RL_SCALE_THREADS;
            if (i < npix) {
                const float r = h[e] / d[e];
                const float xn = ratio ? r : x[e] * r;
                X[o + i] = __builtin_isnan(xn) ? 0.f : xn;
            }
        }
    }
}

// Fill with a constant (used instead of memset so that work stays capturable).
__global__ void k_fill(float* p, long long n, float v) {
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x)
        p[i] = v;
}

// ---------------------------------------------------------------------------
// Host-side launchers.
// ---------------------------------------------------------------------------
namespace flf {

// Whether a plan ends with an odd prime radix above 5 (7, 11, ..., 31; the
// kernels built with that pass are launched only then).  The other radices
// are 2..6, 8, 9, 10 and 12.
bool plan_has_prime(const RadixPlan& rp) {
    if (rp.n == 0) return false;
    const int r = rp.r[rp.n - 1];
    return r == 7 || r == 11 || r > 12;
}
static bool has_prime(const RadixPlan& rp) { return plan_has_prime(rp); }

size_t small_fft_lds(int rY, int rX) {
    return ((size_t)(rY + 1) * (rX / 2 + 1) + 2 * (size_t)(rY + rX) + 1) * sizeof(float2);
}
// Reduced grids above 128 points take the 256-point wave transforms, those up
// to 64 workgroups of 4 waves (a pass of a 64 x 64 grid has 256 butterflies; 8
// workgroups share a CU), the others 12 (a pass of 120 x 120 has 720, LDS holds
// 2 workgroups).
bool small_fft_big(int rY, int rX) { return rY > 128 || rX > 128; }
static SmallFFT small_fft_variant(int rY, int rX) {
    return small_fft_big(rY, rX) ? SFFT_256 : std::max(rY, rX) > 64 ? SFFT_128 : SFFT_64;
}
hipError_t launch_small_fft(const SmallFFTArgs& a, int nsrc, int T, hipStream_t s) {
    size_t lds = small_fft_lds(a.rpY.L, a.rpX.L);
    if (a.rpY.L > 256 || a.rpX.L > 256) return hipErrorInvalidValue;
    const dim3 grid(a.N * a.N, T, nsrc);
    switch (small_fft_variant(a.rpY.L, a.rpX.L)) {
        case SFFT_256: hipLaunchKernelGGL(k_small_fft<SFFT_256>, grid, dim3(64 * sfft_waves(SFFT_256)), lds, s, a); break;
        case SFFT_128: hipLaunchKernelGGL(k_small_fft<SFFT_128>, grid, dim3(64 * sfft_waves(SFFT_128)), lds, s, a); break;
        default: hipLaunchKernelGGL(k_small_fft<SFFT_64>, grid, dim3(64 * sfft_waves(SFFT_64)), lds, s, a);
    }
    return hipGetLastError();
}
hipError_t launch_small_fft_grouped(const SmallFFTGrouped& ga, int N, int T, size_t lds, hipStream_t s) {
    const GroupedGrid& gg = ga.gg;
    if (gg.ngroups < 1 || gg.ngroups > FLF_MAX_GROUPS) return hipErrorInvalidValue;
    SmallFFT v = SFFT_64;
    for (int g = 0; g < gg.ngroups; ++g) v = std::max(v, small_fft_variant(ga.a[g].rpY.L, ga.a[g].rpX.L));
    const dim3 grid(N * N, T, gg.start[gg.ngroups]);
    if (v == SFFT_256) return hipErrorInvalidValue;               // (not grouped)
    if (v == SFFT_128) hipLaunchKernelGGL(k_small_fft_grouped<SFFT_128>, grid, dim3(64 * sfft_waves(v)), lds, s, ga);
    else hipLaunchKernelGGL(k_small_fft_grouped<SFFT_64>, grid, dim3(64 * sfft_waves(v)), lds, s, ga);
    return hipGetLastError();
}
hipError_t launch_psf_rows(const PsfRowArgs& a, int nu, hipStream_t s) {
    size_t lds = (size_t)a.RB * a.rpX.L * sizeof(float2);
    if (has_prime(a.rpX)) hipLaunchKernelGGL(k_psf_rows<true>, dim3((a.s2 + a.RB - 1) / a.RB, nu), dim3(FFT_THREADS), lds, s, a);
    else hipLaunchKernelGGL(k_psf_rows<false>, dim3((a.s2 + a.RB - 1) / a.RB, nu), dim3(FFT_THREADS), lds, s, a);
    return hipGetLastError();
}
hipError_t launch_psf_cols(const PsfColArgs& a, int nu, hipStream_t s) {
    size_t lds = (size_t)a.CB * a.rpY.L * sizeof(float2);
    if (has_prime(a.rpY)) hipLaunchKernelGGL(k_psf_cols<true>, dim3((a.rfX + a.CB - 1) / a.CB, nu), dim3(FFT_THREADS), lds, s, a);
    else hipLaunchKernelGGL(k_psf_cols<false>, dim3((a.rfX + a.CB - 1) / a.CB, nu), dim3(FFT_THREADS), lds, s, a);
    return hipGetLastError();
}
size_t spec_pack_lds(int nu, int slots) {
    return (size_t)nu * PACK_ITEMS * slots * sizeof(float2) + 8 * PACK_ITEMS * sizeof(float);
}
hipError_t launch_spec_pack(const SpecPackArgs& a, int nchunks, hipStream_t s) {
    const size_t lds = spec_pack_lds(a.nu, a.slots);
    hipLaunchKernelGGL(k_spec_pack, dim3((FLF_CHUNK_MAX + PACK_ITEMS - 1) / PACK_ITEMS, nchunks), dim3(256), lds, s, a);
    return hipGetLastError();
}
// Slots per matrix instruction for T frames: as many as leave no column that
// these frames could fill empty (4 slots x 2 frames, 2 x 4, 1 x 8).
int mac_slots_shared(int slots, int T) { return T > 4 ? 1 : (T > 2 || slots == 2 ? 2 : 4); }
int mac_frames(int slots, int T) { return FLF_MAC_FB / mac_slots_shared(slots, T); }
template <class F>
static auto mac_variant(int slots, int ns, bool per_plane, F f) {
    using std::integral_constant;
    auto go = [&](auto s, auto n) {
        return per_plane ? f(s, n, std::true_type{}) : f(s, n, std::false_type{});
    };
    if (slots == 4) {
        if (ns == 4) return go(integral_constant<int, 4>{}, integral_constant<int, 4>{});
        if (ns == 2) return go(integral_constant<int, 4>{}, integral_constant<int, 2>{});
        return go(integral_constant<int, 4>{}, integral_constant<int, 1>{});
    }
    if (ns == 2) return go(integral_constant<int, 2>{}, integral_constant<int, 2>{});
    return go(integral_constant<int, 2>{}, integral_constant<int, 1>{});
}
size_t mac_lds(int slots, int T) {
    return mac_variant(slots, mac_slots_shared(slots, T), false, [](auto s, auto n, auto) { return MacShape<s.value, n.value>::LDS; });
}
static bool mac_args_ok(const MacArgs& a, int slots) {
    return (slots == 2 || slots == 4) && a.T >= 1 && a.kg == (slots == 4 ? a.nu : (a.nu + 1) / 2);
}
hipError_t launch_mac(const MacArgs& a, int slots, int nchunks, int nplanes_grid, hipStream_t s) {
    if (!mac_args_ok(a, slots)) return hipErrorInvalidValue;
    const int fb = mac_frames(slots, a.T);
    const dim3 grid(nchunks * ((a.T + fb - 1) / fb), nplanes_grid), block(MAC_THREADS);
    mac_variant(slots, mac_slots_shared(slots, a.T), a.per_plane != 0, [&](auto sl, auto ns, auto pp) {
        hipLaunchKernelGGL((k_mac<sl.value, ns.value, pp.value>), grid, block, (MacShape<sl.value, ns.value>::LDS), s, a);
    });
    return hipGetLastError();
}
hipError_t launch_mac_grouped(const MacGrouped& ga, int slots, hipStream_t s) {
    const GroupedGrid& gg = ga.gg;
    if (gg.ngroups < 1 || gg.ngroups > FLF_MAX_GROUPS) return hipErrorInvalidValue;
    const int T = ga.a[0].T, fb = mac_frames(slots, T);
    if (ga.nfb != (T + fb - 1) / fb) return hipErrorInvalidValue;
    for (int k = 0; k < gg.ngroups; ++k) {
        if (gg.start[k + 1] - gg.start[k] < gg.nchunks[k] * gg.nranges[k] * ga.nfb) return hipErrorInvalidValue;
        if (!mac_args_ok(ga.a[k], slots) || ga.a[k].per_plane != ga.a[0].per_plane || ga.a[k].T != T) return hipErrorInvalidValue;
    }
    const dim3 grid(gg.start[gg.ngroups]), block(MAC_THREADS);
    mac_variant(slots, mac_slots_shared(slots, T), ga.a[0].per_plane != 0, [&](auto sl, auto ns, auto pp) {
        hipLaunchKernelGGL((k_mac_grouped<sl.value, ns.value, pp.value>), grid, block, (MacShape<sl.value, ns.value>::LDS), s, ga);
    });
    return hipGetLastError();
}
// Transforms longer than 2048 points run out of place (two LDS buffers).
bool wave_big(int L) { return L > 2048; }
size_t ifft_cols_lds(int CB, int fY) {
    return ((size_t)CB * ifft_col_stride(fY, CB) * (wave_big(fY) ? 2 : 1) + fY) * sizeof(float2);
}
// Column blocks of a call: those of a full block of frames, or of the last one
// where fewer frames make more of them.
int ifft_col_blocks(const IfftColArgs& a) {
    int n = 0;
    for (int t0 = 0; t0 < a.T; t0 += a.FB) n = std::max(n, ColBlocks(std::min(a.FB, a.T - t0), a.CB).count(a.rfX));
    return n;
}
hipError_t launch_ifft_cols_grouped(const IfftColGrouped& ga, int CB, bool prime, size_t lds, hipStream_t s) {
    const GroupedGrid& gg = ga.gg;
    if (CB < 1 || CB > 8 || gg.ngroups < 1 || gg.ngroups > FLF_MAX_GROUPS) return hipErrorInvalidValue;
    if (prime) hipLaunchKernelGGL(k_ifft_cols_grouped<true>, dim3(gg.start[gg.ngroups]), dim3(COL_LANES<false> * CB), lds, s, ga);
    else hipLaunchKernelGGL(k_ifft_cols_grouped<false>, dim3(gg.start[gg.ngroups]), dim3(COL_LANES<false> * CB), lds, s, ga);
    return hipGetLastError();
}
hipError_t launch_ifft_cols(const IfftColArgs& a, int nbatch, hipStream_t s) {
    size_t lds = ifft_cols_lds(a.CB, a.rpY.L);
    const dim3 grid(ifft_col_blocks(a), nbatch), block((wave_big(a.rpY.L) ? COL_LANES<true> : COL_LANES<false>) * a.CB);
    const bool big = wave_big(a.rpY.L);
    if (has_prime(a.rpY)) {
        if (big) hipLaunchKernelGGL((k_ifft_cols<true, true>), grid, block, lds, s, a);
        else hipLaunchKernelGGL((k_ifft_cols<true, false>), grid, block, lds, s, a);
    } else {
        if (big) hipLaunchKernelGGL((k_ifft_cols<false, true>), grid, block, lds, s, a);
        else hipLaunchKernelGGL((k_ifft_cols<false, false>), grid, block, lds, s, a);
    }
    return hipGetLastError();
}
// Twiddles (full and half length) and one row.
static size_t row_sum_lds(int maxfX, int wbuf) { return ((size_t)maxfX + maxfX / 2 + 1 + wbuf) * sizeof(float2); }
static int row_blocks(int Y, int T, int rows) { return (Y * std::min(8, T) + rows - 1) / rows; }
// Staged rows: the transform's table and one buffer per wave (149 KB at most,
// rows of 2047).
static int row_stage_waves(int T) {
    int w = 0;
    for (int t0 = 0; t0 < T; t0 += 8) w = std::max(w, ROW_WAVES / std::min(8, T - t0) * std::min(8, T - t0));
    return w;
}
static size_t row_stage_lds(int wbuf, int T) {
    int bs = 0;
    for (int n : {std::min(8, T), T > 8 && T % 8 ? T % 8 : std::min(8, T)}) bs = std::max(bs, row_stage_stride(wbuf, n));
    return ((size_t)wbuf + (size_t)row_stage_waves(T) * bs) * sizeof(float2);
}
// Workgroups over the rows: a block of n frames takes ROW_WAVES / n rows each.
static int row_stage_blocks(int Y, int T) {
    const int R = ROW_WAVES / std::min(8, T);
    return (Y + R - 1) / R;
}
// Calls f with a flag as a compile-time constant.
template <class F>
static void with_bool(bool b, F f) {
    if (b) f(std::true_type{});
    else f(std::false_type{});
}
hipError_t launch_ifft_rows_sum(const IfftRowSumArgs& a, int Y, int T, hipStream_t s) {
    if (a.T != T) return hipErrorInvalidValue;
    bool prime = false, odd = false;
    for (int g = 0; g < a.ngroups; ++g) {
        if (!a.grp[g].active) continue;
        prime = prime || has_prime(a.grp[g].rp) || has_prime(a.grp[g].rph);
        odd = odd || (a.grp[g].rp.L & 1);
    }
    with_bool(prime, [&](auto P) {
        with_bool(odd, [&](auto O) {
            if (T > 1 && !wave_big(a.maxfX))
                hipLaunchKernelGGL((k_ifft_rows_sum_staged<P.value, O.value>), dim3(row_stage_blocks(Y, T), (T + 7) / 8),
                                   dim3(64 * row_stage_waves(T)), row_stage_lds(a.wbuf, T), s, a);
            else
                hipLaunchKernelGGL((k_ifft_rows_sum<P.value, O.value>), dim3(Y * std::min(8, T), (T + 7) / 8),
                                   dim3(ROW_SUM_LANES), row_sum_lds(a.maxfX, a.wbuf), s, a);
        });
    });
    return hipGetLastError();
}
// c2r of an even length runs as a half-length complex FFT in place.
int c2r_wave_buffer(int fX) { return (fX & 1) ? fX : fX / 2; }
size_t ifft_rows_plane_lds(int wbuf, bool big) { return ROWS_PER_WG * (size_t)wbuf * (big ? 2 : 1) * sizeof(float2); }
hipError_t launch_ifft_rows_plane(const IfftRowPlaneArgs& a, int nplanes, hipStream_t s) {
    with_bool(a.prime != 0, [&](auto P) {
        with_bool(a.odd != 0, [&](auto O) {
            if (a.T > 1 && !a.big) {
                hipLaunchKernelGGL((k_ifft_rows_plane_staged<P.value, O.value>),
                                   dim3(row_stage_blocks(a.Y, a.T), (a.T + 7) / 8, nplanes), dim3(64 * row_stage_waves(a.T)),
                                   row_stage_lds(a.wbuf, a.T), s, a);
                return;
            }
            const dim3 grid(row_blocks(a.Y, a.T, ROWS_PER_WG), (a.T + 7) / 8, nplanes), block(64 * ROWS_PER_WG);
            const size_t lds = ifft_rows_plane_lds(a.wbuf, a.big != 0);
            if (a.big) hipLaunchKernelGGL((k_ifft_rows_plane<P.value, true, true>), grid, block, lds, s, a);
            else hipLaunchKernelGGL((k_ifft_rows_plane<P.value, false, O.value>), grid, block, lds, s, a);
        });
    });
    return hipGetLastError();
}
hipError_t launch_fit(const float* img, const float* im, long long n_per_frame, int T, int im_frames, double* part,
                      int nblk, double* out, hipStream_t s) {
    hipLaunchKernelGGL(k_fit_partial, dim3(nblk, T), dim3(256), 0, s, img, im, n_per_frame, im_frames, part, nblk);
    hipLaunchKernelGGL(k_fit_final, dim3(T), dim3(256), 0, s, part, nblk, out);
    return hipGetLastError();
}
hipError_t configure_kernels(size_t max_lds) {
    const void* ks[] = {(const void*)k_small_fft<SFFT_64>, (const void*)k_small_fft<SFFT_128>, (const void*)k_small_fft<SFFT_256>,
                        (const void*)k_psf_rows<false>, (const void*)k_psf_cols<false>,
                        (const void*)k_psf_rows<true>, (const void*)k_psf_cols<true>,
                        (const void*)k_ifft_cols<false, false>, (const void*)k_ifft_cols<true, false>,
                        (const void*)k_ifft_cols<false, true>, (const void*)k_ifft_cols<true, true>,
                        (const void*)k_spec_pack,
                        (const void*)k_small_fft_grouped<SFFT_64>, (const void*)k_small_fft_grouped<SFFT_128>, (const void*)k_ifft_cols_grouped<false>,
                        (const void*)k_ifft_cols_grouped<true>};
    std::vector<const void*> all(std::begin(ks), std::end(ks));
    for (bool prime : {false, true})
        for (bool odd : {false, true})
            with_bool(prime, [&](auto P) {
                with_bool(odd, [&](auto O) {
                    all.push_back((const void*)k_ifft_rows_sum<P.value, O.value>);
                    all.push_back((const void*)k_ifft_rows_sum_staged<P.value, O.value>);
                    all.push_back((const void*)k_ifft_rows_plane<P.value, false, O.value>);
                    all.push_back((const void*)k_ifft_rows_plane_staged<P.value, O.value>);
                    all.push_back((const void*)k_ifft_rows_plane<P.value, true, true>);
                });
            });
    for (int slots : {2, 4})
        for (int ns = 1; ns <= slots; ns *= 2)
            for (bool pp : {false, true})
                mac_variant(slots, ns, pp, [&](auto sl, auto n, auto p) {
                    all.push_back((const void*)k_mac<sl.value, n.value, p.value>);
                    all.push_back((const void*)k_mac_grouped<sl.value, n.value, p.value>);
                });
    for (const void* k : all) {
        hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_lds);
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_rl_scale(float* X, const float* Htf, const float* v, int nz, int T, long long npix, int v_frames,
                           hipStream_t s, bool ratio) {
    const long long ch = (long long)RL_SCALE_THREADS * RL_SCALE_E;
    long long blocks = (npix + ch - 1) / ch;
    if (blocks > 65535) blocks = 65535;
    if (blocks < 1) blocks = 1;
    // slabs on y (nz * T <= 65535 is checked by the caller), pixels on x
    hipLaunchKernelGGL(k_rl_scale, dim3((unsigned)blocks, (unsigned)(nz * T)), dim3(RL_SCALE_THREADS), 0, s, X, Htf,
                       v, T, npix, v_frames, ratio ? 1 : 0);
    return hipGetLastError();
}
hipError_t launch_fill(float* p, long long n, float v, hipStream_t s) {
    long long blocks = (n + 255) / 256;
    if (blocks > 65536) blocks = 65536;
    if (blocks < 1) blocks = 1;
    hipLaunchKernelGGL(k_fill, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
    return hipGetLastError();
}

}  // namespace flf
