// Kernel argument blocks and host launchers (internal to libflf_hip).
#pragma once
#include "flf_common.h"

#define FLF_MAX_GROUPS 8
#define FLF_SMAX_WAYS 4          // words that share the maximum of one (plane, frame)
#define FLF_MAX_PLANES 256       // planes per plan: the plane selection travels in kernel arguments

// Planes of a grid group selected for one projection, as a bitmask carried
// by value in the kernel arguments (a captured graph replays its own
// selection, whatever later calls select).
struct PlaneMask {
    unsigned int w[FLF_MAX_PLANES / 32];
    __host__ __device__ bool on(int p) const { return (w[p >> 5] >> (p & 31)) & 1u; }
};

// Block ranges of a grouped launch (one dispatch for every active grid group
// of a projection).  start[g] is group g's first flattened block,
// start[ngroups] the total; nchunks/nranges split a group's blocks (MAC:
// chunks x plane ranges, each group's range padded to a multiple of 8;
// column transform: column blocks x batches).
struct GroupedGrid {
    int ngroups;
    int start[FLF_MAX_GROUPS + 1];
    int nchunks[FLF_MAX_GROUPS];
    int nranges[FLF_MAX_GROUPS];
};

struct SmallFFTArgs {
    const float* src;            // source base
    const long long* src_off;    // per source plane z: element offset (device array)
    long long src_tstride;       // per frame
    int src_pitch;               // row pitch (elements)
    int Y, X, N;
    RadixPlan rpY, rpX;          // lengths rY, rX
    const float2* twY;           // exp(-2 pi i m / rY), m < rY
    const float2* twX;           // exp(-2 pi i m / rX)
    const unsigned* sidx;        // [chunk][NH]: H column, H row << 8, conjugate << 31 (output order)
    int nchunks, NH;             // chunks; residues stored per chunk (4 quad / 2 pair)
    int fY, fX;
    float2* S;                   // [chunk][N*N][NH] per source plane and frame
    const long long* S_off;      // per source plane z: element offset into S (device array)
    long long S_tstride;         // per frame
    const int2* fdims;           // per frame valid (Y, X) <= (Y, X), or null (all full size)
    float* smax;                 // per source plane and frame: largest |component| of S, in FLF_SMAX_WAYS parts
    int smax_zstride;
    const float* src2;           // frames t >= tsplit read from src2 (frame t - tsplit), or null
    int tsplit;
};

struct PsfRowArgs {
    const float* Q;              // quadrant (h, h, s2, s2)
    int h, s2, RB;
    const int* u_bu;
    const int* u_au;
    RadixPlan rpX;               // length fX
    float2* tmp;                 // (nu, s2, rfX)
};

struct PsfColArgs {
    const float2* tmp;           // (nu, s2, rfX)
    int s2, rfX, CB;
    RadixPlan rpY;               // length fY
    float2* spec;                // (nu, fY, rfX)
};

struct SpecPackArgs {
    const float2* spec;          // (nu, fY, rfX) natural layout, one plane
    const ChunkDesc* chunks;
    const ItemDesc* items;
    const int* u_bu;
    const int* u_au;
    int fY, fX, rfX, N, slots, nu, nP, p;
    int kg;                      // 16-byte units per item, plane and half (square: nu, else ceil(nu / 2))
    int s2;                      // PSF side of the plane (sets the folded phase ratios)
    uint4* G;                    // orbit-major split spectra of the grid group
    float2* E;                   // output factors of the grid group
    float2* psi;                 // flip factors of the grid group
};

struct MacArgs {
    const uint4* G;              // k_spec_pack's G, E and psi
    const float2* E;
    const float2* psi;
    const ChunkDesc* chunks;
    const ushort4* wpos;         // per item: the place of each slot's bin in its chunk (GridTables::wpos)
    const TileDesc* tiles;
    const int2* pairs;           // [nu][slots]: the plain and conjugated use of each pair type (GridTables::pairs)
    const float2* S;
    long long S_pstride;         // per plane in group (0: one image for all)
    long long S_tstride;
    const float* smax;           // SmallFFTArgs::smax; smax_pstride floats per plane (0: one image for all)
    int smax_pstride;
    PlaneMask enable;            // planes of the group in this projection
    int nP;
    float2* A;
    long long A_tstride, A_pstride;
    int N, nu;
    int kg;                      // 16-byte units per item and plane
    int T;                       // frames, in blocks of mac_frames(slots, T)
    int per_plane;               // 1: store each plane's accumulator at A + p * A_pstride (back
                                 // projection); 0: sum the planes of a range, store at
                                 // A + range * A_pstride (forward projection)
    int fgroup;                  // frame blocks dispatched side by side per chunk (0: all)
};

struct IfftColArgs {
    const float2* A;
    long long A_bstride;         // per frame
    const int* colidx;           // [k1][y0][m]: place of bin (y0 + m rY, k1) (GridTables::colidx)
    int N, rY;
    int T, FB;                   // frames, interleaved in blocks of FB (mac_frames)
    int nsum;                    // partial accumulators summed on load (>= 1)
    long long A_sstride;
    int rfX, CB, Yout;
    RadixPlan rpY;
    const float2* twY;           // exp(-2 pi i m / fY)
    float2* out;
    long long out_bstride;
};

// Every active grid group's arguments of one stage, by value in the kernel
// arguments (pointers read from kernel arguments are known to be global, so
// the kernels load through them with global rather than flat loads).
struct SmallFFTGrouped {
    SmallFFTArgs a[FLF_MAX_GROUPS];
    GroupedGrid gg;
};
struct MacGrouped {
    MacArgs a[FLF_MAX_GROUPS];
    GroupedGrid gg;                               // blocks per group: nchunks x nranges x nfb, padded to 8
    int nfb;                                      // frame blocks
};
struct IfftColGrouped {
    IfftColArgs a[FLF_MAX_GROUPS];
    GroupedGrid gg;
};

struct IfftRowGroup {
    const float2* T;             // per block of FB frames (Y, rfX, frames)
    long long tstride;           // per frame
    int rfX;
    int FB;
    int active;
    float scale;
    RadixPlan rp;                // length fX
    RadixPlan rph;               // length fX/2 (even fX)
    const float2* twf;           // exp(-2 pi i m / fX)
    const float2* twh;           // exp(-2 pi i m / (fX/2))
};

struct IfftRowSumArgs {
    IfftRowGroup grp[FLF_MAX_GROUPS];
    float* smax;                 // nsmax maxima to zero (SmallFFTArgs::smax)
    int nsmax;
    int ngroups;
    int maxfX;
    int wbuf;                    // c2r_wave_buffer, max over the active groups
    int X, Y, T;
    float* img;                  // forward image, or null (not stored)
    long long img_tstride;
    const int2* fdims;           // per frame valid size; outside it the image is 0
    const float* im;             // with ratio: the measured image (T, Y, X)
    float* ratio;                // if set: ratio = im / image (standard RL, lfdeconv.py:191), 0 outside
};

struct RowPlaneDesc {
    long long T_off;             // element offset of this plane's column transforms
    long long T_tstride;         // per frame
    int rfX;
    int slots;                   // of the grid (4 square, 2 else)
    float scale;
    RadixPlan rp;                // length fX
    RadixPlan rph;               // length fX/2 (even fX)
    const float2* twf;
    const float2* twh;
};

struct IfftRowPlaneArgs {
    const RowPlaneDesc* pd;      // per plane z
    unsigned short plane_ids[FLF_MAX_PLANES];   // planes to process (grid z), by value
    float* smax;                 // nsmax maxima to zero
    int nsmax;
    const float2* Tbuf;
    float* vol;                  // (nz, T, Y, X)
    const float* Htf;            // mode 1
    const float* trust;          // mode 2 (optional, (nz, 1, Y, X))
    int mode;                    // 0 store, 1 Prevedel update, 2 standard update
    int T, Y, X;
    int FB4, FB2;                // frames interleaved per block on square and other grids
    int wbuf;                    // per-wave LDS buffer (float2): max over planes of fX/2 (even) or fX
    const int2* fdims;           // per frame valid size; outside it the volume is set to 0
    int prime;                   // some plane's row plan ends with an odd prime radix above 5
    int odd;                     // some plane's rows have an odd length
    int big;                     // some plane's rows are longer than 2048 (out-of-place transforms)
};

namespace flf {
size_t small_fft_lds(int rY, int rX);
size_t ifft_cols_lds(int CB, int fY);
// LDS stride of one column of the column transform: fY padded so that the CB
// columns of one row, written and read by consecutive threads, fall on
// distinct banks (FLF_COLS_BANKS banks of 4 bytes; 0: unpadded).
#ifndef FLF_COLS_BANKS
#define FLF_COLS_BANKS 64
#endif
__host__ __device__ inline int ifft_col_stride(int fY, int CB) {
    if (FLF_COLS_BANKS == 0 || CB < 2) return fY;
    const int m = FLF_COLS_BANKS / 2;      // float2 entries per sweep of the banks
    const int r = (m / CB) % m;
    return fY + ((r - fY) % m + m) % m;
}
size_t ifft_rows_plane_lds(int wbuf, bool big);
bool wave_big(int L);
bool small_fft_big(int rY, int rX);
int c2r_wave_buffer(int fX);
hipError_t launch_small_fft(const SmallFFTArgs& a, int nsrc, int T, hipStream_t s);
// Grouped launches (the groups' arguments by value).
hipError_t launch_small_fft_grouped(const SmallFFTGrouped& ga, int N, int T, size_t lds, hipStream_t s);
hipError_t launch_mac_grouped(const MacGrouped& ga, int slots, hipStream_t s);
hipError_t launch_ifft_cols_grouped(const IfftColGrouped& ga, int CB, bool prime, size_t lds, hipStream_t s);
hipError_t launch_psf_rows(const PsfRowArgs& a, int nu, hipStream_t s);
hipError_t launch_psf_cols(const PsfColArgs& a, int nu, hipStream_t s);
size_t spec_pack_lds(int nu, int slots);
hipError_t launch_spec_pack(const SpecPackArgs& a, int nchunks, hipStream_t s);
int mac_frames(int slots, int T);             // frames per MAC workgroup
size_t mac_lds(int slots, int T);
hipError_t launch_mac(const MacArgs& a, int slots, int nchunks, int nplanes_grid, hipStream_t s);
int ifft_col_blocks(const IfftColArgs& a);
hipError_t launch_ifft_cols(const IfftColArgs& a, int nbatch, hipStream_t s);
hipError_t launch_ifft_rows_sum(const IfftRowSumArgs& a, int Y, int T, hipStream_t s);
hipError_t launch_ifft_rows_plane(const IfftRowPlaneArgs& a, int nplanes, hipStream_t s);
// Data-fit sums: frame t of img against frame t % im_frames of im; part holds
// 2 * nblk * T doubles of partial sums, out 2 * T.
hipError_t launch_fit(const float* img, const float* im, long long n_per_frame, int T, int im_frames, double* part,
                      int nblk, double* out, hipStream_t s);
hipError_t launch_fill(float* p, long long n, float v, hipStream_t s);
// X = [X *] Htf / v over nslab (plane, frame) slabs of npix values; v holds
// one slab per plane (v_frames = 1, shared by the T frames) or per slab
// (v_frames = T).
hipError_t launch_rl_scale(float* X, const float* Htf, const float* v, int nz, int T, long long npix, int v_frames,
                           hipStream_t s, bool ratio = false);
// Whether a radix plan ends with an odd prime radix above 5.
bool plan_has_prime(const RadixPlan& rp);
// Raise the dynamic-LDS limit of the FFT kernels to max_lds bytes.
hipError_t configure_kernels(size_t max_lds);
}  // namespace flf
