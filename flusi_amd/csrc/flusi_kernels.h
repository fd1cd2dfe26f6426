// Kernel argument blocks and launcher declarations shared by the transform
// passes (passes.hip), the field kernels (fields.hip) and the solver host code.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace flusi {

// Element offsets of a 3-D complex array walked as (a = FFT axis,
// b = tile axis, c = outer axis).
struct Strides { long a, b, c; };

// Batched launches.  The members of a batch (simulations of one grid and one
// parameter set) keep identical buffer layouts in slabs `mstride` bytes
// apart.  A batched launch adds one grid dimension over its nmem members and
// shifts every device pointer of the argument block by member * mstride;
// nmem <= 1 is a plain launch.
template <typename P> __host__ __device__ __forceinline__ P* mshift(P* p, long off) {
  return p ? reinterpret_cast<P*>(reinterpret_cast<uintptr_t>(p) + off) : p;
}
struct Batch {
  int nmem;      // members in the launch (0 or 1: not batched)
  long mstride;  // bytes between two members' slabs (a multiple of 256)
};
__host__ __device__ __forceinline__ int batch_n(const Batch& b) { return b.nmem > 1 ? b.nmem : 1; }

// Dealiased ("pruned") passes.  With dealiasing every stepper writes zero to
// the modes outside the ellipsoid (kx/Kx)^2 + (ky/Ky)^2 + (kz/Kz)^2 < 1,
// K = 2/3 (n/2 - 1) (vis.f90:23-53): 15 % of the half spectrum is left, its
// (kx, ky) shadow is 35 %, its kx range 2/3.  The pruned passes move and
// transform only what those modes need and what they produce.  Their Q layout
// is compact: row position p holds ky = p - ym0, nyp positions a row.
struct Prune {
  int ym0;                 // largest |ky| of the region
  int nyp;                 // Q row length: 2 ym0 + 1 rounded up to whole 128-byte lines
  int nkx;                 // kx = 0..nkx-1 hold the region
  const int16_t* ylim;     // per kx (nkx): largest |ky|
  const int16_t* zlim;     // per (kx, p) (nkx x nyp): largest |kz|, -1 outside
};
// the passes' use of the region
enum PruneMode {
  PR_NONE = 0,
  PR_ZINV = 1,   // state rows inside the region -> compact Q rows
  PR_YINV = 2,   // compact Q rows -> P, kx < nkx
  PR_YFWD = 3,   // P, kx < nkx -> the compact Q rows' region (whole 128-byte lines of it)
};

enum TileOp { OP_COPY = 0, OP_DERIV = 1, OP_DERIV_MINUS = 2 };

// One job reads its operands once and writes one or two transforms of them.
struct TileJob {
  const void* in0;   // complex field, layout given by Strides in
  const void* in1;   // second operand of OP_DERIV_MINUS (nullptr: not read)
  void* out;
  int op;            // out = in0 | i k_a in0 | i k_a in0 - in1
  void* out2;        // second output of the same operands (nullptr: none)
  int op2;
};

struct TilePassArgs {
  TileJob jobs[6];
  int njobs;
  int nb, nc;          // extents of the tile axis and the outer axis
  int nb_store;        // in-wave passes: lines the segment-side store covers (>= nb; lines
                       // beyond nb are row padding no kernel reads, stored as zeros so that
                       // the last tile writes whole 128-byte segments); 0 = nb
  Strides sin, sout;
  double kscale;       // k_a = kscale * wrap(a): wavenumbers along the FFT axis
  double scale;        // applied to every stored value
  const void* tw;      // L twiddles exp(-2 pi i m / L), element type of the pass
  int pf;              // block passes: load the next job's operand while the current one is transformed
  unsigned ibytes, obytes;  // bytes of one input / output field (buffer descriptors)
  int prune;           // PruneMode
  Prune pr;
  const uint32_t* tiles;  // PR_ZINV: (c << 16 | first line / TL) per workgroup, ntiles of them
  int ntiles;
  Batch bat;           // grid z: member
};

// x pass modes
enum XMode {
  XM_RHS = 0,       // 6 spectral fields -> u x w - chi (u - us) [+ sponge] -> 3 [6] spectral
  XM_INV_UW = 1,    // 6 spectral fields -> u (3) and w (3) in physical space
  XM_INV = 2,       // nf spectral fields -> nf physical fields
  XM_FWD = 3,       // nf physical fields -> nf spectral fields
};

struct XPassArgs {
  const void* in;      // nf spectral (P layout) or physical fields, field stride fstride_in
  void* out;           // outputs, field stride fstride_out
  long fstride_in, fstride_out;
  int nf;              // fields for XM_INV / XM_FWD
  int nlines;          // ny*nz
  int nx, ny, nxh;
  long prow;           // row stride of the spectral (P-layout) side
  int kin, kout;       // spectral entries read (the others are zero) and written per line
  unsigned fbytes;     // bytes of one P field (buffer descriptor)
  const double* kx;    // nxh wavenumbers
  double kx_scale;     // kx = kx_scale * k
  const void* twM;     // M = nx/2 twiddles
  const void* twN;     // nxh twiddles exp(-2 pi i k / nx)
  const void* twX;     // nx twiddles exp(-2 pi i m / nx)
  // RHS extras
  const void* mask;    // N reals (element type of the pass)
  const void* us;      // 3N reals, component stride N
  const uint8_t* mflag;  // per x line (ny*nz): 0 where the line's mask is all zero (not read); null: read every line
  long npts;           // N
  double eps_inv;      // 1/eta
  int sponge;          // 0 none, 1 cavity, 2 outlet_x
  int sponge_thickness;
  double sponge_eps_inv;
  double sponge_mask_thr;
  int nz;
  double* partial;     // per block: umax^2, sum chi(u-us) x,y,z (4 doubles)
  int want_stats;      // write the per-block statistics (adaptive dt / dynamic mean flow)
  Batch bat;           // grid y: member
};

// XPassArgs with its pointers moved to batch member m
__host__ __device__ __forceinline__ void to_member(XPassArgs& a, int m) {
  const long o = (long)m * a.bat.mstride;
  a.in = mshift(a.in, o); a.out = mshift(a.out, o); a.kx = mshift(a.kx, o);
  a.twM = mshift(a.twM, o); a.twN = mshift(a.twN, o); a.twX = mshift(a.twX, o);
  a.mask = mshift(a.mask, o); a.us = mshift(a.us, o); a.partial = mshift(a.partial, o);
}

// z-forward pass with the fused spectral epilogue (projection, explicit
// diffusion, dealiasing, stepper update, zero-mode forcing, Parseval sum)
enum StepMode {
  SM_RHS_ONLY = 0,   // out0 = nlk (projected)
  SM_EULER = 1,      // AB2 start-up Euler step
  SM_AB2 = 2,
  SM_RK2_1 = 3,
  SM_RK2_2 = 4,
  SM_RK4_1 = 5,
  SM_RK4_2 = 6,
  SM_RK4_3 = 7,
  SM_RK4_4 = 8,
  SM_PRESSURE = 9,   // out0 = -i k.nlk / k^2 of the unprojected right-hand side (1 field)
};

struct ZStepArgs {
  const void* nq;        // 3 (6 with sponge) Q-layout fields, field stride fs
  long fs;
  int nx, ny, nz, nxh;
  const double* kx; const double* ky; const double* kz;
  const double* kxt2; const double* kyt2; const double* kzt2;  // dealias predicate terms
  const void* tw;        // nz twiddles
  double scale;          // 1/(nx ny nz)
  int mode;
  int sponge;
  int dealias_on;        // iDealias
  double nu;
  // state (S layout, 3 fields each, field stride fs)
  void* u;               // uk (AB2/RK2), u_n (RK4)
  const void* udiff;     // field the explicit diffusion term is taken from (stage input)
  void* ustage;          // RK4 next-stage input (written)
  void* acc;             // RK4 accumulator
  void* r0;              // AB2: nlk(n0) out; RK2: N0 (out in stage 1, in stage 2)
  const void* r1;        // AB2: nlk(n1) in
  void* rhs_out;         // SM_RHS_ONLY output
  double dt, b10, b11;
  double vis_dt_new;     // IF exponent dt (<0: factor is zero)
  double vis_dt_old;     // RK2 stale IF (<0: zero)
  int explicit_diffusion;
  // zero mode forcing
  int meanflow_dynamic[3];
  const double* pen_sum; // device sum chi(u-us) over the grid (3 doubles)
  double dynamic_scale;  // dx dy dz * startup / m_fluid (negated applied)
  int set_mean[3];       // post-step zero-mode overwrite (fixed/sinusoidal)
  double mean_value[3];
  double* energy_partial;  // per block Parseval partial sum (final stages only)
  int wave;              // 1: transform each z line inside one wavefront (nz = 64..512)
  int eu;                // block kernel, nz >= 256: epilogue positions scheduled together (0 = all)
  // prune & 1: the state operands are zero outside the dealiased region and
  // are not read there; prune & 2: the result is, too - Q is compact and only
  // the region (its whole 128-byte lines) is transformed and written
  int prune;
  Prune pr;
  const uint32_t* tiles;  // prune & 2: (kx << 16 | first line / TL) per workgroup, ntiles of them
  int ntiles;
  Batch bat;             // grid z: member
};

// launchers (passes.hip)
template <typename T> void launch_tile_pass(const TilePassArgs& a, int L, int dir, bool contig_in, hipStream_t s);
// the same passes with each line transformed inside one wavefront (tiles_wave.hip)
template <typename T> void launch_tile_wave(const TilePassArgs& a, int L, int dir, bool contig_in, hipStream_t s);
bool tile_wave_supported(int L);
bool zstep_wave_supported(int nz);  // in-wave z step (else the block kernel)
template <typename T> void launch_x_pass(const XPassArgs& a, int mode, hipStream_t s);
template <typename T> void launch_zstep(const ZStepArgs& a, hipStream_t s);
int x_pass_blocks(int nx, int nlines, bool fp64);
// the right-hand-side x pass with pairs of lines inside one wavefront (xrhs_wave.hip)
template <typename T> void launch_x_rhs_wave(const XPassArgs& a, hipStream_t s);
// its inverse transforms alone: XM_INV (1 or 3 fields) and XM_INV_UW
template <typename T> void launch_x_inv_wave(const XPassArgs& a, int mode, hipStream_t s);
bool x_rhs_wave_supported(int nx);
int x_rhs_wave_blocks(int nx, int nlines, bool fp64);
// per x line (iy, iz) of [y0, y1] x [z0, z1]: flag[iz ny + iy] = 1 where any
// mask value of the line is nonzero, else 0 (xrhs_wave.hip)
template <typename T>
void launch_mask_flags(const void* mask, uint8_t* flag, int nx, int ny, int y0, int y1, int z0, int z1, hipStream_t s);
// lines per workgroup of the pruned z passes: the tile lists are built for them
int tile_lines(bool fp64);                                  // z inverse
int zstep_tile_lines(int nz, bool fp64, bool wave);
// energy partial sums one z-step launch writes per member (the block kernel
// or, wave = true, the in-wave kernel)
int zstep_blocks(int nz, int ny, int nxh, bool fp64, bool wave);
bool fft_length_supported(int n);   // y/z line lengths
bool x_length_supported(int m);     // nx/2 of the real x axis

// reductions (fields.hip)
// out[v] = combine over rows of partial[row*nv + v]; kind[v]: 0 = Neumaier sum, 1 = max, 2 = min
// mirror (mapped host memory, may be null) receives the results, too
void launch_reduce_rows(const double* partial, int nrows, int nv, const int* kinds_dev, double* mid, double* out, hipStream_t s,
                        double* mirror = nullptr);
size_t reduce_rows_scratch(int nv);  // doubles of `mid` needed for nv values

}  // namespace flusi
