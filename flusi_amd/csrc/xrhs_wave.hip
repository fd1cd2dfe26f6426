// x pass of the right-hand side: two x lines (neighbours in y) per complex
// transform of length nx, inside one wavefront.
//
// The lines' spectra A and B are combined to Z = A + i B over all nx modes
// (Z[nx - k] = conj A[k] + i conj B[k]), so that one complex transform of
// length nx gives line a in its real and line b in its imaginary parts, and
// the other way round.  Against one length-nx/2 transform per line with the
// even/odd split, a pair needs no split twiddles and, with E = 8 (12 where 3
// divides nx) positions a lane instead of 4, exchanges its values twice
// through LDS instead of three or four times: the pass was bound by its VALU
// issue and its LDS traffic together (nx = 512, FP32: 2000 VALU and 400 LDS
// instructions a line, 78 % VALU issue).  A pair takes about 2640 VALU and 300
// LDS instructions: 512^3 FP32 1291 -> 719 us (3.3 GB: 4.6 TB/s), 192x96x384
// FP32 (block pass before) 205 -> 79 us.
//
// A pair lives in the registers of G = nx/E lanes, lane l holding positions
// l + qG (q = 0..E-1) before and after every transform; 64/G pairs a wave.
// Stages exchange through the pair's own LDS row with wave-scope ordering
// only: waves never wait for each other.
//
// Per line (rhs.f90:147-330 cal_nlk_fsi, nonlinear and penalisation part):
//   load the six spectra V_x, V_y, V_z, w_x, A = dz u_x, B = dy u_x
//   form w_y = A - i kx V_z, w_z = i kx V_y - B            (basic_operators.f90:185-215)
//   C2R of u and w                                         (cof_p3dfft.f90:65-83)
//   nl = u x w - mask/eta (u - us) [- w/eta_sponge in the sponge]
//   R2C of nl [and of the sponge term]                      (cof_p3dfft.f90:33-56)
//   per block: max |u|^2 and the compensated sums of mask/eta (u - us)
#include "fft_core.h"
#include "flusi_kernels.h"
#include <cstdlib>
#include <stdexcept>
#include <string>

#ifndef FLUSI_PART
#define FLUSI_PART 0
#endif

namespace flusi {

namespace {

constexpr int XW_NT = 256;  // most threads of a block: independent waves

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ double wsum(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}
__device__ __forceinline__ double wmax(double v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = nanmax(v, __shfl_xor(v, o, 64));
  return v;
}

// E = 8: 512 = 8.8.8, 256 = 8.8.4, 128 = 8.4.4, 64 = 8.8, 32 = 8.4;
// E = 4: 256 = 4.4.4.4, 128 = 4.4.4.2, 64 = 4.4.4, 32 = 4.4.2, 96 = 6.4.4 (its
// first stage reads its inputs from the row, see pstage0);
// E = 12: 384 = 12.4.4.2, 192 = 12.4.4, 96 = 12.4.2, 48 = 12.4
template <int N_, int E_> struct PairPlan {
  static constexpr int N = N_, E = E_;
  static constexpr int G = N / E;     // lanes of a pair
  static constexpr int PPW = 64 / G;  // pairs of a wave
  // 96 over 24 lanes leaves 16 lanes of a wave idle: they run the same code on
  // a spare row, which the kernel clears first, so that all they hold is zero
  // (a few positions of that row are read that no lane writes), and neither
  // store nor enter the statistics
  static constexpr int IDLE = 64 - PPW * G;
  static constexpr int ROWS = PPW + (IDLE > 0 ? 1 : 0);
  static constexpr bool ROW0 = E == 4 && N % 3 == 0;
  static_assert(E * G == N && (IDLE == 0 || N == 96), "in-wave pair length");
  static constexpr __host__ __device__ int radix(int s) {
    int m = N;
    for (int i = 0;; ++i) {
      const int r = i == 0 ? (ROW0 ? 6 : E) : (E == 8 && (m == 8 || m == 64 || m == 32) ? 8 : (m % 4 == 0 ? 4 : 2));
      if (i == s) return r;
      m /= r;
    }
  }
  static constexpr __host__ __device__ int ns(int s) { int p = 1; for (int i = 0; i < s; ++i) p *= radix(i); return p; }
  static constexpr int QL = (E + 2) / 3;  // groups l + qG that hold the modes of a dealiased state (k < N/3 + 1)
};

// lp(b + k) = lp(b) + lp(k) for a lane's accesses: one address per lane and
// stage then serves all elements through the instruction's immediate offset
template <typename T, typename PP> constexpr bool split_rd() {
  for (int l = 0; l < PP::G; ++l)
    for (int q = 0; q < PP::E; ++q)
      if (lp<T>(l + q * PP::G) != lp<T>(l) + lp<T>(q * PP::G) || lp<T>(PP::G - l + q * PP::G) != lp<T>(PP::G - l) + lp<T>(q * PP::G))
        return false;
  return true;
}
template <typename T, typename PP, int s> constexpr bool split_wr() {
  constexpr int N = PP::N;
  constexpr int R = PP::radix(s), Ns = PP::ns(s);
  for (int j = 0; j < N / R; ++j)
    for (int q = 0; q < R; ++q) {
      const int b = (j / Ns) * Ns * R + j % Ns;
      if (lp<T>(b + q * Ns) != lp<T>(b) + lp<T>(q * Ns)) return false;
    }
  return true;
}

// reads positions l + qG of the pair's row
template <typename T, typename PP> __device__ __forceinline__ void row_read(cplx<T> (&v)[PP::E], const cplx<T>* ln, int l) {
  constexpr int E = PP::E, G = PP::G;
  const cplx<T>* rd = ln + lp<T>(l);
#pragma unroll
  for (int q = 0; q < E; ++q) v[q] = split_rd<T, PP>() ? rd[lp<T>(q * G)] : ln[lp<T>(l + q * G)];
}

// Stage s: B = E/R butterflies per lane, j = l + bG; input q of butterfly b
// is register b + qB (position j + q N/R); outputs go to (j/Ns) Ns R + j%Ns +
// q Ns, which for the last stage is again register b + qB.  tw: the block's
// LDS copy of exp(-2 pi i m / N).
template <typename T, typename PP, int S, int s>
__device__ __forceinline__ void pstage(cplx<T> (&v)[PP::E], const cplx<T>* tw, cplx<T>* ln, int l) {
  constexpr int N = PP::N, E = PP::E, G = PP::G, R = PP::radix(s), Ns = PP::ns(s), B = E / R;
  constexpr bool last = Ns * R == N;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const unsigned j = (unsigned)l + b * G;
    cplx<T> x[R];
#pragma unroll
    for (int q = 0; q < R; ++q) x[q] = v[b + q * B];
    if constexpr (s > 0) {
      const int step = (int)(j % Ns) * (N / (Ns * R));
#pragma unroll
      for (int q = 1; q < R; ++q) x[q] = (S < 0) ? cmul(x[q], tw[q * step]) : conjmul(x[q], tw[q * step]);
    }
    Bfly<R, S, T>::run(x);
    if constexpr (last) {
#pragma unroll
      for (int q = 0; q < R; ++q) v[b + q * B] = x[q];
    } else {
      const int base = (int)(j / Ns) * Ns * R + (int)(j % Ns);
      cplx<T>* wr = ln + lp<T>(base);
#pragma unroll
      for (int q = 0; q < R; ++q) {
        if constexpr (split_wr<T, PP, s>()) wr[lp<T>(q * Ns)] = x[q];
        else ln[lp<T>(base + q * Ns)] = x[q];
      }
    }
  }
  if constexpr (!last) {
    wave_sync();
    row_read<T, PP>(v, ln, l);
    wave_sync();
    pstage<T, PP, S, s + 1>(v, tw, ln, l);
  }
}

// Stage 0 of a plan whose first radix is not the lane's E (96 = 6.4.4 over 24
// lanes): the row holds the inputs at their positions, the first N/R lanes
// take one butterfly each.
template <typename T, typename PP, int S>
__device__ __forceinline__ void pstage0(cplx<T> (&v)[PP::E], const cplx<T>* tw, cplx<T>* ln, int l) {
  constexpr int N = PP::N, R = PP::radix(0);
  const int j = l < N / R ? l : 0;
  cplx<T> x[R];
#pragma unroll
  for (int q = 0; q < R; ++q) x[q] = ln[lp<T>(j + q * (N / R))];
  wave_sync();
  Bfly<R, S, T>::run(x);
  if (l < N / R) {
#pragma unroll
    for (int q = 0; q < R; ++q) ln[lp<T>(R * j + q)] = x[q];
  }
  wave_sync();
  row_read<T, PP>(v, ln, l);
  wave_sync();
  pstage<T, PP, S, 1>(v, tw, ln, l);
}

// (a plan with ROW0: the row holds the inputs)
template <typename T, typename PP, int S>
__device__ __forceinline__ void pfft(cplx<T> (&v)[PP::E], const cplx<T>* tw, cplx<T>* ln, int l_) {
  // recompute the LDS addresses in every transform instead of keeping a
  // few dozen of them live across the whole kernel
  int l = l_;
  asm volatile("" : "+v"(l));
  if constexpr (PP::ROW0) pstage0<T, PP, S>(v, tw, ln, l);
  else pstage<T, PP, S, 0>(v, tw, ln, l);
}

// i k x a pair's combined modes: Z takes i kx Z, the mirrored M its conjugate
template <typename T> __device__ __forceinline__ cplx<T> ik_p(T k, cplx<T> v) { return mk<T>(-k * v.y, k * v.x); }

// complex load through a buffer with a wave-uniform byte offset on top of the
// lane's (an out-of-range lane offset reads zero).  Stores carry the whole
// offset in the lane's register (bst): the hazard of a 16-byte store whose data
// registers the next instruction overwrites is not covered by the compiler
// where the store has a scalar offset (seen: four lanes' data replaced).
template <typename T> __device__ __forceinline__ cplx<T> bld_s(brsrc r, unsigned off, unsigned soff) {
  if constexpr (sizeof(T) == 4) return __builtin_bit_cast(cplx<T>, __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0));
  else return __builtin_bit_cast(cplx<T>, __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, 0));
}
// one real through a buffer
template <typename T> __device__ __forceinline__ T rld(brsrc r, unsigned off) {
  if constexpr (sizeof(T) == 4) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
  else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}
template <typename T, int N> constexpr int pair_row() { return line_stride<T>(N + 1); }
template <typename T, typename PP> constexpr size_t pair_smem(int waves) {
  return sizeof(cplx<T>) * ((size_t)waves * PP::ROWS * pair_row<T, PP::N>() + PP::N);
}

// waves per SIMD the register allocation must allow
template <typename T, int N, int E, int VAR, int PR, int NF> constexpr int pair_wpe() {
  if (NF < 6) return sizeof(T) == 4 ? 4 : 3;
  if (E == 12) return sizeof(T) == 4 ? 2 : 1;
  if (E == 4) return sizeof(T) == 4 ? 4 : (N % 3 == 0 ? 2 : 3);
  return sizeof(T) == 4 ? (VAR == 0 && PR > 0 ? 4 : 3) : 2;
}

// PR 1: the spectra are zero at k >= QL G (a dealiased state), so that only QL
// groups a line are loaded and mirrored; PR 2: no more are stored, either.
// VAR: 0 plain, 1 with the statistics, 2 sponge (and the statistics if asked),
// 3 the inverse transforms alone, to physical fields: NF = 6 (u and w), 3 or 1
// fields as they come
template <typename T, int N, int E, int VAR, int PR, int NF>
__global__ __launch_bounds__(XW_NT) __attribute__((amdgpu_waves_per_eu(pair_wpe<T, N, E, VAR, PR, NF>()))) void x_rhs_pair_k(XPassArgs a) {
  to_member(a, blockIdx.y);
  using PP = PairPlan<N, E>;
  constexpr int G = PP::G, PPW = PP::PPW, H = E / 2;
  constexpr bool PIN = PR > 0;
  constexpr int QL = PIN ? PP::QL : H, QO = PR == 2 ? PP::QL : H;
  constexpr int LS = pair_row<T, N>();
  constexpr bool SPONGE = VAR == 2;
  constexpr unsigned ES = sizeof(cplx<T>);
  extern __shared__ char smem_raw[];
  __shared__ double red[XW_NT / 64][4];
  cplx<T>* twl = reinterpret_cast<cplx<T>*>(smem_raw);
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, wpb = blockDim.x >> 6;
  const int l = lane % G;
  const int pair = (blockIdx.x * wpb + wv) * PPW + lane / G;  // lines 2 pair, 2 pair + 1
  const bool live = lane < PPW * G && 2 * pair < a.nlines;
  const int gl = live ? 2 * pair : 0;
  cplx<T>* ln = twl + N + (wv * PP::ROWS + lane / G) * LS;
  const bool stats = VAR == 1 || (VAR == 2 && a.want_stats);

  {
    const gptr<const cplx<T>> t = (gptr<const cplx<T>>)a.twX;
    for (int i = threadIdx.x; i < N; i += blockDim.x) twl[i] = gld<T>(t + i);
  }

  // ---- loads: the two lines' spectra at k = l + qG in X[f][q] and
  // X[f][E - QL + q], and (not PIN) at k = N/2 on lane 0
  const unsigned rowb = (unsigned)a.prow * ES;
  const unsigned lb = (unsigned)gl * rowb + (unsigned)l * ES;
  auto field = [&](const void* base, long stride, int f) {
    return make_brsrc(reinterpret_cast<const cplx<T>*>(base) + f * stride, a.fbytes);
  };
  cplx<T> X[NF][E], nyq[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const brsrc r = field(a.in, a.fstride_in, f);
#pragma unroll
    for (int q = 0; q < QL; ++q) {
      const unsigned off = live && l + q * G < a.kin ? lb + q * G * ES : kOob;
      X[f][q] = bld_s<T>(r, off, 0);
      X[f][E - QL + q] = bld_s<T>(r, off, rowb);
    }
    if constexpr (!PIN) {
      const unsigned off = live && l == 0 && N / 2 < a.kin ? lb + N / 2 * ES : kOob;
      const cplx<T> xa = bld_s<T>(r, off, 0), xb = bld_s<T>(r, off, rowb);
      nyq[f] = xa;  // (real part of line a, of line b); w below
      nyq[f].y = xb.x;
      if constexpr (NF == 6)
      if (f == 4 || f == 5) {  // w_y = A - i kx V_z, w_z = i kx V_y - B: real parts at k = N/2
        const T kx = (T)(a.kx_scale * double(N / 2));
        const brsrc rv = field(a.in, a.fstride_in, f == 4 ? 2 : 1);
        const cplx<T> va = bld_s<T>(rv, off, 0), vb = bld_s<T>(rv, off, rowb);
        nyq[f] = f == 4 ? mk<T>(xa.x + kx * va.y, xb.x + kx * vb.y) : mk<T>(-kx * va.y - xa.x, -kx * vb.y - xb.x);
      }
    }
  }
  if constexpr (PP::IDLE > 0) {  // the idle lanes' row (see PairPlan)
    if (lane >= PPW * G)
      for (int i = l; i < LS; i += PP::IDLE) ln[i] = mk<T>(T(0), T(0));
  }
  // Whether any line of the wave meets the mask.  The mask and us are read
  // through buffers, whose out-of-range offset stands for "not needed"; a line
  // whose flag says that its mask is all zero is not read.
  const brsrc rm = make_brsrc(a.mask, (unsigned)(a.npts * sizeof(T)));
  const unsigned pb = (unsigned)(gl * N + l) * (unsigned)sizeof(T);
  bool ma = live, mb = live;
  if (VAR < 3 && a.mflag) {
    ma = live && ((gptr<const uint8_t>)a.mflag)[gl] != 0;
    mb = live && ((gptr<const uint8_t>)a.mflag)[gl + 1] != 0;
  }
  bool masked = ma || mb;
  if (VAR < 3 && !a.mflag) {  // no flags (members of a batch): the wave looks at its own points
    bool any = false;
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const unsigned pq = live ? pb + (unsigned)(q * G) * sizeof(T) : kOob;
      any = any || rld<T>(rm, pq) != T(0) || rld<T>(rm, pq + N * sizeof(T)) != T(0);
    }
    masked = any;
  }
  masked = __any(masked);

  __syncthreads();  // twiddle table (the only block-wide wait besides the statistics)

  // ---- Z = A + i B and its mirrored modes M = conj A + i conj B, then w_y, w_z
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int q = 0; q < QL; ++q) {
      cplx<T> xa = X[f][q], xb = X[f][E - QL + q];
      if (q == 0 && l == 0) { xa.y = T(0); xb.y = T(0); }  // a C2R transform ignores these (cof_p3dfft.f90:65-83)
      X[f][q] = mk<T>(xa.x - xb.y, xa.y + xb.x);
      X[f][E - QL + q] = mk<T>(xa.x + xb.y, xb.x - xa.y);
    }
  if constexpr (NF == 6)
#pragma unroll
  for (int q = 0; q < QL; ++q) {
    const T kx = (T)(a.kx_scale * double(l + q * G));
    const int m = E - QL + q;
    X[4][q] = sub(X[4][q], ik_p<T>(kx, X[2][q]));
    X[5][q] = sub(ik_p<T>(kx, X[1][q]), X[5][q]);
    X[4][m] = add(X[4][m], ik_p<T>(kx, X[2][m]));
    X[5][m] = sub(ik_p<T>(-kx, X[1][m]), X[5][m]);
  }

  // ---- C2R of the fields
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    // one field at a time: keeps the scheduler from interleaving the
    // independent transforms (their temporaries would exhaust the registers)
    __builtin_amdgcn_sched_barrier(0);
    int lo = l;
    asm volatile("" : "+v"(lo));
    if constexpr (PP::ROW0) {
      // the whole of Z goes to the row, from which the first stage reads
#pragma unroll
      for (int q = 0; q < QL; ++q) {
        ln[lp<T>(lo + q * G)] = X[f][q];
        ln[lp<T>(N - lo - q * G)] = X[f][E - QL + q];
      }
      if (lo == 0) ln[lp<T>(N / 2)] = PIN ? mk<T>(T(0), T(0)) : nyq[f];
      wave_sync();
    } else {
      // mode N - k of k = l + qG comes through the row: position p reads N - p
      // = (G - l) + (E - 1 - q) G
      cplx<T>* rw = ln + lp<T>(lo);
      const cplx<T>* mr = ln + lp<T>(G - lo);
  #pragma unroll
      for (int q = 0; q < QL; ++q) {
        if constexpr (split_rd<T, PP>()) rw[lp<T>(q * G)] = X[f][E - QL + q];
        else ln[lp<T>(lo + q * G)] = X[f][E - QL + q];
      }
      wave_sync();
  #pragma unroll
      for (int q = E - QL; q < E; ++q) {
        if constexpr (split_rd<T, PP>()) X[f][q] = mr[lp<T>((E - 1 - q) * G)];
        else X[f][q] = ln[lp<T>(G - lo + (E - 1 - q) * G)];
      }
      wave_sync();
      // lane 0's N - p = QL G was not written: k = N/2, or beyond the region
      if (l == 0) X[f][E - QL] = PIN ? mk<T>(T(0), T(0)) : nyq[f];
  #pragma unroll
      for (int q = QL; q < E - QL; ++q) X[f][q] = mk<T>(T(0), T(0));
    }
    pfft<T, PP, +1>(X[f], twl, ln, l);
    if constexpr (VAR == 3) {
      const gptr<T> o = (gptr<T>)a.out + f * a.fstride_out + (long)gl * N + l;
      if (live) {
#pragma unroll
        for (int q = 0; q < E; ++q) { o[q * G] = X[f][q].x; o[N + q * G] = X[f][q].y; }
      }
    }
  }
  if constexpr (VAR < 3) {

  // ---- u x w - chi (u - us) [+ sponge], in place: X[0..2] (and X[3..5])
  double umax2 = 0.0, fs[3] = {0.0, 0.0, 0.0}, fc[3] = {0.0, 0.0, 0.0};
  if (stats && live) {
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const double ax = X[0][q].x, ay = X[1][q].x, az = X[2][q].x, bx = X[0][q].y, by = X[1][q].y, bz = X[2][q].y;
      umax2 = nanmax(nanmax(umax2, ax * ax + ay * ay + az * az), bx * bx + by * by + bz * bz);
    }
  }
  // u x w in place of w (of u with the sponge, which needs w).  FP32-mixed:
  // in FP32, the precision of the transforms that produced u and w.
  constexpr int OF = SPONGE ? 0 : 3;  // the outputs' registers
  // The penalisation term - chi (u - us), in FP64 (chi = mask/eta is large at
  // small eta).  Most waves of a flow around a small body meet no mask.  A
  // rolled loop rotates the positions through the first register: unrolled,
  // the FP64 temporaries of several positions were live at once.
  auto cross = [&](int q, cplx<T> (&nl)[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      const int c1 = (c + 1) % 3, c2 = (c + 2) % 3;
      const cplx<T> u1 = X[c1][q], u2 = X[c2][q], w1 = X[3 + c1][q], w2 = X[3 + c2][q];
      nl[c] = mk<T>(u1.x * w2.x - u2.x * w1.x, u1.y * w2.y - u2.y * w1.y);
    }
  };
  if (!SPONGE || !masked) {
#pragma unroll
    for (int q = 0; q < E; ++q) {
      cplx<T> nl[3];
      cross(q, nl);
#pragma unroll
      for (int c = 0; c < 3; ++c) X[OF + c][q] = nl[c];
    }
  }
  if (masked) {
    brsrc ru[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) ru[c] = make_brsrc((const T*)a.us + c * a.npts, (unsigned)(a.npts * sizeof(T)));
    cplx<T> mn = mk<T>(rld<T>(rm, ma ? pb : kOob), rld<T>(rm, mb ? pb + N * sizeof(T) : kOob));
    // (keeps the block before the loop, where the loop's copies of X belong:
    // merged with the branch's own block they were live on both paths)
    asm volatile("" : "+v"(mn.x), "+v"(mn.y));
#pragma unroll 1
    for (int q = 0; q < E; ++q) {
      const cplx<T> m = mn;
      const unsigned pq = pb + (unsigned)(q * G) * sizeof(T), pn = pq + G * sizeof(T);
      const bool more = q + 1 < E;
      mn = mk<T>(rld<T>(rm, ma && more ? pn : kOob), rld<T>(rm, mb && more ? pn + N * sizeof(T) : kOob));
      cplx<T> nl[3];
      if constexpr (SPONGE) cross(0, nl);
      else { nl[0] = X[3][0]; nl[1] = X[4][0]; nl[2] = X[5][0]; }
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        const double usa = rld<T>(ru[c], m.x != T(0) ? pq : kOob), usb = rld<T>(ru[c], m.y != T(0) ? pq + N * sizeof(T) : kOob);
        const double pa = (double)m.x * a.eps_inv * ((double)X[c][0].x - usa), pv = (double)m.y * a.eps_inv * ((double)X[c][0].y - usb);
        nl[c] = mk<T>((T)((double)nl[c].x - pa), (T)((double)nl[c].y - pv));
        if (stats && live) {
          double t = fs[c] + pa;
          fc[c] += (fabs(fs[c]) >= fabs(pa)) ? (fs[c] - t) + pa : (pa - t) + fs[c];
          fs[c] = t;
          t = fs[c] + pv;
          fc[c] += (fabs(fs[c]) >= fabs(pv)) ? (fs[c] - t) + pv : (pv - t) + fs[c];
          fs[c] = t;
        }
      }
#pragma unroll
      for (int f = 0; f < 6; ++f) {
        const int c = f - OF;
        const cplx<T> back = c >= 0 && c < 3 ? nl[c >= 0 && c < 3 ? c : 0] : X[f][0];
#pragma unroll
        for (int e = 0; e + 1 < E; ++e) X[f][e] = X[f][e + 1];
        X[f][E - 1] = back;
      }
    }
  }
  if constexpr (SPONGE) {  // -w / eta_sponge at the sponge's points, in place of w
    const int th = a.sponge_thickness;
    bool yz[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int iy = (gl + h) % a.ny, iz = (gl + h) / a.ny;
      yz[h] = a.sponge == 1 && (iy <= th - 1 || iy >= a.ny - th || iz <= th - 1 || iz >= a.nz - th);
    }
#pragma unroll
    for (int q = 0; q < E; ++q) {
      const int ix = l + q * G;
      const bool x = a.sponge == 1 ? N > 4 && (ix <= th - 1 || ix >= N - th) : a.sponge == 2 && ix >= N - th;
      const unsigned pq = pb + (unsigned)(q * G) * sizeof(T);
      const T m0 = rld<T>(rm, ma && masked ? pq : kOob), m1 = rld<T>(rm, mb && masked ? pq + N * sizeof(T) : kOob);
      const bool s0 = (x || yz[0]) && (double)m0 < a.sponge_mask_thr, s1 = (x || yz[1]) && (double)m1 < a.sponge_mask_thr;
#pragma unroll
      for (int c = 3; c < 6; ++c)
        X[c][q] = mk<T>(s0 ? (T)(-(double)X[c][q].x * a.sponge_eps_inv) : T(0), s1 ? (T)(-(double)X[c][q].y * a.sponge_eps_inv) : T(0));
    }
  }

  // ---- R2C of the outputs: A = (Z[k] + conj Z[N-k]) / 2, B = -i (Z[k] - conj Z[N-k]) / 2
  const T half = T(0.5);
#pragma unroll
  for (int c = 0; c < (SPONGE ? 6 : 3); ++c) {
    __builtin_amdgcn_sched_barrier(0);
    const int f = OF + c;
    if constexpr (PP::ROW0) {
#pragma unroll
      for (int q = 0; q < E; ++q) ln[lp<T>(l + q * G)] = X[f][q];
      wave_sync();
    }
    pfft<T, PP, -1>(X[f], twl, ln, l);
    int lo = l;
    asm volatile("" : "+v"(lo));
    cplx<T>* rw = ln + lp<T>(lo);
    const cplx<T>* mr = ln + lp<T>(G - lo);
#pragma unroll
    for (int q = E - QO; q < E; ++q) {
      if constexpr (split_rd<T, PP>()) rw[lp<T>(q * G)] = X[f][q];
      else ln[lp<T>(lo + q * G)] = X[f][q];
    }
    wave_sync();
    const brsrc r = field(a.out, a.fstride_out, c);
#pragma unroll
    for (int q = 0; q < QO; ++q) {
      const cplx<T> z = X[f][q];
      cplx<T> zm = split_rd<T, PP>() ? mr[lp<T>((E - 1 - q) * G)] : ln[lp<T>(G - lo + (E - 1 - q) * G)];
      if (q == 0 && l == 0) zm = z;
      const unsigned off = live && l + q * G < a.kout ? lb + q * G * ES : kOob;
      bst<T, 0>(r, off, mk<T>((z.x + zm.x) * half, (z.y - zm.y) * half));
      bst<T, 0>(r, off + rowb, mk<T>((z.y + zm.y) * half, (zm.x - z.x) * half));
    }
    if constexpr (PR < 2) {  // k = N/2: its own partner
      const cplx<T> z = X[f][H];
      const unsigned off = live && l == 0 && N / 2 < a.kout ? lb + N / 2 * ES : kOob;
      bst<T, 0>(r, off, mk<T>(z.x, T(0)));
      bst<T, 0>(r, off + rowb, mk<T>(z.y, T(0)));
    }
    wave_sync();
  }

  if (VAR > 0 && stats) {
    double v4[4] = {wmax(umax2), wsum(fs[0] + fc[0]), wsum(fs[1] + fc[1]), wsum(fs[2] + fc[2])};
    if (lane == 0) {
#pragma unroll
      for (int c = 0; c < 4; ++c) red[wv][c] = v4[c];
    }
    __syncthreads();
    if (threadIdx.x == 0) {
      double r[4] = {red[0][0], red[0][1], red[0][2], red[0][3]};
      for (int w = 1; w < wpb; ++w) {
        r[0] = nanmax(r[0], red[w][0]);
        for (int c = 1; c < 4; ++c) r[c] += red[w][c];
      }
      for (int c = 0; c < 4; ++c) ((gptr<double>)a.partial)[(long)blockIdx.x * 4 + c] = r[c];
    }
  }
  }  // VAR < 3
}

// Positions a lane.  Four keep every wave's instruction stream short and
// spread a small grid over more waves, eight exchange less through LDS (x
// pass, four / eight a lane: FP32 64^3 11.4 / 12.8 us, 128^3 29.0 / 26.4 us;
// FP32 96x64x64, four / twelve: 14.1 / 19.6 us).  FP64 keeps four up to nx = 256: eight
// positions of six fields leave no room for a second wave per SIMD without
// spills (64^3 13.2 / 13.9 us, 256x128x128 76 / 82 us).  The plan does not
// depend on the batch: a member's results are those of its own run.
int pair_e(int nx, long nlines, bool fp64) {
  const bool small = nlines * nx < (1L << 20);
  if (nx % 3 == 0) return nx == 96 && small ? 4 : 12;
  return nx <= 256 && (fp64 || small) ? 4 : 8;
}

// Waves of a block: four share a twiddle table; a grid that leaves compute
// units idle spreads its waves over more of them instead.
int pair_waves(int nx, long nlines, int e) {
  const long waves = (nlines / 2 * (nx / e) + 63) / 64;
  return waves >= 1024 ? XW_NT / 64 : 1;
}

template <typename T, int N, int E, int VAR, int PR, int NF = 6>
void run_pair(const XPassArgs& a, hipStream_t s) {
  using PP = PairPlan<N, E>;
  // with statistics one member's lines decide: the waves of a block are their
  // order of summation, which must not depend on the batch
  const bool stats = VAR == 1 || (VAR == 2 && a.want_stats);
  const int w = pair_waves(N, (long)a.nlines * (stats ? 1 : batch_n(a.bat)), E), ppb = w * PP::PPW;
  static_assert(pair_smem<T, PP>(XW_NT / 64) + sizeof(double) * XW_NT / 16 <= 65536, "LDS of a block");
  const int blocks = (a.nlines / 2 + ppb - 1) / ppb;
  const size_t smem = pair_smem<T, PP>(w);
  hipLaunchKernelGGL((x_rhs_pair_k<T, N, E, VAR, PR, NF>), dim3(blocks, batch_n(a.bat)), dim3(64 * w), smem, s, a);
}
// inv: the inverse transforms of that many fields alone (0: the right-hand side)
template <typename T, int N, int E>
void run_pair_e(const XPassArgs& a, int inv, hipStream_t s) {
  constexpr int KQ = PairPlan<N, E>::QL * PairPlan<N, E>::G;
  if (inv) {
    const bool pin = a.kin <= KQ;
    if (inv == 6) pin ? run_pair<T, N, E, 3, 1, 6>(a, s) : run_pair<T, N, E, 3, 0, 6>(a, s);
    else if (inv == 3) pin ? run_pair<T, N, E, 3, 1, 3>(a, s) : run_pair<T, N, E, 3, 0, 3>(a, s);
    else pin ? run_pair<T, N, E, 3, 1, 1>(a, s) : run_pair<T, N, E, 3, 0, 1>(a, s);
    return;
  }
  const int var = a.sponge ? 2 : (a.want_stats ? 1 : 0);
  const int pr = a.kin > KQ ? 0 : (a.kout > KQ ? 1 : 2);
  switch (3 * var + pr) {
    case 0: run_pair<T, N, E, 0, 0>(a, s); break;
    case 1: run_pair<T, N, E, 0, 1>(a, s); break;
    case 2: run_pair<T, N, E, 0, 2>(a, s); break;
    case 3: run_pair<T, N, E, 1, 0>(a, s); break;
    case 4: run_pair<T, N, E, 1, 1>(a, s); break;
    case 5: run_pair<T, N, E, 1, 2>(a, s); break;
    case 6: run_pair<T, N, E, 2, 0>(a, s); break;
    case 7: run_pair<T, N, E, 2, 1>(a, s); break;
    default: run_pair<T, N, E, 2, 2>(a, s); break;
  }
}
template <typename T, int N>
void run_pair_n(const XPassArgs& a, int inv, hipStream_t s) {
  const int e = pair_e(N, a.nlines, sizeof(T) == 8);
  if constexpr (N % 3 == 0) {
    if constexpr (N == 96) { if (e == 4) { run_pair_e<T, N, 4>(a, inv, s); return; } }
    run_pair_e<T, N, 12>(a, inv, s);
  } else if constexpr (N <= 256) {
    if constexpr (sizeof(T) == 4) { if (e == 8) { run_pair_e<T, N, 8>(a, inv, s); return; } }
    run_pair_e<T, N, 4>(a, inv, s);
  } else {
    run_pair_e<T, N, 8>(a, inv, s);
  }
}

}  // namespace

// Compiled in parts (per precision and family of lengths) for compile time.
template <typename T, int N, int... M>
static void pair_dispatch(const XPassArgs& a, int inv, hipStream_t s) {
  if (a.nx == N) run_pair_n<T, N>(a, inv, s);
  else if constexpr (sizeof...(M) > 0) pair_dispatch<T, M...>(a, inv, s);
  else throw std::runtime_error("in-wave x pass: unsupported nx " + std::to_string(a.nx));
}
void launch_pair_f32_2(const XPassArgs& a, int inv, hipStream_t s);
void launch_pair_f32_3(const XPassArgs& a, int inv, hipStream_t s);
void launch_pair_f64_2(const XPassArgs& a, int inv, hipStream_t s);
void launch_pair_f64_3(const XPassArgs& a, int inv, hipStream_t s);
#if FLUSI_PART == 0
void launch_pair_f32_2(const XPassArgs& a, int inv, hipStream_t s) { pair_dispatch<float, 32, 64, 128, 256, 512>(a, inv, s); }
#elif FLUSI_PART == 1
void launch_pair_f32_3(const XPassArgs& a, int inv, hipStream_t s) { pair_dispatch<float, 48, 96, 192, 384>(a, inv, s); }
#elif FLUSI_PART == 2
void launch_pair_f64_2(const XPassArgs& a, int inv, hipStream_t s) { pair_dispatch<double, 32, 64, 128, 256, 512>(a, inv, s); }
#elif FLUSI_PART == 3
void launch_pair_f64_3(const XPassArgs& a, int inv, hipStream_t s) { pair_dispatch<double, 48, 96, 192, 384>(a, inv, s); }
#endif

#if FLUSI_PART == 0
namespace {

// One wavefront per x line of the region: the line's flag is 1 where any of
// its nx mask values is nonzero (NaN included).  The wavefront returns as a
// whole (w depends on the wave only).
template <typename T>
__global__ __launch_bounds__(256) void mask_flags_k(const T* __restrict__ mask, uint8_t* __restrict__ flag, int nx, int ny,
                                                    int y0, int ey, int z0, long nl) {
  const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (w >= nl) return;
  const int lane = threadIdx.x & 63;
  const long line = (long)(z0 + (int)(w / ey)) * ny + (y0 + (int)(w % ey));
  const T* row = mask + line * nx;
  bool nzv = false;
  for (int i = lane; i < nx; i += 64) nzv = nzv || !(row[i] == T(0));
  const bool any = __any(nzv);
  if (lane == 0) flag[line] = any ? 1 : 0;
}

}  // namespace

template <typename T>
void launch_mask_flags(const void* mask, uint8_t* flag, int nx, int ny, int y0, int y1, int z0, int z1, hipStream_t s) {
  if (y1 < y0 || z1 < z0) return;
  const int ey = y1 - y0 + 1;
  const long nl = (long)ey * (z1 - z0 + 1);
  hipLaunchKernelGGL(mask_flags_k<T>, dim3((unsigned)((nl + 3) / 4)), dim3(256), 0, s, (const T*)mask, flag, nx, ny, y0,
                     ey, z0, nl);
}
template void launch_mask_flags<float>(const void*, uint8_t*, int, int, int, int, int, int, hipStream_t);
template void launch_mask_flags<double>(const void*, uint8_t*, int, int, int, int, int, int, hipStream_t);

bool x_rhs_wave_supported(int nx) {
  return nx == 32 || nx == 48 || nx == 64 || nx == 96 || nx == 128 || nx == 192 || nx == 256 || nx == 384 || nx == 512;
}

// with statistics: the rows of `partial` per member
int x_rhs_wave_blocks(int nx, int nlines, bool fp64) {
  const int e = pair_e(nx, nlines, fp64);
  const int ppb = pair_waves(nx, nlines, e) * (64 / (nx / e));
  return (nlines / 2 + ppb - 1) / ppb;
}

template <typename T>
static void launch_pair(const XPassArgs& a, int inv, hipStream_t s) {
  if (a.nlines % 2) throw std::runtime_error("in-wave x pass: the lines come in pairs");
  if (a.fbytes >= kOob || a.npts * (long)sizeof(T) >= (long)kOob)
    throw std::runtime_error("in-wave x pass: field too large for 32-bit offsets");
  if (a.nx % 3 == 0) sizeof(T) == 4 ? launch_pair_f32_3(a, inv, s) : launch_pair_f64_3(a, inv, s);
  else sizeof(T) == 4 ? launch_pair_f32_2(a, inv, s) : launch_pair_f64_2(a, inv, s);
}
template <typename T>
void launch_x_rhs_wave(const XPassArgs& a, hipStream_t s) {
  launch_pair<T>(a, 0, s);
}
template <typename T>
void launch_x_inv_wave(const XPassArgs& a, int mode, hipStream_t s) {
  if (mode == XM_INV ? (a.nf != 1 && a.nf != 3) : mode != XM_INV_UW) throw std::runtime_error("x inverse pass: nf must be 1 or 3");
  launch_pair<T>(a, mode == XM_INV ? a.nf : 6, s);
}
template void launch_x_rhs_wave<float>(const XPassArgs&, hipStream_t);
template void launch_x_rhs_wave<double>(const XPassArgs&, hipStream_t);
template void launch_x_inv_wave<float>(const XPassArgs&, int, hipStream_t);
template void launch_x_inv_wave<double>(const XPassArgs&, int, hipStream_t);
#endif

}  // namespace flusi
