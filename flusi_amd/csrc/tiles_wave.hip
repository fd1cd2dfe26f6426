// y and z tile passes (ZINV, YINV, YFWD, plain z forward) with every line
// transformed inside one wavefront, for line lengths 64, 96, 128, 192, 256,
// 384 and 512.
//
// A workgroup owns TL lines (16 FP32 / 8 FP64: 128-byte segments on the
// strided side) and one LDS row per line.  A line of L points lives in the
// registers of G = L/E lanes, lane l holding positions l + qG (q = 0..E-1,
// E = 8, or 12 where 3 divides L) before and after the transform; the Stockham
// stages exchange through the line's own LDS row with wave-scope ordering only.  The block
// waits twice per transform: once to turn the tile around between the
// contiguous side (a wave's own line) and the 128-byte segments of TL lines,
// and once before the tile is reused.  The next job's loads are issued as
// soon as the current operands are consumed.
//
// Bound by HBM from 128^3 on (4-5.4 TB/s).  The radix-3 lengths ran in block
// passes before, whose stages wait for the whole block: 96^3 FP32, two members,
// 38 -> 28 us, 192x96x384 FP32 z inverse 37 -> 26 us, y inverse 45 -> 40 us,
// 64x384x96 FP64 y inverse 65 -> 43 us; at a few thousand lines both forms
// take the latency of their stages (64x32x96 FP64: 15-16 us).
#include "fft_core.h"
#include "flusi_kernels.h"
#include "pass_common.h"
#include "wave_fft.h"
#include <type_traits>
#include <stdexcept>
#include <string>

namespace flusi {

namespace {

using namespace wavefft;

template <typename T> struct TWTile { static constexpr int TL = 16; };
template <> struct TWTile<double> { static constexpr int TL = 8; };

template <typename T, int L> struct TWShape {
  static constexpr int TL = TWTile<T>::TL;
  static constexpr int NW = TL / TWPlan<L>::LPW;     // waves per block
  static constexpr int NT = NW * 64;
  static constexpr int LS = line_stride<T>(L);
  static constexpr int K = TL * L / NT;              // tile elements per thread (E)
  // twiddles in LDS when two blocks still fit in 160 KB, and where the
  // registers hold one block to a compute unit anyway (FP64, L = 512: eight
  // waves of 168): from global memory each of the 14 a lane needs was waited
  // for by itself, and every such wait also covered the prefetched operands
  // (128x512x512 FP64 RK4 step, z / y inverse / y forward 685 / 1693 / 974 us,
  // from LDS 527 / 1303 / 743)
  static constexpr bool TWL = (sizeof(T) == 8 && L == 512) || 2 * (TL * LS + L) * (int)sizeof(cplx<T>) <= 160 * 1024;
  static constexpr size_t smem = (size_t)(TL * LS + (TWL ? L : 0)) * sizeof(cplx<T>);
};

template <typename T, int L>
__device__ __forceinline__ cplx<T> apply_op(int op, double kscale, int aa, cplx<T> x0, cplx<T> x1) {
  if (op == OP_COPY) return x0;
  const T k = (T)(kscale * double(aa < L / 2 ? aa : aa - L));
  cplx<T> x = mk<T>(-k * x0.y, k * x0.x);
  if (op == OP_DERIV_MINUS) x = sub(x, x1);
  return x;
}

// Loads and stores go through buffer descriptors (see make_brsrc): a line
// beyond the tile axis and a position outside the dealiased region are
// out-of-range offsets, so that no access carries a branch and the wait for
// the next job's prefetched operands does not have to cover the current job's
// stores (with a guard, the compiler cannot count the stores in flight and
// waits for all of them).
// PR: the pass is pruned (a.prune).  Full passes (small grids, undealiased
// states, transforms at the boundary) have kernels of their own, without the
// region's tests (512x64x64 FP32, forward y pass: 12.0 us with them, 11.3
// without).
template <typename T, int L, int S, bool CONTIG_IN, bool PR>
__global__ __launch_bounds__((TWShape<T, L>::NT)) void tile_wave_k(TilePassArgs a) {
  using Sh = TWShape<T, L>;
  constexpr int TL = Sh::TL, NT = Sh::NT, LS = Sh::LS, K = Sh::K;
  constexpr int G = TWPlan<L>::G, E = TWPlan<L>::E;
  constexpr unsigned ES = sizeof(cplx<T>);
  extern __shared__ char smem_raw[];
  cplx<T>* tile = reinterpret_cast<cplx<T>*>(smem_raw);
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int line = wv * TWPlan<L>::LPW + lane / G, l = lane % G;
  cplx<T>* ln = tile + line * LS;
  int b0 = blockIdx.x * TL, c = blockIdx.y;
  if (PR && a.tiles) {  // the tiles that meet the dealiased region
    const uint32_t t = ((gptr<const uint32_t>)a.tiles)[blockIdx.x];
    b0 = (int)(t & 0xffffu) * TL;
    c = (int)(t >> 16);
  }
  const int nbs = a.nb_store > a.nb ? a.nb_store : a.nb;  // lines >= nb hold zeros
  const long moff = (long)blockIdx.z * a.bat.mstride;  // batch member's slab
  const T sc = (T)a.scale;
  // twiddles: the block's LDS copy, or global memory where it does not fit
  std::conditional_t<Sh::TWL, const cplx<T>*, gptr<const cplx<T>>> tw;
  if constexpr (Sh::TWL) {
    cplx<T>* twl = tile + TL * LS;
    const gptr<const cplx<T>> twg = (gptr<const cplx<T>>)mshift(a.tw, moff);
    for (int i = tid; i < L; i += NT) twl[i] = gld<T>(twg + i);
    tw = twl;
    __syncthreads();
  } else {
    tw = (gptr<const cplx<T>>)mshift(a.tw, moff);
  }

  // This lane's line on the contiguous side: the byte offset of its position
  // 0, the shift of its upper half (positions L/2.., the negative wave
  // numbers) and what it holds.  Reading (CONTIG_IN): positions of |wave
  // number| <= lim.  Writing (PR_YFWD): compact positions [plo, phi).
  const int b = b0 + line;
  const bool lok = b < a.nb;
  int lim = lok ? L : -1, row = b;
  unsigned lo = 0, hi = 0;  // element shifts of the lower and the upper half
  int plo = 0, phi = 0;
  if (PR && CONTIG_IN && a.prune == PR_ZINV) {
    lim = ((gptr<const int16_t>)a.pr.zlim)[c * a.pr.nyp + b];
    row = b - a.pr.ym0;
    if (row < 0) row += a.nb;
  } else if (PR && CONTIG_IN && a.prune == PR_YINV) {
    lim = lok ? ((gptr<const int16_t>)a.pr.ylim)[b] : -1;
    lo = a.pr.ym0;
    hi = (unsigned)(a.pr.ym0 - L);
  } else if (PR && !CONTIG_IN && a.prune == PR_YFWD) {
    constexpr int SEG = 128 / ES;
    const int ym = lok ? ((gptr<const int16_t>)a.pr.ylim)[b] : -1;
    plo = (a.pr.ym0 - ym) & ~(SEG - 1);
    phi = lok ? min(a.pr.nyp, ((a.pr.ym0 + ym) | (SEG - 1)) + 1) : 0;
  }

  // operands: CONTIG_IN - the lane's E positions of its own line;
  // otherwise - the thread's K tile elements (bb = e % TL, a = e / TL)
  cplx<T> r0[E], r1[E];
  auto load = [&](int jb, int which) {
    const brsrc in = make_brsrc(mshift(which ? a.jobs[jb].in1 : a.jobs[jb].in0, moff), a.ibytes);
    if (CONTIG_IN) {
      const unsigned base = (unsigned)c * (unsigned)a.sin.c + (unsigned)row * (unsigned)a.sin.b + l;
      const unsigned line0 = lok ? base * ES : kOob;  // (a full pass; kOob + q G ES is out of range, too)
#pragma unroll
      for (int q = 0; q < E; ++q) {
        const int w = q < E / 2 ? l + q * G : L - l - q * G;  // |wave number|
        const unsigned off = !PR ? line0 + q * G * ES : (w <= lim ? (base + (q < E / 2 ? lo : hi) + q * G) * ES : kOob);
        const cplx<T> x = bld<T>(in, off);
        if (which) r1[q] = x; else r0[q] = x;
      }
    } else {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int e = tid + k * NT, bb = e % TL, aa = e / TL;
        const unsigned off = (unsigned)c * (unsigned)a.sin.c + (unsigned)(b0 + bb) + (unsigned)aa * (unsigned)a.sin.a;
        const cplx<T> x = bld<T>(in, b0 + bb < a.nb ? off * ES : kOob);
        if (which) r1[k] = x; else r0[k] = x;
      }
    }
  };

  // a job's operands (both inputs) are loaded while the previous job is
  // transformed and before its stores: a wait for them then never covers
  // stores in flight
  auto load_job = [&](int jb) {
    load(jb, 0);
    if (a.jobs[jb].in1) load(jb, 1);
  };
  load_job(0);
  for (int jb = 0; jb < a.njobs; ++jb) {
    const int nout = a.jobs[jb].out2 ? 2 : 1;
    for (int o = 0; o < nout; ++o) {
      const int op = o ? a.jobs[jb].op2 : a.jobs[jb].op;
      const brsrc out = make_brsrc(mshift(o ? a.jobs[jb].out2 : a.jobs[jb].out, moff), a.obytes);
      const bool pf = (o == nout - 1) && (jb + 1 < a.njobs);
      cplx<T> v[E];
      if (CONTIG_IN) {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = apply_op<T, L>(op, a.kscale, l + q * G, r0[q], r1[q]);
        if (pf) load_job(jb + 1);
        twfft<T, L, S>(v, tw, ln, l);
        // turn the tile: natural order into the line's row, then 128-byte
        // segments of TL lines out
#pragma unroll
        for (int q = 0; q < E; ++q) ln[lp<T>(l + q * G)] = v[q];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int e = tid + k * NT, bb = e % TL, aa = e / TL;
          const cplx<T> x = tile[bb * LS + lp<T>(aa)];
          const unsigned off = (unsigned)c * (unsigned)a.sout.c + (unsigned)(b0 + bb) + (unsigned)aa * (unsigned)a.sout.a;
          bst<T>(out, b0 + bb < nbs ? off * ES : kOob, mk<T>(x.x * sc, x.y * sc));
        }
        __syncthreads();
      } else {
#pragma unroll
        for (int k = 0; k < K; ++k) {
          const int e = tid + k * NT, bb = e % TL, aa = e / TL;
          tile[bb * LS + lp<T>(aa)] = apply_op<T, L>(op, a.kscale, aa, r0[k], r1[k]);
        }
        __syncthreads();
        if (pf) load_job(jb + 1);
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = ln[lp<T>(l + q * G)];
        wave_sync();
        twfft<T, L, S>(v, tw, ln, l);
        const unsigned base = (unsigned)c * (unsigned)a.sout.c + (unsigned)b * (unsigned)a.sout.b;
        const unsigned line0 = lok ? (base + l) * ES : kOob;
#pragma unroll
        for (int q = 0; q < E; ++q) {
          const int aa = l + q * G;
          unsigned off;
          if (PR && a.prune == PR_YFWD) {
            const int p = a.pr.ym0 + (q < E / 2 ? aa : aa - L);
            off = p >= plo && p < phi ? (base + (unsigned)p) * ES : kOob;
          } else {
            off = line0 + q * G * ES;
          }
          bst<T>(out, off, mk<T>(v[q].x * sc, v[q].y * sc));
        }
        __syncthreads();
      }
    }
  }
}

template <typename T, int L, int S, bool CI, bool PR>
void run_tw_pr(const TilePassArgs& a, hipStream_t s) {
  using Sh = TWShape<T, L>;
  static bool init = false;
  if (!init) { set_smem(tile_wave_k<T, L, S, CI, PR>, Sh::smem); init = true; }
  const dim3 grid = PR && a.tiles ? dim3(a.ntiles, 1, batch_n(a.bat))
                                  : dim3((a.nb + Sh::TL - 1) / Sh::TL, a.nc, batch_n(a.bat));
  hipLaunchKernelGGL((tile_wave_k<T, L, S, CI, PR>), grid, dim3(Sh::NT), Sh::smem, s, a);
}
template <typename T, int L, int S, bool CI>
void run_tw(const TilePassArgs& a, hipStream_t s) {
  if constexpr (CI == (S > 0)) {  // the pruned passes: inverse from lines, forward to lines
    if (a.prune) { run_tw_pr<T, L, S, CI, true>(a, s); return; }
  }
  run_tw_pr<T, L, S, CI, false>(a, s);
}

template <typename T, int L>
void run_tw_dir(const TilePassArgs& a, int dir, bool ci, hipStream_t s) {
  if (dir > 0) { if (ci) run_tw<T, L, +1, true>(a, s); else run_tw<T, L, +1, false>(a, s); }
  else { if (ci) run_tw<T, L, -1, true>(a, s); else run_tw<T, L, -1, false>(a, s); }
}

}  // namespace

int tile_lines(bool fp64) { return fp64 ? TWTile<double>::TL : TWTile<float>::TL; }

bool tile_wave_supported(int L) { return L == 64 || L == 96 || L == 128 || L == 192 || L == 256 || L == 384 || L == 512; }

template <typename T>
void launch_tile_wave(const TilePassArgs& a, int L, int dir, bool ci, hipStream_t s) {
  const bool unit = ci ? (a.sin.a == 1 && a.sout.b == 1) : (a.sin.b == 1 && a.sout.a == 1);
  if (!unit) throw std::runtime_error("tile pass: the contiguous axes must have unit stride");
  if (a.njobs < 1 || a.njobs > 6) throw std::runtime_error("tile pass: 1..6 jobs");
  if (a.prune && ci != (dir > 0)) throw std::runtime_error("tile pass: no such pruned pass");
  if (a.ibytes >= kOob || a.obytes >= kOob) throw std::runtime_error("tile pass: field too large for 32-bit offsets");
  switch (L) {
    case 64: run_tw_dir<T, 64>(a, dir, ci, s); break;
    case 96: run_tw_dir<T, 96>(a, dir, ci, s); break;
    case 128: run_tw_dir<T, 128>(a, dir, ci, s); break;
    case 192: run_tw_dir<T, 192>(a, dir, ci, s); break;
    case 256: run_tw_dir<T, 256>(a, dir, ci, s); break;
    case 384: run_tw_dir<T, 384>(a, dir, ci, s); break;
    case 512: run_tw_dir<T, 512>(a, dir, ci, s); break;
    default: throw std::runtime_error("in-wave tile pass: unsupported length " + std::to_string(L));
  }
}
template void launch_tile_wave<float>(const TilePassArgs&, int, int, bool, hipStream_t);
template void launch_tile_wave<double>(const TilePassArgs&, int, int, bool, hipStream_t);

}  // namespace flusi
