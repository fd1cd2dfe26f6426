// In-wave line transforms shared by the y/z tile passes (tiles_wave.hip) and
// the z-forward step pass (zstep.hip).
//
// A line of L points lives in the registers of G = L/E lanes, E = 8 (L = 64,
// 128, 256, 512) or 12 (L = 96, 192, 384), lane l holding positions l + qG
// (q = 0..E-1) before and after the transform.  Stockham stages exchange
// through the line's own LDS row with wave-scope ordering only.
#pragma once
#include "fft_core.h"

namespace flusi {
namespace wavefft {

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// radix plans: 512 = 8.8.8, 256 = 8.8.4, 128 = 8.4.4, 64 = 8.8; 384 = 12.4.4.2,
// 192 = 12.4.4, 96 = 12.4.2 (every radix divides E)
template <int L> struct TWPlan {
  static_assert(L == 64 || L == 128 || L == 256 || L == 512 || L == 96 || L == 192 || L == 384, "in-wave line length");
  static constexpr int E = L % 3 == 0 ? 12 : 8;
  static constexpr int G = L / E;      // lanes per line
  static constexpr int LPW = 64 / G;   // lines per wave
  static constexpr __host__ __device__ int radix(int s) {
    if (E == 12) return s == 0 ? 12 : (ns(s) * 4 <= L ? 4 : 2);
    return L == 256 ? (s == 2 ? 4 : 8) : (L == 128 ? (s == 0 ? 8 : 4) : 8);
  }
  static constexpr __host__ __device__ int ns(int s) { return s == 0 ? 1 : ns(s - 1) * radix(s - 1); }
};

template <int S, typename C> __device__ __forceinline__ C twm(C v, C w) {
  return (S < 0) ? cmul(v, w) : conjmul(v, w);
}

// Stage s: B = E/R butterflies per lane, j = l + bG; input q of butterfly b
// is register b + qB (position j + q L/R); outputs go to
// (j/Ns) Ns R + j%Ns + q Ns, which for the last stage is again register b + qB.
template <typename T, int L, int S, int s, typename TWP>
__device__ __forceinline__ void twstage(cplx<T> (&v)[TWPlan<L>::E], TWP tw, cplx<T>* ln, int l) {
  constexpr int E = TWPlan<L>::E, G = TWPlan<L>::G;
  constexpr int R = TWPlan<L>::radix(s), Ns = TWPlan<L>::ns(s), B = E / R;
  constexpr bool last = Ns * R == L;
#pragma unroll
  for (int b = 0; b < B; ++b) {
    // unsigned: j % Ns and j / Ns become a mask and a shift (l is an opaque
    // copy whose sign the compiler cannot see)
    const unsigned j = (unsigned)l + b * G;
    cplx<T> x[R];
#pragma unroll
    for (int q = 0; q < R; ++q) x[q] = v[b + q * B];
    if (s > 0) {
      const int step = (int)(j % Ns) * (L / (Ns * R));
#pragma unroll
      for (int q = 1; q < R; ++q) x[q] = twm<S>(x[q], twv<T>(tw, q * step));
    }
    Bfly<R, S, T>::run(x);
    if (last) {
#pragma unroll
      for (int q = 0; q < R; ++q) v[b + q * B] = x[q];
    } else {
      const int base = (int)(j / Ns) * Ns * R + (int)(j % Ns);
#pragma unroll
      for (int q = 0; q < R; ++q) ln[lp<T>(base + q * Ns)] = x[q];
    }
  }
  if constexpr (!last) {
    wave_sync();
#pragma unroll
    for (int r = 0; r < E; ++r) v[r] = ln[lp<T>(l + r * G)];
    wave_sync();
    twstage<T, L, S, s + 1>(v, tw, ln, l);
  }
}

template <typename T, int L, int S, typename TWP>
__device__ __forceinline__ void twfft(cplx<T> (&v)[TWPlan<L>::E], TWP tw, cplx<T>* ln, int l_) {
  int l = l_;
  asm volatile("" : "+v"(l));  // recompute addresses per transform (register pressure)
  twstage<T, L, S, 0>(v, tw, ln, l);
}

}  // namespace wavefft
}  // namespace flusi
