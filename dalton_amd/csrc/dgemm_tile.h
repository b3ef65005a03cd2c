// Staging of FP64 block tiles (gfx950), shared by the GEMM launches and the
// (T) passes: operand order, LDS layouts and the global-load cursor.
#pragma once
#include "common.h"

namespace ccgpu {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));

enum { KFAST = 0, RFAST = 1 };  // loader order: k fastest / row (m or n) fastest

// K steps and LDS staging of a T x T block tile: TK columns of K per step, of
// which every thread stages EPT elements per operand.  Steps of 16 (32 tile:
// 32) are short enough that a product over K = v of a small molecule is not
// mostly padding, and leave the registers and LDS for more than two of the
// small tiles per CU: with steps twice as long, v^3 products at v = 93..170
// took 1.1-1.4x the time.  An operand loaded k-fastest is stored [row][k] with
// row stride TK + 2, one loaded row-fastest [k][row] with stride T + 16 (the
// 32 tile: stride 32, odd k with row bit 4 flipped); the 8-byte fragment
// reads of a half wave then fall on all 64 banks once.
template <int T>
struct Step {
  static constexpr int TK = T == 32 ? 32 : 16, EPT = T * TK / 256, LDK = TK + 2, LDR = T == 32 ? T : T + 16;
};
template <int MODE, int T>
struct Stage;
template <int T>
struct __attribute__((aligned(16))) Stage<KFAST, T> {
  double s[T * Step<T>::LDK];
  __device__ __forceinline__ double& at(int r, int k) { return s[r * Step<T>::LDK + k]; }
};
template <int T>
struct __attribute__((aligned(16))) Stage<RFAST, T> {
  double s[Step<T>::TK * Step<T>::LDR];
  __device__ __forceinline__ double& at(int r, int k) {
    return s[k * Step<T>::LDR + (T == 32 ? r ^ ((k & 1) << 4) : r)];
  }
};

// Element offset of k: two-level K by a multiply-high with the truncated
// 2^32 / Kin, at most 2^32 - 1 (the quotient is at most one short for k < 2^32).
struct KMap {
  long s_k, s_ko;
  unsigned Kin, magic;
};
template <bool K2>
__device__ __forceinline__ long koff(const KMap& m, long k) {
  if (!K2) return k * m.s_k;
  unsigned q = __umulhi((unsigned)k, m.magic), r = (unsigned)k - q * m.Kin;
  if (r >= m.Kin) {
    r -= m.Kin;
    ++q;
  }
  return (long)q * m.s_ko + (long)r * m.s_k;
}

// This thread's EPT elements of one K step of an operand tile whose first
// row is at base: k-fastest, column tid % TK of rows tid / TK + (256 / TK) i;
// row-fastest, row tid % T of columns tid / T + (256 / T) i.  One pointer per
// operand walks K (two-level K recomputes it per step) and the elements
// are uniform steps from it.  An element past the matrix (EDGE;
// rmax = last row of the tile inside it) re-reads a row inside it, whose
// results are never stored; only the last, partial step (TAIL) compares k
// with kend, re-reads a column inside and takes zeros.
template <int MODE, bool K2, int T, bool EDGE, typename P = const double*>
struct Cursor {
  static constexpr int TK = Step<T>::TK, NR = MODE == KFAST ? 256 / TK : 256 / T;
  P p;
  long s_r;
  KMap km;
  int r0, c0, rmax;

  __device__ __forceinline__ Cursor(P base, long sr, const KMap& m, int rm, long kbeg, int tid)
      : s_r(sr), km(m), rmax(rm) {
    r0 = MODE == KFAST ? tid / TK : tid % T;
    c0 = MODE == KFAST ? tid % TK : tid / T;
    if (EDGE) r0 = min(r0, rmax);
    p = base + r0 * s_r;
    if (!K2) p += (kbeg + c0) * km.s_k;
  }
  template <bool TAIL>
  __device__ __forceinline__ void load(double (&v)[Step<T>::EPT], long k0, long kend) {
    const long k = k0 + c0;
    if (MODE == KFAST) {
      P q = p;
      if (K2)
        q += koff<true>(km, TAIL ? min(k, kend - 1) : k);
      else if (TAIL && k >= kend)
        q -= (k - (kend - 1)) * km.s_k;
      const long st = NR * s_r;
      int r = r0;
#pragma unroll
      for (int i = 0; i < Step<T>::EPT; ++i) {
        v[i] = *q;
        if (EDGE) {
          r += NR;
          q += r <= rmax ? st : 0;
        } else {
          q += st;
        }
      }
      if (TAIL && k >= kend) {
#pragma unroll
        for (int i = 0; i < Step<T>::EPT; ++i) v[i] = 0.0;
      }
    } else if (K2) {
#pragma unroll
      for (int i = 0; i < Step<T>::EPT; ++i) {
        const long ki = k + NR * i;
        const double x = p[koff<true>(km, TAIL ? min(ki, kend - 1) : ki)];
        v[i] = (TAIL && ki >= kend) ? 0.0 : x;
      }
    } else {
      P q = p;
      if (TAIL && k >= kend) q -= (k - (kend - 1)) * km.s_k;
      const long st = NR * km.s_k;
#pragma unroll
      for (int i = 0; i < Step<T>::EPT; ++i) {
        const double x = *q;
        v[i] = (TAIL && k + NR * i >= kend) ? 0.0 : x;
        if (TAIL)
          q += k + NR * (i + 1) < kend ? st : 0;
        else
          q += st;
      }
    }
    if (!K2) p += TK * km.s_k;
  }
};

template <int MODE, int T>
__device__ __forceinline__ void stage_step(Stage<MODE, T>& S, const double (&v)[Step<T>::EPT], int tid) {
  constexpr int TK = Step<T>::TK;
#pragma unroll
  for (int i = 0; i < Step<T>::EPT; ++i) {
    if (MODE == KFAST)
      S.at(tid / TK + (256 / TK) * i, tid % TK) = v[i];
    else
      S.at(tid % T, tid / T + (256 / T) * i) = v[i];
  }
}

}  // namespace ccgpu
