// (T) energy as one persistent kernel over a range of triples i >= j >= k
// (mlcc/mlccsdpt_e_calc.F90:71, loop :326-411; W as in w_calc :966, energy
// as in w_prod :1547-1640 and v_calc :1345, :1483-1527).
//
// A cooperative launch of as many blocks as the device holds at once walks
// the triples of the launch in order.  Per triple q three GEMM passes build
// W_q (G1: W[a][(b,c)] with beta = 0; G2: W[a][b][c] += ..., rows b, batched
// over a in the mixed passes, columns (a,c) in FP64;
// G3: W[(a,b)][c] += ...; four of the twelve terms each, one 128 x 128
// output tile per item) and an energy pass (E, one item per group of
// canonical 8x8x8 virtual blocks) reads it.  The passes form a software
// pipeline over the four W slots (triple q owns slot q mod 4): step s runs
//   E(s-3) | G3(s-2) | G2(s-1) | G1(s)
// and ends with one grid-wide barrier (cooperative groups), so every item
// depends only on items of earlier steps, and a triple costs one barrier.
// Items of a step are claimed dynamically, from one counter per XCD group
// that is never waited on; each group takes its range of energy items first
// (long items, started early) and then its ranges of the G3, G2 and G1 tiles
// (neighbouring tiles share operand panels, neighbouring canonical blocks W
// cache lines, in the XCD's L2).  The partial
// energies of a triple are summed in a fixed order by block 0 after the
// barrier that completes them.  Every block runs every barrier: the loop
// bounds depend only on the launch, and the runtime refuses a cooperative
// grid larger than what can be resident together.
//
// The energy pass reads W once: for canonical blocks A <= B <= C it stages
// the six block permutations of W, the eighteen 8x8 blocks of the (ia|jb)
// integrals and the t1 slices it needs in LDS and evaluates the
// permutation-symmetrised functional per orbit {a <= b <= c}.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include <hip/hip_cooperative_groups.h>

#include "bf16x3_tile.h"
#include "ccsd.h"
#include "dgemm_tile.h"
#include "kernels.h"
#include "ops.h"

namespace ccgpu {

namespace {

// ------------------------------------------------------------ FP64 tiles
// One term of a multi-term FP64 product: A(m,k) at A + m a_m + k a_k, B(n,k)
// at B + n b_n + k b_k.
struct DTerm {
  const double* A;
  const double* B;
  long a_m, a_k;
  long b_n, b_k;
  long K;
  double alpha;
  int akf;  // 1: A is read along k and B along n; 0: A along m and B along k
};
// C(m,n) (at C + m c_m + (n % nin) + (n / nin) c_no) = sum_t alpha_t A_t B_t^T + beta C
struct DMulti {
  DTerm t[4];
  int nterm;
  long M, N;
  double beta;
  double* C;
  long c_m, c_no;
  int nin;
};

namespace dt {
// Tile 128 x 128, K step 16, 256 threads; operands staged global -> registers ->
// LDS as in the FP64 GEMM (one pointer per operand walks K, rows past the
// matrix re-read a row inside it, only a last partial K step compares k with
// K), the next step's loads issued before the MFMAs.  LONG: the four waves lie
// side by side along the long dimension (n for X, m for !X): the other one is
// v, and its 16-row parts past v are left out of the products of all waves
// alike (2 x 2 waves: only the waves that own them, and the others set the
// time of a step; o=12 v=101 full list 17.5 against 16.0 ms).  A 64 x 64 tile
// with four blocks per CU took 16.8 ms.
constexpr int T = 128, TK = Step<T>::TK;
struct __attribute__((aligned(16))) Smem {
  static constexpr size_t N = std::max(sizeof(Stage<KFAST, T>), sizeof(Stage<RFAST, T>)) / sizeof(double);
  double A[N];
  double B[N];
};

// Waves of a tile and their 16 x 16 parts: all along the long side, or 2 x 2.
template <bool X, bool LONG>
struct Waves {
  static constexpr int WM = LONG ? (X ? 1 : 4) : 2, WN = 4 / WM, IM = T / 16 / WM, IN = T / 16 / WN;
};

// E: the tile reaches past M or N.
template <bool X, bool AKF, bool E, bool LONG>
__device__ __forceinline__ void term(const DTerm& t, int ma, int nb, long m0, long n0,
                                     d4 (&acc)[Waves<X, LONG>::IM][Waves<X, LONG>::IN], Smem& S) {
  using W = Waves<X, LONG>;
  constexpr int AM = AKF ? KFAST : RFAST, BM = AKF ? RFAST : KFAST, IM = W::IM, IN = W::IN;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // thread-index arithmetic stays inside the item (not hoisted into the claim loop)
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave / W::WN * (IM * 16), wn = wave % W::WN * (IN * 16);
  const int nv = (X ? ma : nb) / 16 + 1;  // 16-row parts inside the matrix
  const long K = t.K;
  const double al = t.alpha;
  using GP = const CCGPU_GLOBAL double*;
  Cursor<AM, false, T, E, GP> ca(gptr(t.A + m0 * t.a_m), t.a_m, KMap{t.a_k, 0, 0u, 0u}, ma, 0, tid);
  Cursor<BM, false, T, E, GP> cb(gptr(t.B + n0 * t.b_n), t.b_n, KMap{t.b_k, 0, 0u, 0u}, nb, 0, tid);
  Stage<AM, T>& SA = *reinterpret_cast<Stage<AM, T>*>(S.A);
  Stage<BM, T>& SB = *reinterpret_cast<Stage<BM, T>*>(S.B);
  double ra[Step<T>::EPT], rb[Step<T>::EPT];
  auto load = [&](long k0) {
    if (k0 + TK <= K) {
      ca.template load<false>(ra, k0, K);
      cb.template load<false>(rb, k0, K);
    } else {
      ca.template load<true>(ra, k0, K);
      cb.template load<true>(rb, k0, K);
    }
  };
  const int lr = lane & 15, lk = lane >> 4;
  load(0);
  for (long k0 = 0; k0 < K; k0 += TK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < Step<T>::EPT; ++i) ra[i] *= al;
    stage_step<AM, T>(SA, ra, tid);
    stage_step<BM, T>(SB, rb, tid);
    __syncthreads();
    if (k0 + TK < K) load(k0 + TK);
#pragma unroll
    for (int kk = 0; kk < TK / 4; ++kk) {
      if (k0 + kk * 4 >= K) break;
      double a[IM], b[IN];
#pragma unroll
      for (int u = 0; u < IM; ++u) a[u] = SA.at(wm + u * 16 + lr, kk * 4 + lk);
#pragma unroll
      for (int u = 0; u < IN; ++u) b[u] = SB.at(wn + u * 16 + lr, kk * 4 + lk);
#pragma unroll
      for (int i = 0; i < (X ? IM : IN); ++i) {
        if (E && LONG && i >= nv) break;
#pragma unroll
        for (int j = 0; j < (X ? IN : IM); ++j) {
          d4& c = X ? acc[i][j] : acc[j][i];
          c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[X ? i : j], b[X ? j : i], c, 0, 0, 0);
        }
      }
    }
  }
}

// Four terms, the first two read with A along k (X) or along m (!X), the
// other two the other way; the sequence is static so the accumulators stay
// in registers from term to term.
template <bool X, bool E, bool LONG>
__device__ __forceinline__ void tile4(const DMulti& p, long m0, long n0, Smem& S) {
  using W = Waves<X, LONG>;
  constexpr int IM = W::IM, IN = W::IN;
  d4 acc[IM][IN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < IN; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  const int ma = (int)min((long)T - 1, p.M - 1 - m0), nb = (int)min((long)T - 1, p.N - 1 - n0);
  term<X, X, E, LONG>(p.t[0], ma, nb, m0, n0, acc, S);
  term<X, X, E, LONG>(p.t[1], ma, nb, m0, n0, acc, S);
  term<X, !X, E, LONG>(p.t[2], ma, nb, m0, n0, acc, S);
  term<X, !X, E, LONG>(p.t[3], ma, nb, m0, n0, acc, S);
  __syncthreads();  // the next item reuses the LDS
  // D[i][j] of a 16x16 f64 MFMA tile: lane = j + 16*(i%4), element i/4.
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int wm = wave / W::WN * (IM * 16), wn = wave % W::WN * (IN * 16);
  // the descriptor's fields are read once (a store through C could alias them)
  CCGPU_GLOBAL double* C = gptr(p.C);
  const long c_m = p.c_m, c_no = p.c_no;
  const int nin = p.nin;
  const double beta = p.beta;
  long co[IN];  // column offsets, clamped into C
#pragma unroll
  for (int j = 0; j < IN; ++j) {
    const int n = (int)n0 + min(wn + j * 16 + lr, nb), q = n / nin;
    co[j] = q * c_no + (n - q * nin);
  }
  // per 16-row block: C read (beta != 0) before any of the block's stores,
  // so the loads overlap instead of each waiting behind a store
#pragma unroll
  for (int i = 0; i < IM; ++i) {
    if (E && wm + i * 16 > ma) break;
    double cv[IN][4] = {};
    if (beta != 0.0) {  // uniform; indices clamped into C: no per-element branch
#pragma unroll
      for (int j = 0; j < IN; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) cv[j][r] = C[(m0 + min(wm + i * 16 + r * 4 + lk, ma)) * c_m + co[j]];
    }
#pragma unroll
    for (int j = 0; j < IN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = wm + i * 16 + r * 4 + lk;
        if (m <= ma && wn + j * 16 + lr <= nb) {
          double v = acc[i][j][r];
          if (beta != 0.0) v += beta * cv[j][r];
          C[(m0 + m) * c_m + co[j]] = v;
        }
      }
  }
}
}  // namespace dt

// ------------------------------------------------------------ energy items
// Inputs of the energy evaluation of one triple.
struct EArgs {
  const int* ctab;  // canonical blocks A | B << 10 | C << 20
  const double* J;   // (ia|jb) as [(i,a)][(j,b)]
  const double* t1;  // [i][a]
  const double* eps;  // occupied first
  int o, v;
  long nE, nct;  // energy items (blocks) and canonical blocks
};

// LDS of an energy item of NT threads that stages NB canonical blocks at a
// time (block u of a round in w[u], jb[u], t1s[u], code[u]).
template <typename WT, int NB, int NT>
struct __attribute__((aligned(16))) ESmem {
  WT w[NB][6][8 * 72];     // block permutation p of W: [x][y][z] at x*72 + y*9 + z
  double jb[NB][18][64];   // (ia|jb) blocks: [m*6 + pair][r*8 + c]
  double t1s[NB][3][3][8];  // t1 of i, j, k over the blocks A, B, C
  double red[2][NT / 64];
};

// Positions (0 = A, 1 = B, 2 = C) of x, y, z in slot s: abc, acb, bac, bca, cab, cba.
__device__ constexpr int PX[6] = {0, 0, 1, 1, 2, 2};
__device__ constexpr int PY[6] = {1, 2, 0, 2, 0, 1};
__device__ constexpr int PZ[6] = {2, 1, 2, 0, 1, 0};
// index of the ordered position pair (u, w), u != w
__host__ __device__ constexpr int pair_ix(int u, int w) { return u * 2 + (w > u ? w - 1 : w); }

struct PtRun {
  const void* desc;  // three descriptors per triple (G1, G2, G3): BMulti or DMulti
  void* W;           // four slots of v^3 (float or double)
  long wslot;
  double* part;  // four slots of 2 nE energy partials
  double* etrip;  // (E4, E5) per triple of the launch
  unsigned long long* claims;  // one item counter per block group (zero at launch)
  const int* tri;  // (i, j, k) per triple
  EArgs e;
  long nq;
  long ng[3];        // items of G1, G2, G3
  long tm[3], tn[3];  // tiles per batch of G1, G2, G3 (m, n)
};

// Tile (tm, tn) of a linear index: groups of 8 m-tiles walked n-major, so
// consecutive claims share B panels.
__device__ __forceinline__ void tile_grouped(long t, long tiles_m, long tiles_n, long& tm, long& tn) {
  constexpr long GM = 8;
  const long grp = t / (GM * tiles_n);
  const long fm = grp * GM;
  const long gsz = min(tiles_m - fm, GM);
  const long r = t - grp * GM * tiles_n;
  tm = fm + r % gsz;
  tn = r / gsz;
}

// A block-uniform value read back from LDS, marked uniform so that what is
// derived from it (item, triple, descriptor address) stays in scalar registers.
__device__ __forceinline__ long uniform64(long x) {
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)(unsigned long)x);
  const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)((unsigned long)x >> 32));
  return (long)(((unsigned long)hi << 32) | lo);
}

// Energy item e of triple (i, j, k): canonical blocks e, e + nE, ..., NB
// of them staged per round (more loads in flight per barrier); NT threads.
// Writes its scaled (E4, E5) partial to part[2e], part[2e + 1].  With NB = 1
// the per-thread order of the sums is that of one block per round.
template <typename WT, int NB, int NT>
__device__ __forceinline__ void energy_item(const EArgs& r, const WT* W_, int i, int j, int k, long e, double* part,
                                            ESmem<WT, NB, NT>& S) {
  static_assert((NB * 512) % NT == 0 && NT % 64 == 0, "energy item: whole elements per thread");
  const int o = r.o, v = r.v;
  const CCGPU_GLOBAL WT* W = gptr(W_);
  const CCGPU_GLOBAL double* J = gptr(r.J);
  const CCGPU_GLOBAL double* t1 = gptr(r.t1);
  const CCGPU_GLOBAL double* eps = gptr(r.eps);
  const CCGPU_GLOBAL int* ctab = gptr(r.ctab);
  const long nov = (long)o * v, vv = (long)v * v;
  int tid = threadIdx.x;
  asm volatile("" : "+v"(tid));  // thread-index arithmetic stays inside the item
  const double eijk = eps[i] + eps[j] + eps[k];
  const bool vec = (v % 4) == 0;
  const long nE = r.nE, nct = r.nct;
  double s4 = 0.0, s5 = 0.0;
  for (long ct0 = e; ct0 < nct; ct0 += (long)NB * nE) {
    // the round's canonical blocks (-1 past the list), block-uniform
    int codes[NB];
#pragma unroll
    for (int u = 0; u < NB; ++u) {
      const long ct = ct0 + (long)u * nE;
      codes[u] = ct < nct ? ctab[ct] : -1;
    }
    auto code_of = [&](int u) {  // selects, no indexed local array
      int c = codes[0];
#pragma unroll
      for (int q = 1; q < NB; ++q) c = (u == q) ? codes[q] : c;
      return c;
    };
    // Every global load of the round is issued into registers first (fixed
    // trip counts, fully unrolled), then written to LDS after the barrier
    // that ends the previous round's reads: the loads overlap each other and
    // that round's tail, instead of each waiting before its LDS store.
    // six W block permutations per block: 384 rows of 8
    constexpr int WIT = (NB * 384 + NT - 1) / NT, JIT = (NB * 18 * 64 + NT - 1) / NT, TIT = (NB * 72 + NT - 1) / NT;
    WT wv[WIT][8];
#pragma unroll
    for (int it = 0; it < WIT; ++it) {
      const int row = tid + it * NT;
#pragma unroll
      for (int z = 0; z < 8; ++z) wv[it][z] = (WT)0;
      if (row < NB * 384) {
        const int u = row / 384, rr = row - u * 384;
        const int code = code_of(u);
        const int b0 = code & 1023, b1 = (code >> 10) & 1023, b2 = (code >> 20) & 1023;
        auto blk = [&](int q) { return q == 0 ? b0 : (q == 1 ? b1 : b2); };  // selects, no indexed local array
        const int p = rr >> 6, x8 = (rr >> 3) & 7, y8 = rr & 7;
        const int px = p >> 1, lo = px == 0 ? 1 : 0, hi = px == 2 ? 1 : 2;
        const int py = (p & 1) ? hi : lo, pz = (p & 1) ? lo : hi;
        const long gx = blk(px) * 8 + x8, gy = blk(py) * 8 + y8, z0 = blk(pz) * 8;
        if (code >= 0 && gx < v && gy < v) {
          const CCGPU_GLOBAL WT* src = W + gx * vv + gy * v + z0;
          if (vec && z0 + 8 <= v) {
            if (sizeof(WT) == 4) {
              const f4 x0 = *reinterpret_cast<const CCGPU_GLOBAL f4*>(src);
              const f4 x1 = *reinterpret_cast<const CCGPU_GLOBAL f4*>(src + 4);
#pragma unroll
              for (int h = 0; h < 4; ++h) {
                wv[it][h] = (WT)x0[h];
                wv[it][4 + h] = (WT)x1[h];
              }
            } else {
#pragma unroll
              for (int h = 0; h < 4; ++h) {
                const d2 x = *reinterpret_cast<const CCGPU_GLOBAL d2*>(src + 2 * h);
                wv[it][2 * h] = (WT)x[0];
                wv[it][2 * h + 1] = (WT)x[1];
              }
            }
          } else {
#pragma unroll
            for (int z = 0; z < 8; ++z) wv[it][z] = (z0 + z < v) ? src[z] : (WT)0;
          }
        }
      }
    }
    // (ia|jb) blocks: m = 0 J_jk[y][z], 1 J_ik[x][z], 2 J_ij[x][y]; pair (u, w) of positions
    double jv[JIT];
#pragma unroll
    for (int it = 0; it < JIT; ++it) {
      const int q = tid + it * NT;
      jv[it] = 0.0;
      if (q < NB * 18 * 64) {
        const int u = q / (18 * 64), qq = q - u * (18 * 64);
        const int code = code_of(u);
        const int b0 = code & 1023, b1 = (code >> 10) & 1023, b2 = (code >> 20) & 1023;
        auto blk = [&](int x) { return x == 0 ? b0 : (x == 1 ? b1 : b2); };
        const int b = qq >> 6, m = b / 6, pi = b - m * 6;
        const int pu = pi >> 1, wi = pi & 1, pw = wi + (wi >= pu ? 1 : 0);
        const int rr = (qq >> 3) & 7, cc = qq & 7;
        const int p1 = m == 0 ? j : i, p2 = m == 2 ? j : k;
        const long row = blk(pu) * 8 + rr, col = blk(pw) * 8 + cc;
        if (code >= 0 && row < v && col < v) jv[it] = J[((long)p1 * v + row) * nov + (long)p2 * v + col];
      }
    }
    double tv[TIT];
#pragma unroll
    for (int it = 0; it < TIT; ++it) {
      const int q = tid + it * NT;
      tv[it] = 0.0;
      if (q < NB * 72) {
        const int u = q / 72, qq = q - u * 72;
        const int code = code_of(u);
        const int b0 = code & 1023, b1 = (code >> 10) & 1023, b2 = (code >> 20) & 1023;
        const int m = qq / 24, pu = (qq / 8) % 3, x8 = qq & 7;
        const long x = (pu == 0 ? b0 : (pu == 1 ? b1 : b2)) * 8 + x8;
        const int om = m == 0 ? i : (m == 1 ? j : k);
        if (code >= 0 && x < v) tv[it] = t1[(long)om * v + x];
      }
    }
    __syncthreads();  // the previous round's LDS reads are done
#pragma unroll
    for (int it = 0; it < WIT; ++it) {
      const int row = tid + it * NT;
      if (row < NB * 384) {
        const int u = row / 384, rr = row - u * 384;
        const int p = rr >> 6, x8 = (rr >> 3) & 7, y8 = rr & 7;
        WT* dst = &S.w[u][p][x8 * 72 + y8 * 9];
#pragma unroll
        for (int z = 0; z < 8; ++z) dst[z] = wv[it][z];
      }
    }
#pragma unroll
    for (int it = 0; it < JIT; ++it) {
      const int q = tid + it * NT;
      if (q < NB * 18 * 64) {
        const int u = q / (18 * 64), qq = q - u * (18 * 64);
        const int b = qq >> 6, rr = (qq >> 3) & 7, cc = qq & 7;
        S.jb[u][b][rr * 8 + cc] = jv[it];
      }
    }
#pragma unroll
    for (int it = 0; it < TIT; ++it) {
      const int q = tid + it * NT;
      if (q < NB * 72) {
        const int u = q / 72, qq = q - u * 72;
        const int m = qq / 24, pu = (qq / 8) % 3, x8 = qq & 7;
        S.t1s[u][m][pu][x8] = tv[it];
      }
    }
    __syncthreads();
#pragma unroll
    for (int h = 0; h < NB * 512 / NT; ++h) {
      const int el = tid + NT * h;
      const int u = el >> 9, l0 = (el >> 6) & 7, l1 = (el >> 3) & 7, l2 = el & 7;
      const int code = code_of(u);
      if (code < 0) continue;
      const int b0 = code & 1023, b1 = (code >> 10) & 1023, b2 = (code >> 20) & 1023;
      auto loc = [&](int x) { return x == 0 ? l0 : (x == 1 ? l1 : l2); };
      const int a = b0 * 8 + l0, b = b1 * 8 + l1, c = b2 * 8 + l2;
      if (!(a <= b && b <= c && c < v)) continue;
      double w[6], y[6];
#pragma unroll
      for (int s = 0; s < 6; ++s) {
        const int xl = loc(PX[s]), yl = loc(PY[s]), zl = loc(PZ[s]);
        w[s] = (double)S.w[u][s][xl * 72 + yl * 9 + zl];
        y[s] = S.t1s[u][0][PX[s]][xl] * S.jb[u][pair_ix(PY[s], PZ[s])][yl * 8 + zl] +
               S.t1s[u][1][PY[s]][yl] * S.jb[u][6 + pair_ix(PX[s], PZ[s])][xl * 8 + zl] +
               S.t1s[u][2][PZ[s]][zl] * S.jb[u][12 + pair_ix(PX[s], PY[s])][xl * 8 + yl];
      }
      // slots 0 abc, 1 acb, 2 bac, 3 bca, 4 cab, 5 cba; even class {0,3,4}, odd {1,2,5}
      const double wE = w[0] + w[3] + w[4], wO = w[1] + w[2] + w[5];
      const double yE = y[0] + y[3] + y[4], yO = y[1] + y[2] + y[5];
      double ww = 0.0, wy = 0.0;
#pragma unroll
      for (int s = 0; s < 6; ++s) {
        ww += w[s] * w[s];
        wy += w[s] * y[s];
      }
      // sum over the 6 slots of W_p (4X_p + X_cyc1 + X_cyc2 - 2 X_swaps)
      const double f4 = 3.0 * ww + 3.0 * (wE * wE + wO * wO) - 2.0 * (wE + wO) * (wE + wO);
      const double f5 = 3.0 * wy + 3.0 * (wE * yE + wO * yO) - 2.0 * (wE + wO) * (yE + yO);
      // each distinct tuple once: slots alias when indices coincide
      const double wt = (a == b && b == c) ? (1.0 / 6.0) : ((a == b || b == c) ? 0.5 : 1.0);
      const double rD = wt / (eijk - eps[o + a] - eps[o + b] - eps[o + c]);
      s4 += f4 * rD;
      s5 += f5 * rD;
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    s4 += __shfl_down(s4, off, 64);
    s5 += __shfl_down(s5, off, 64);
  }
  const int lane = tid & 63, wv = tid >> 6;
  __syncthreads();
  if (lane == 0) {
    S.red[0][wv] = s4;
    S.red[1][wv] = s5;
  }
  __syncthreads();
  if (tid == 0) {
    // (i == j or j == k) counts the triple 3 times, otherwise 6: scale mult / 3
    const double scale = (i == j || j == k) ? 1.0 : 2.0;
    double r4 = S.red[0][0], r5 = S.red[1][0];
#pragma unroll
    for (int q = 1; q < NT / 64; ++q) {
      r4 += S.red[0][q];
      r5 += S.red[1][q];
    }
    part[2 * e] = scale * r4;
    part[2 * e + 1] = scale * r5;
  }
}

// (E4, E5) of one triple = sum of its nE partials in a fixed order (NT threads).
template <int NT>
__device__ __forceinline__ void reduce_partials(const double* part, long nE, double* out, double (&red)[2][NT / 64]) {
  const int tid = threadIdx.x;
  double s4 = 0.0, s5 = 0.0;
  for (long q = tid; q < nE; q += NT) {
    s4 += part[2 * q];
    s5 += part[2 * q + 1];
  }
  for (int off = 32; off > 0; off >>= 1) {
    s4 += __shfl_down(s4, off, 64);
    s5 += __shfl_down(s5, off, 64);
  }
  const int lane = tid & 63, wv = tid >> 6;
  __syncthreads();
  if (lane == 0) {
    red[0][wv] = s4;
    red[1][wv] = s5;
  }
  __syncthreads();
  if (tid == 0) {
    double r4 = red[0][0], r5 = red[1][0];
#pragma unroll
    for (int q = 1; q < NT / 64; ++q) {
      r4 += red[0][q];
      r5 += red[1][q];
    }
    out[0] = r4;
    out[1] = r5;
  }
}

// One GEMM tile (item t of pass ph of triple q) into W slot q mod 4.
template <bool MIXED>
__device__ __forceinline__ void pass_tile(const PtRun& r, long q, int ph, long t, unsigned char* lds) {
  const long tmn = r.tm[ph] * r.tn[ph];
  const long z = t / tmn;
  long tmi, tni;
  tile_grouped(t - z * tmn, r.tm[ph], r.tn[ph], tmi, tni);
  if constexpr (MIXED) {
    const BMulti& d = static_cast<const BMulti*>(r.desc)[q * 3 + ph];
    bf3w8::tile<float, true>(d, tmi * bf3w8::DT, tni * bf3w8::DT, z, *reinterpret_cast<bf3w8::Smem*>(lds));
  } else {
    const DMulti& d = static_cast<const DMulti*>(r.desc)[q * 3 + ph];
    dt::Smem& GS = *reinterpret_cast<dt::Smem*>(lds);
    const long m0 = tmi * 128, n0 = tni * 128;
    const bool inside = m0 + 128 <= d.M && n0 + 128 <= d.N;
    if (ph < 2) {
      if (inside)
        dt::tile4<true, false, true>(d, m0, n0, GS);
      else
        dt::tile4<true, true, true>(d, m0, n0, GS);
    } else {
      if (inside)
        dt::tile4<false, false, true>(d, m0, n0, GS);
      else
        dt::tile4<false, true, true>(d, m0, n0, GS);
    }
  }
}

// Dynamic claims per block group.  Blocks run on XCD b mod 8, so the items
// of a phase are cut into min(8, nb) contiguous ranges, one per group of
// blocks b = x (mod groups), and the group's blocks claim the items of their
// range from the group's counter (neighbouring tiles then share operand
// panels in one XCD's L2, and a slow item delays nothing else).  Each block
// of a group makes exactly one claim past the range per phase, so the
// counter advances by (range + blocks in the group) per phase and every
// block knows its base without reading it; claims never wait on other
// blocks.
struct GroupClaims {
  unsigned long long* ctr;
  long G, x, nbx, base = 0;
  __device__ GroupClaims(unsigned long long* c, long b, long nb) : ctr(c) {
    G = nb < 8 ? nb : 8;
    x = b % G;
    nbx = (nb - x + G - 1) / G;
  }
  __device__ long lo(long T) const { return T * x / G; }
  __device__ long hi(long T) const { return T * (x + 1) / G; }
  // Next position in this group's list of count items, or -1 (then the
  // phase is done for this block).
  __device__ long next(long count, long* s_claim) {
    if (threadIdx.x == 0) s_claim[0] = (long)__hip_atomic_fetch_add(ctr + x, 1ull, __ATOMIC_RELAXED,
                                                                     __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const long c = uniform64(s_claim[0]) - base;
    __syncthreads();
    return c < count ? c : -1;
  }
  __device__ void end_phase(long count) { base += count + nbx; }
};

// Block shape of the persistent kernel: the mixed path runs 256 x 256 tiles
// with eight waves (one block per CU) and stages two canonical blocks per
// energy round (at o=64 v=512: 1.2% faster than four, 3% faster than one);
// the FP64 path 128 x 128 tiles with four waves (two blocks per CU), one
// canonical block per round.
template <bool MIXED>
struct PtShape {
  static constexpr int NT = MIXED ? 512 : 256;
  static constexpr int NB = MIXED ? 2 : 1;
  static constexpr int TILE = MIXED ? bf3w8::DT : 128;
};

template <bool MIXED>
// The launch block is read through a pointer: its fields are re-read per
// item instead of being held in registers across the GEMM loops.
__global__ __launch_bounds__(PtShape<MIXED>::NT, MIXED ? 1 : 2) void k_pt_persistent(const PtRun* rp) {
  constexpr int NT = PtShape<MIXED>::NT, NB = PtShape<MIXED>::NB;
  const PtRun& r = *rp;
  using WT = typename std::conditional<MIXED, float, double>::type;
  using ES_t = ESmem<WT, NB, NT>;
  constexpr size_t SG = MIXED ? sizeof(bf3w8::Smem) : sizeof(dt::Smem);
  constexpr size_t SE = sizeof(ES_t);
  __shared__ __attribute__((aligned(16))) unsigned char lds[SG > SE ? SG : SE];
  ES_t& ES = *reinterpret_cast<ES_t*>(lds);
  __shared__ long s_claim[1];
  cooperative_groups::grid_group grid = cooperative_groups::this_grid();
  const long nE = r.e.nE, nq = r.nq;
  const long b0 = blockIdx.x;
  GroupClaims gc(r.claims, b0, gridDim.x);
  // step s: E(s-3) | G3(s-2) | G2(s-1) | G1(s), one grid barrier per step
  for (long st = 0; st < nq + 3; ++st) {
    if (st >= 4 && b0 == 0) {  // energy of triple st-4 (finished in step st-1), partials in a fixed order
      const long p = st - 4;
      reduce_partials<NT>(r.part + (p & 3) * 2 * nE, nE, r.etrip + 2 * p, ES.red);
      __syncthreads();
    }
    const long qe = st - 3;
    const long ne = (qe >= 0 && qe < nq) ? nE : 0;
    const long ne_x = gc.hi(ne) - gc.lo(ne);
    long cnt[3];
    for (int ph = 0; ph < 3; ++ph) {
      const long q = st - ph;
      const long T = (q >= 0 && q < nq) ? r.ng[ph] : 0;
      cnt[ph] = gc.hi(T) - gc.lo(T);
    }
    // this group's list: its range of energy items (long, claimed first; neighbouring canonical blocks
    // share W cache lines in the XCD's L2), then its ranges of the G3, G2 and G1 tiles
    const long n1 = ne_x + cnt[2] + cnt[1] + cnt[0];
    for (long c; (c = gc.next(n1, s_claim)) >= 0;) {
      if (c < ne_x) {
        const int* tq = r.tri + 3 * qe;
        const WT* W = static_cast<const WT*>(r.W) + (qe & 3) * r.wslot;
        energy_item<WT, NB, NT>(r.e, W, tq[0], tq[1], tq[2], gc.lo(ne) + c, r.part + (qe & 3) * 2 * nE, ES);
      } else {
        long k = c - ne_x;
        int ph = 2;
        while (k >= cnt[ph]) k -= cnt[ph--];
        const long q = st - ph;
        pass_tile<MIXED>(r, q, ph, gc.lo(r.ng[ph]) + k, lds);
      }
      __syncthreads();  // the next item reuses the LDS
    }
    gc.end_phase(n1);
    grid.sync();
  }
  if (b0 == 0 && nq >= 1) {  // energy of the last triple
    const long p = nq - 1;
    reduce_partials<NT>(r.part + (p & 3) * 2 * nE, nE, r.etrip + 2 * p, ES.red);
  }
}

// ------------------------------------------------ per-triple launches
// The same W passes and energy evaluation as plain launches (stream order
// instead of in-kernel dependencies).

// Tile and batch of block b of a triple, nx = grid_xcd(tiles) blocks a triple:
// each XCD (block b runs on XCD b % 8) gets a contiguous range of batches and,
// in a batch, of tiles walked in groups of 8 m-tiles, the same range for every
// triple.  false: a block past the range.
__device__ __forceinline__ bool tile_xcd(long b, long nx, long tiles_m, long tiles_n, long batch, long& tm, long& tn,
                                         long& z) {
  const long per = nx / 8, t = (b % 8) * per + b / 8, nt = tiles_m * tiles_n;
  if (t >= nt * batch) return false;
  z = t / nt;
  tile_grouped(t - z * nt, tiles_m, tiles_n, tm, tn);
  return true;
}
unsigned grid_xcd(long tiles) { return (unsigned)((tiles + 7) / 8 * 8); }

// One W pass of several triples: blockIdx.y takes the triple (its descriptor
// in list), blockIdx.x the tile.  Bound by the matrix cores once the chip is
// full, which a single triple's pass does not do below v = 256 (80 blocks at
// v = 101, 50 us a launch).  The full list at o=12 v=101, FP64: 87.9 ms in
// 1760 launches one triple at a time, 18.6 ms with 26 triples each, 16.0 with
// the columns of G2 flat (v batches of v x v pad both sides: 470 against 400
// us a launch) and the waves along the long side, 15.0 with 25 triples.
template <bool X, bool LONG>
__global__ __launch_bounds__(256, 2) void k_dtile4(const DMulti* list, long tiles_m, long tiles_n) {
  __shared__ dt::Smem S;
  const DMulti& p = list[blockIdx.y];
  long tm, tn, z;
  if (!tile_xcd(blockIdx.x, gridDim.x, tiles_m, tiles_n, 1, tm, tn, z)) return;
  const long m0 = tm * dt::T, n0 = tn * dt::T;
  if (m0 + dt::T <= p.M && n0 + dt::T <= p.N)
    dt::tile4<X, false, LONG>(p, m0, n0, S);
  else
    dt::tile4<X, true, LONG>(p, m0, n0, S);
}

// The mixed passes: the 256x256 tile (W8) or the 128x128 one.
template <bool W8>
__global__ __launch_bounds__(W8 ? 512 : 256, W8 ? 1 : 2) void k_btile4(const BMulti* list, long tiles_m, long tiles_n,
                                                                       long batch) {
  const BMulti& p = list[blockIdx.y];
  long tm, tn, z;
  if (!tile_xcd(blockIdx.x, gridDim.x, tiles_m, tiles_n, batch, tm, tn, z)) return;
  if constexpr (W8) {
    __shared__ bf3w8::Smem S;
    bf3w8::tile<float, true>(p, tm * bf3w8::DT, tn * bf3w8::DT, z, S);
  } else {
    __shared__ bf3::Smem<2> S;
    bf3::tile<float, 2>(p, tm * 128, tn * 128, z, S);
  }
}

// Item of block b: each XCD (block b runs on XCD b % 8) gets a contiguous
// range of items, whose canonical blocks are neighbours along C and share W
// cache lines in that XCD's L2 (the item's blocks, and so its partial, do not
// depend on the mapping).  Triple blockIdx.y of the group: its W slot and its
// nE partials.
template <typename WT>
__global__ __launch_bounds__(256) void k_pt_energy_blocked(EArgs a, const WT* W, long wslot, const int* tri,
                                                           double* part) {
  __shared__ ESmem<WT, 1, 256> S;
  const long b = blockIdx.x, per = (long)gridDim.x / 8, full = per * 8, t = blockIdx.y;
  energy_item<WT, 1, 256>(a, W + t * wslot, tri[3 * t], tri[3 * t + 1], tri[3 * t + 2],
                          (b < full) ? (b % 8) * per + b / 8 : b, part + 2 * a.nE * t, S);
}

__global__ __launch_bounds__(256) void k_reduce_pairs(const double* part, long n, double* out) {
  __shared__ double red[2][4];
  reduce_partials<256>(part + 2 * n * blockIdx.x, n, out + 2 * blockIdx.x, red);
}

__global__ void k_zero_u64(unsigned long long* p, int n) {
  if ((int)threadIdx.x < n) p[threadIdx.x] = 0ull;
}

// FP64 descriptor with every operand span checked.
DMulti d_desc(std::initializer_list<DTerm> terms, long M, long N, double* C, long c_m, long nin, long c_no,
              double beta) {
  DMulti p{};
  CCGPU_REQUIRE(terms.size() >= 1 && terms.size() <= 4, "pt: 1..4 terms");
  CCGPU_REQUIRE(N < (1L << 31) && nin > 0 && N % nin == 0, "pt: columns in whole rows of C");
  for (const DTerm& t : terms) {
    check_span(t.A, 0, (M - 1) * t.a_m + (t.K - 1) * t.a_k, sizeof(double), "pt A");
    check_span(t.B, 0, (N - 1) * t.b_n + (t.K - 1) * t.b_k, sizeof(double), "pt B");
    p.t[p.nterm++] = t;
  }
  CCGPU_REQUIRE(p.nterm == 4 && p.t[0].akf == p.t[1].akf && p.t[2].akf == p.t[3].akf && p.t[0].akf != p.t[2].akf,
                "pt: FP64 tiles take four terms in two read orders");
  p.M = M;
  p.N = N;
  p.beta = beta;
  p.C = C;
  p.c_m = c_m;
  p.c_no = c_no;
  p.nin = (int)nin;
  check_span(C, 0, (M - 1) * c_m + (N / nin - 1) * c_no + nin - 1, sizeof(double), "pt C");
  return p;
}

struct Resident {
  int blocks = 0;
};

template <bool MIXED>
int resident_blocks() {
  static Resident r;
  if (r.blocks == 0) {
    if (dryrun()) return 512;
    int dev = 0, per = 0;
    CCGPU_HIP(hipGetDevice(&dev));
    hipDeviceProp_t pr;
    CCGPU_HIP(hipGetDeviceProperties(&pr, dev));
    CCGPU_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k_pt_persistent<MIXED>, PtShape<MIXED>::NT, 0));
    r.blocks = std::max(1, per) * pr.multiProcessorCount;
  }
  return r.blocks;
}

// Bytes reserved for the launch block at the head of the descriptor buffer.
constexpr size_t kRunBytes = (sizeof(PtRun) + 255) / 256 * 256;

long env_long(const char* name, long dflt) {
  const char* e = std::getenv(name);
  return (e && *e) ? std::atol(e) : dflt;
}

// Tiles of the three W passes: G1 v x v^2, G2 v x v^2 (mixed: v batches of v x v), G3 v^2 x v.
struct PassShape {
  long M[3], N[3], tm[3], tn[3], batch[3], ng[3];
};
PassShape pass_shape(bool mixed, int v) {
  PassShape ps{};
  const long vv = (long)v * v;
  const long Ms[3] = {v, v, vv}, Ns[3] = {vv, mixed ? v : vv, v}, Bs[3] = {1, mixed ? v : 1, 1};
  for (int g = 0; g < 3; ++g) {
    // mixed: 256 x 256 tiles over operands padded to 256 rows; FP64: 128 x 128
    ps.tm[g] = mixed ? cdiv(bf16x3_rpad(Ms[g]), bf3w8::DT) : cdiv(Ms[g], 128);
    ps.tn[g] = mixed ? cdiv(bf16x3_rpad(Ns[g]), bf3w8::DT) : cdiv(Ns[g], 128);
    ps.M[g] = Ms[g];
    ps.N[g] = Ns[g];
    ps.batch[g] = Bs[g];
    ps.ng[g] = ps.tm[g] * ps.tn[g] * Bs[g];
  }
  return ps;
}

}  // namespace

size_t CCSD::pt_desc_bytes() const { return pt_mode_ == GemmPrec::BF16X3 ? sizeof(BMulti) : sizeof(DMulti); }

// Descriptors of the three W passes of triple (i, j, k) into W slot `slot`
// (BMulti for the mixed path, DMulti for FP64), every operand span checked.
void CCSD::pt_descs(int i, int j, int k, int slot, unsigned char* out) {
  const bool mixed = pt_mode_ == GemmPrec::BF16X3;
  const int o = dm_.o, v = dm_.v;
  const long nov = dm_.nov, vv = (long)v * v, vvv = vv * v;
  if (mixed) {
    const long Kpv = bf16x3_kpad(v), Kpo = bf16x3_kpad(o), Rv = bf16x3_rpad(v), Rvv = bf16x3_rpad(vv) + 256;
    const long gk = vv * Kpv, Kcv = bf16x3_kcols(v), Kco = bf16x3_kcols(o);
    auto Tm = [&](int p, int q, bool hi) { return (hi ? ppH_[0].p : ppL_[0].p) + ((long)p * o + q) * Rv * Kpv; };
    auto Qm = [&](int p, int q, bool hi) { return (hi ? ppH_[1].p : ppL_[1].p) + ((long)p * o + q) * Rv * Kpo; };
    auto Pm = [&](int p, bool hi) { return (hi ? ppH_[2].p : ppL_[2].p) + (long)p * Rvv * Kpo; };
    auto Sm = [&](int p, bool hi) { return (hi ? ppH_[3].p : ppL_[3].p) + (long)p * Rvv * Kpo; };
    auto TT = [&](int p, int q, const unsigned short* Bh, const unsigned short* Bl, long bbs) {  // T(p,q) x G
      return BTerm{Tm(p, q, true), Tm(p, q, false), Bh, Bl, Kpv, 0, bbs, Kcv};
    };
    auto QP = [&](int p, int q, const unsigned short* Bh, const unsigned short* Bl, long bbs) {  // Q_pq x Tvvo
      return BTerm{Qm(p, q, true), Qm(p, q, false), Bh, Bl, Kpo, 0, bbs, Kco};
    };
    float* Wq = W32_.p + slot * vvv;
    const unsigned short *GTk = GTh_.p + k * gk, *GTkl = GTl_.p + k * gk;
    BMulti* d = reinterpret_cast<BMulti*>(out);
    // G1: W[a][(b,c)] = t_ij^{ad} (bd|ck) + t_ik^{ad} (cd|bj) - (ai|lk) t_jl^{bc} - (ai|lj) t_kl^{cb}
    const BTerm g1[4] = {TT(i, j, GTk, GTkl, 0), TT(i, k, GpTh_.p + j * gk, GpTl_.p + j * gk, 0),
                         QP(i, k, Pm(j, true), Pm(j, false), 0), QP(i, j, Sm(k, true), Sm(k, false), 0)};
    d[0] = bf16x3_desc(g1, 4, v, vv, 1, Wq, true, vv, 1, 0, 1.0, 0.0);
    // G2 (batch a): W[a][b][c] += t_ji^{bd} (ad|ck) + t_jk^{bd} (cd|ai) - t_il^{ac} (bj|lk) - t_kl^{ca} (bj|li)
    const BTerm g2[4] = {TT(j, i, GTk, GTkl, v * Kpv), TT(j, k, GpTh_.p + i * gk, GpTl_.p + i * gk, v * Kpv),
                         QP(j, k, Pm(i, true), Pm(i, false), v * Kpo), QP(j, i, Sm(k, true), Sm(k, false), v * Kpo)};
    d[1] = bf16x3_desc(g2, 4, v, v, v, Wq, true, v, 1, vv, 1.0, 1.0);
    // G3: W[(a,b)][c] += (ad|bj) t_ki^{cd} + (bd|ai) t_kj^{cd} - t_il^{ab} (ck|lj) - t_jl^{ba} (ck|li)
    const BTerm g3[4] = {BTerm{GTh_.p + j * gk, GTl_.p + j * gk, Tm(k, i, true), Tm(k, i, false), Kpv, 0, 0, Kcv},
                         BTerm{GpTh_.p + i * gk, GpTl_.p + i * gk, Tm(k, j, true), Tm(k, j, false), Kpv, 0, 0, Kcv},
                         BTerm{Pm(i, true), Pm(i, false), Qm(k, j, true), Qm(k, j, false), Kpo, 0, 0, Kco},
                         BTerm{Sm(j, true), Sm(j, false), Qm(k, i, true), Qm(k, i, false), Kpo, 0, 0, Kco}};
    d[2] = bf16x3_desc(g3, 4, vv, v, 1, Wq, true, v, 1, 0, 1.0, 1.0);
  } else {
    auto Td = [&](int p, int q) { return T_.p + (long)p * v * nov + (long)q * v; };  // [x][d], row stride nov
    auto Qd = [&](int p, int q) { return Q_.p + ((long)p * o + q) * o * v; };       // [l][z]
    auto Pd = [&](int p) { return Tvvo_.p + (long)p * vv * o; };                    // [x][y][l]
    auto Sd = [&](int p) { return TvvoS_.p + (long)p * vv * o; };                   // [x][y][l] = Tvvo_p[y][x][l]
    double* Wq = Wt_.p + slot * vvv;
    const double* Gk = G_.p + (long)k * vvv;
    DMulti* d = reinterpret_cast<DMulti*>(out);
    // the same twelve terms; A read along k and B along n for the G terms of G1 and G2, the other way round
    // for their occupied terms; the reverse in G3
    d[0] = d_desc({DTerm{Td(i, j), Gk, nov, 1, 1, vv, v, 1.0, 1},
                   DTerm{Td(i, k), Gp_.p + (long)j * vvv, nov, 1, 1, vv, v, 1.0, 1},
                   DTerm{Qd(i, k), Pd(j), 1, v, o, 1, o, -1.0, 0},
                   DTerm{Qd(i, j), Sd(k), 1, v, o, 1, o, -1.0, 0}},
                  v, vv, Wq, vv, vv, 0, 0.0);
    // G2: the columns are (a, c), a slowest, as they lie in the B operands
    d[1] = d_desc({DTerm{Td(j, i), Gk, nov, 1, 1, vv, v, 1.0, 1},
                   DTerm{Td(j, k), Gp_.p + (long)i * vvv, nov, 1, 1, vv, v, 1.0, 1},
                   DTerm{Qd(j, k), Pd(i), 1, v, o, 1, o, -1.0, 0},
                   DTerm{Qd(j, i), Sd(k), 1, v, o, 1, o, -1.0, 0}},
                  v, vv, Wq, v, v, vv, 1.0);
    d[2] = d_desc({DTerm{G_.p + (long)j * vvv, Td(k, i), 1, vv, nov, 1, v, 1.0, 0},
                   DTerm{Gp_.p + (long)i * vvv, Td(k, j), 1, vv, nov, 1, v, 1.0, 0},
                   DTerm{Pd(i), Qd(k, j), o, 1, 1, v, o, -1.0, 1},
                   DTerm{Sd(j), Qd(k, i), o, 1, 1, v, o, -1.0, 1}},
                  vv, v, Wq, v, v, 0, 1.0);
  }
}

namespace {
EArgs energy_args(const int* ctab, const double* J, const double* t1, const double* eps, int o, int v) {
  const long nb = cdiv(v, 8), nct = nb * (nb + 1) * (nb + 2) / 6;
  return EArgs{ctab, J, t1, eps, o, v, std::min<long>(nct, 2048), nct};
}
}  // namespace

namespace {
// The 256 tile where its whole rounds of blocks (one a CU) take no longer than
// those of the 128 tile (two a CU), at 361 against 307 TFLOP/s in full rounds.
// A launch of few triples is a round or two, where padding to 256 rows and a
// part-filled chip matter less than a second round: with the area rule of the
// BF16x3 GEMM (and a full round of 256 tiles) one triple took 261 us at v = 200
// and 343 at v = 230, now 214 and 287; full groups take the same tile as before.
bool pt_large_tile(long t256, long t128) {
  if (bf16x3_rpad(1) != bf3w8::DT) return false;  // operands padded to 128 rows only
  return cdiv(t256, 256) * 4.0 / 361.0 <= cdiv(t128, 512) * 2.0 / 307.0;
}
}  // namespace

// Triples per launch of the W passes: just below four waves of blocks over the
// CUs (two 128 x 128 blocks or one 256 x 256 block per CU; just above, a fifth
// one is nearly empty: v=101 26 triples 16.0 ms the full list, 25 15.0), at
// most 64, with their W slots inside 256 MB, about what the last-level cache
// holds (G2, G3 and the energy re-read W).  One at v = 512.
long CCSD::pt_group(bool mixed) const {
  const PassShape ps = pass_shape(mixed, dm_.v);
  const long fewest = std::min(std::min(ps.ng[0], ps.ng[1]), ps.ng[2]), vvv = (long)dm_.v * dm_.v * dm_.v;
  const long fill = (mixed ? 1024 : 2048) / fewest;
  const long room = (256L << 20) / (vvv * (long)(mixed ? sizeof(float) : sizeof(double)));
  return std::max<long>(1, std::min<long>({fill, room, 64, pt_ntriples()}));
}

// (T) as launches per group of triples: three W passes, the blocked energy,
// the sums; the descriptors and indices of a range of triples are copied over
// before its launches.
void CCSD::pt_energy_launches(long first, long n, long stride, double* e4, double* e5) {
  const bool mixed = pt_mode_ == GemmPrec::BF16X3;
  const int o = dm_.o, v = dm_.v;
  const long vv = (long)v * v, vvv = vv * v;
  const EArgs ea = energy_args(ptctab_.p, J_.p, t1_.p, eps_.p, o, v);
  const PassShape ps = pass_shape(mixed, v);
  const long ng = pt_group(mixed);
  const void* W = mixed ? (const void*)W32_.p : (const void*)Wt_.p;
  check_span(ptpart_.p, 0, 2 * ea.nE * ng - 1, sizeof(double), "pt partials");
  check_span(ea.ctab, 0, ea.nct - 1, sizeof(int), "pt block table");
  check_span(ea.J, 0, dm_.nov2 - 1, sizeof(double), "pt J");
  check_span(W, 0, ng * vvv - 1, mixed ? sizeof(float) : sizeof(double), "pt W");
  etrip_.ensure(2 * (size_t)std::max<long>(n, 1));
  // flops of a pass of one triple: two K = v and two K = o terms
  const double fg = 2.0 * (2.0 * (double)vv * vv + 2.0 * (double)vv * v * o);
  constexpr long kRange = 4096;  // triples whose descriptors are held at once
  const long nr = std::min(n, kRange);
  const size_t dsz = pt_desc_bytes();
  const size_t dend = 3 * nr * dsz;  // the indices follow the descriptors: one copy
  if (n > 0) ptdesc_.ensure(dend + 3 * nr * sizeof(int));
  std::vector<unsigned char> hd(dend + 3 * nr * sizeof(int)), one(3 * dsz);
  int* const ht = reinterpret_cast<int*>(hd.data() + dend);
  const int* const tri = reinterpret_cast<const int*>(ptdesc_.p + dend);
  struct Drain {  // an error on the way leaves with the copy done
    hipStream_t s;
    ~Drain() {
      if (!dryrun()) (void)hipStreamSynchronize(s);
    }
  } drain{st_};
  for (long r0 = 0; r0 < n; r0 += kRange) {
    const long nq = std::min(kRange, n - r0);
    for (long q = 0; q < nq; ++q) {
      const long t = first + (r0 + q) * stride;
      const int i = tri_i_[t], j = tri_j_[t], k = tri_k_[t];
      ht[3 * q] = i;
      ht[3 * q + 1] = j;
      ht[3 * q + 2] = k;
      pt_descs(i, j, k, (int)(q % ng), one.data());
      for (int g = 0; g < 3; ++g) std::memcpy(hd.data() + (g * nr + q) * dsz, one.data() + g * dsz, dsz);
    }
    // the previous range's launches precede the copy on the stream, and the
    // host array is refilled only after the copy has left it
    CCGPU_HIPX(hipMemcpyAsync(ptdesc_.p, hd.data(), hd.size(), hipMemcpyHostToDevice, st_));
    if (r0 + nq < n) CCGPU_HIPX(hipStreamSynchronize(st_));
    for (long q0 = 0; q0 < nq; q0 += ng) {
      const unsigned gn = (unsigned)std::min(ng, nq - q0);
      for (int g = 0; g < 3; ++g) {
        const unsigned char* list = ptdesc_.p + (g * nr + q0) * dsz;
        const unsigned nb = (unsigned)ps.batch[g];
        CCGPU_REQUIRE(ps.tm[g] * ps.tn[g] * ps.batch[g] < (1L << 22), "pt: grid too large");
        if (mixed) {
          const BMulti* d = reinterpret_cast<const BMulti*>(list);
          const long tm1 = cdiv(ps.M[g], 128), tn1 = cdiv(ps.N[g], 128);
          const bool w8 = pt_large_tile(ps.tm[g] * ps.tn[g] * nb * gn, tm1 * tn1 * nb * gn);
          const int id = prof_begin("k_gemm_bf16x3", fg * gn, st_);
          if (w8)
            CCGPU_LAUNCH(k_btile4<true>, dim3(grid_xcd(ps.tm[g] * ps.tn[g] * nb), gn), dim3(512), 0, st_, d, ps.tm[g],
                         ps.tn[g], (long)nb);
          else
            CCGPU_LAUNCH(k_btile4<false>, dim3(grid_xcd(tm1 * tn1 * nb), gn), dim3(256), 0, st_, d, tm1, tn1, (long)nb);
          prof_end(id, st_);
        } else {
          const DMulti* d = reinterpret_cast<const DMulti*>(list);
          const dim3 grid(grid_xcd(ps.tm[g] * ps.tn[g] * nb), gn);
          const int id = prof_begin(g < 2 ? "k_dtile4<true>" : "k_dtile4<false>", fg * gn, st_);
          // The waves side by side read a quarter more from LDS (2 x 2 is 3% faster at v = 256, 384 and
          // 512): only where they leave out more than that of the 16-row parts.
          const long parts = cdiv(v, 16), all = 8L * cdiv(v, 128);
          const bool lng = 24 * (all - parts) >= all;
          auto* kern = g < 2 ? (lng ? k_dtile4<true, true> : k_dtile4<true, false>)
                             : (lng ? k_dtile4<false, true> : k_dtile4<false, false>);
          CCGPU_LAUNCH(kern, grid, dim3(256), 0, st_, d, ps.tm[g], ps.tn[g]);
          prof_end(id, st_);
        }
      }
      const int id = prof_begin(mixed ? "k_pt_energy_blocked<float>" : "k_pt_energy_blocked<double>", 0.0, st_);
      const dim3 egrid((unsigned)ea.nE, gn);
      if (mixed)
        CCGPU_LAUNCH(k_pt_energy_blocked<float>, egrid, dim3(256), 0, st_, ea, W32_.p, vvv, tri + 3 * q0,
                     ptpart_.p);
      else
        CCGPU_LAUNCH(k_pt_energy_blocked<double>, egrid, dim3(256), 0, st_, ea, Wt_.p, vvv, tri + 3 * q0,
                     ptpart_.p);
      prof_end(id, st_);
      CCGPU_LAUNCH(k_reduce_pairs, dim3(gn), dim3(256), 0, st_, ptpart_.p, ea.nE, etrip_.p + 2 * (r0 + q0));
      CCGPU_HIPX(hipGetLastError());
    }
  }
  double s4 = 0.0, s5 = 0.0;
  if (n > 0) {
    std::vector<double> et(2 * n, 0.0);
    CCGPU_HIPX(hipMemcpyAsync(et.data(), etrip_.p, 2 * n * sizeof(double), hipMemcpyDeviceToHost, st_));
    CCGPU_HIPX(hipStreamSynchronize(st_));
    for (long q = 0; q < n; ++q) {
      s4 += et[2 * q];
      s5 += et[2 * q + 1];
    }
  }
  if (e4) *e4 = s4;
  if (e5) *e5 = s5;
}

// Host side of the persistent (T): descriptors per triple, one cooperative
// launch over the whole range (CCGPU_PT_CHUNK=n: launches of n triples).
void CCSD::pt_energy_persistent(long first, long n, long stride, double* e4, double* e5) {
  const bool mixed = pt_mode_ == GemmPrec::BF16X3;
  const int o = dm_.o, v = dm_.v;
  const long vv = (long)v * v, vvv = vv * v;
  // the 256 x 256 tiles read whole 256-row panels: the packed operands must
  // be padded to 256 rows (the default BF16x3 block tile)
  CCGPU_REQUIRE(!mixed || (bf16x3_rpad(v) % bf3w8::DT == 0 && bf16x3_rpad(vv) % bf3w8::DT == 0),
                "persistent (T): the mixed path needs operands padded to 256 rows (CCGPU_BF16X3_VARIANT=1)");
  PtRun r{};
  r.W = mixed ? (void*)W32_.p : (void*)Wt_.p;
  r.wslot = vvv;
  r.part = ptpart_.p;
  r.e = energy_args(ptctab_.p, J_.p, t1_.p, eps_.p, o, v);
  const long nE = r.e.nE;
  check_span(r.W, 0, 4 * vvv - 1, mixed ? sizeof(float) : sizeof(double), "pt W slots");
  check_span(r.part, 0, 8 * nE - 1, sizeof(double), "pt partials");
  check_span(r.e.ctab, 0, r.e.nct - 1, sizeof(int), "pt block table");
  check_span(r.e.J, 0, dm_.nov2 - 1, sizeof(double), "pt J");
  const PassShape ps = pass_shape(mixed, v);
  for (int g = 0; g < 3; ++g) {
    r.tm[g] = ps.tm[g];
    r.tn[g] = ps.tn[g];
    r.ng[g] = ps.ng[g];
  }
  const double ftri = 12.0 * (double)vv * vv + 12.0 * (double)o * vvv;
  long chunk = env_long("CCGPU_PT_CHUNK", 0);
  if (chunk <= 0) chunk = std::max<long>(n, 1);  // the whole range in one cooperative launch
  etrip_.ensure(2 * (size_t)std::max<long>(n, 1));
  const size_t dsz = pt_desc_bytes();
  const long cq = std::min(chunk, std::max<long>(n, 1));
  ptdesc_.ensure(kRunBytes + 3 * cq * dsz);
  pttri_.ensure(3 * (size_t)cq);
  ptclaim_.ensure(8);
  std::vector<unsigned char> hd(kRunBytes + 3 * cq * dsz);
  std::vector<int> ht(3 * cq);
  double s4 = 0.0, s5 = 0.0;
  for (long c0 = 0; c0 < n; c0 += chunk) {
    const long nq = std::min(chunk, n - c0);
    for (long q = 0; q < nq; ++q) {
      const long t = first + (c0 + q) * stride;
      const int i = tri_i_[t], j = tri_j_[t], k = tri_k_[t];
      ht[3 * q] = i;
      ht[3 * q + 1] = j;
      ht[3 * q + 2] = k;
      pt_descs(i, j, k, (int)(q & 3), hd.data() + kRunBytes + 3 * q * dsz);
    }
    r.nq = nq;
    r.desc = ptdesc_.p + kRunBytes;
    r.tri = pttri_.p;
    r.claims = ptclaim_.p;
    r.etrip = etrip_.p + 2 * c0;
    check_span(r.etrip, 0, 2 * nq - 1, sizeof(double), "pt energies");
    std::memcpy(hd.data(), &r, sizeof(PtRun));
    CCGPU_HIPX(hipMemcpyAsync(ptdesc_.p, hd.data(), kRunBytes + 3 * nq * dsz, hipMemcpyHostToDevice, st_));
    CCGPU_HIPX(hipMemcpyAsync(pttri_.p, ht.data(), 3 * nq * sizeof(int), hipMemcpyHostToDevice, st_));
    check_span(ptclaim_.p, 0, 7, sizeof(unsigned long long), "pt claim counters");
    CCGPU_LAUNCH(k_zero_u64, dim3(1), dim3(64), 0, st_, ptclaim_.p, 8);
    const PtRun* run = reinterpret_cast<const PtRun*>(ptdesc_.p);
    // every block of a cooperative grid must be resident at once: at most
    // the occupancy limit, and no more blocks than the widest phase has items
    const long widest = nE + r.ng[0] + r.ng[1] + r.ng[2];  // items of one full pipeline step
    const long grid = std::max<long>(1, std::min<long>(widest, mixed ? resident_blocks<true>()
                                                                       : resident_blocks<false>()));
    const int id = prof_begin(mixed ? "k_pt_persistent<true>" : "k_pt_persistent<false>", (double)nq * ftri, st_);
    if (!dryrun()) {
      void* args[] = {(void*)&run};
      const void* fn = mixed ? reinterpret_cast<const void*>(&k_pt_persistent<true>)
                             : reinterpret_cast<const void*>(&k_pt_persistent<false>);
      CCGPU_HIP(hipLaunchCooperativeKernel(fn, dim3((unsigned)grid), dim3(mixed ? PtShape<true>::NT : PtShape<false>::NT),
                                           args, 0, st_));
    }
    prof_end(id, st_);
  }
  if (n > 0) {
    std::vector<double> et(2 * n, 0.0);
    CCGPU_HIPX(hipMemcpyAsync(et.data(), etrip_.p, 2 * n * sizeof(double), hipMemcpyDeviceToHost, st_));
    CCGPU_HIPX(hipStreamSynchronize(st_));
    for (long q = 0; q < n; ++q) {
      s4 += et[2 * q];
      s5 += et[2 * q + 1];
    }
  }
  if (e4) *e4 = s4;
  if (e5) *e5 = s5;
}

}  // namespace ccgpu
