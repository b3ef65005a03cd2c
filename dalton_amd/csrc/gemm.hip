// Strided / batched / split-K GEMM on CDNA4 matrix cores (gfx950).
//
// FP64: v_mfma_f64_16x16x4f64.  Block tile 128x128, 64x64 (K step 16) or 32x32
// (K step 32), 256 threads as 2x2 waves.  Operands are staged global ->
// registers -> LDS (padded so a wave's 16x4 fragment reads hit all 64 banks
// once per half-wave); the next K step's global loads are issued before the
// MFMAs of the current one.  No load is bounds-checked but those of a last,
// partial K step.  Large products are bound by the matrix cores (68 TFLOP/s of
// the 77 they sustain alone; 8192^3 in order k-fast x row-fast), small ones by
// the latency of a K step, so tile and K chunks are planned per shape.  Sum
// of the 20 products of one vector function, before (one 128 tile, every load
// checked where K is not a multiple of 16, chunks of 1024 or more) and with
// this kernel: o=5 v=19 1124 -> 136 us, o=11 v=93 3357 -> 1521, o=13 v=117
// 5829 -> 3980, o=21 v=170 27900 -> 24440, o=32 v=256 72540 -> 69790.
//
// All operands are described by element strides, so the same kernel serves
// row-major, transposed, batched and two-level-K (k = ko*Kin + ki)
// contractions.  Which dimension the loader walks fastest (for coalescing)
// is a template parameter chosen from the strides on the host.
#include <algorithm>
#include <cmath>
#include <map>
#include <mutex>
#include <type_traits>

#include "common.h"
#include "dgemm_tile.h"

namespace ccgpu {

// Logical tile for a linear block id.  Workgroups are dispatched round-robin
// over the 8 XCDs (block b runs on XCD b % 8), each with its own L2: give each
// XCD a contiguous range of tiles, and walk that range in groups of 8 m-tiles
// so the workgroups resident on one XCD share A and B panels in its L2.
__device__ __forceinline__ void tile_of(long b, long tiles_m, long tiles_n, long& tm, long& tn) {
  const long nt = tiles_m * tiles_n;
  const long per = nt / 8, full = per * 8;
  const long lg = (b < full) ? (b % 8) * per + b / 8 : b;
  constexpr long GM = 8;
  const long grp = lg / (GM * tiles_n);
  const long fm = grp * GM;
  const long gsz = min(tiles_m - fm, GM);
  const long r = lg - grp * GM * tiles_n;
  tm = fm + r % gsz;
  tn = r / gsz;
}

// Block tile T x T (T = 128, 64 or 32), 2x2 waves of (T/2)x(T/2), each wave
// (T/32)x(T/32) MFMA 16x16 tiles.  The next step's global loads are in
// flight while the current step's MFMAs run; one LDS stage, two barriers a
// step: a second stage saves a barrier but costs the blocks that hide it
// (128 tile 61 against 68 TFLOP/s; 64 tile, two blocks a CU instead of four to six,
// 1150^3 to 3570^3 products 1.2-1.3x the time).
template <int AMODE, int BMODE, bool K2, int T>
__global__ __launch_bounds__(256, T == 128 ? 2 : (T == 64 ? 4 : 5)) void k_dgemm(GemmDesc d, long kchunk, int nz,
                                                                               unsigned magic, double* ws) {
  constexpr int TM = T, TN = T, TK = Step<T>::TK;
  constexpr int IW = T / 32;      // MFMA tiles per wave and dimension
  // both operands [row][k]: a lane takes two consecutive k of a group of
  // eight for two MFMAs in turn, in 16-byte reads
  constexpr bool PAIR = AMODE == KFAST && BMODE == KFAST;
  __shared__ Stage<AMODE, T> As;
  __shared__ Stage<BMODE, T> Bs;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const long tiles_m = (d.M + TM - 1) / TM, tiles_n = (d.N + TN - 1) / TN;
  long tm, tn;
  tile_of(blockIdx.x, tiles_m, tiles_n, tm, tn);
  const long m0 = tm * TM, n0 = tn * TN;
  const double* A = static_cast<const double*>(d.A) + m0 * d.a_m;
  const double* B = static_cast<const double*>(d.B) + n0 * d.b_n;
  long kbeg = 0, kend = d.K;
  long z = blockIdx.z;  // batch; with split K, batch x chunk
  if (kchunk > 0) {
    z = blockIdx.z / nz;
    kbeg = (blockIdx.z - z * nz) * kchunk;
    kend = min(d.K, kbeg + kchunk);
  }
  A += z * d.a_b;
  B += z * d.b_b;
  const KMap ka{d.a_k, d.a_ko, (unsigned)d.Kin, magic}, kb{d.b_k, d.b_ko, (unsigned)d.Kin, magic};
  const int ma = (int)min((long)TM - 1, d.M - 1 - m0), nb = (int)min((long)TN - 1, d.N - 1 - n0);
  const long nfull = (kend - kbeg) / TK;
  const int rem = (int)((kend - kbeg) - nfull * TK);

  const int lr = lane & 15, lk = lane >> 4;

  auto run = [&](auto edge) {
    constexpr bool E = decltype(edge)::value;
    d4 acc[IW][IW];
#pragma unroll
    for (int i = 0; i < IW; ++i)
#pragma unroll
      for (int j = 0; j < IW; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    double ra[Step<T>::EPT], rb[Step<T>::EPT];
    Cursor<AMODE, K2, T, E> ca(A, d.a_m, ka, ma, kbeg, tid);
    Cursor<BMODE, K2, T, E> cb(B, d.b_n, kb, nb, kbeg, tid);
    auto load = [&](long k0, auto tail) {
      constexpr bool TL = decltype(tail)::value;
      ca.template load<TL>(ra, k0, kend);
      cb.template load<TL>(rb, k0, kend);
    };
    auto mfma8 = [&](int k) {  // k .. k + 7 of the staged step
      d2 pa[IW], pb[IW];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        double a[IW], b[IW];
#pragma unroll
        for (int t = 0; t < IW; ++t) {
          const int ra0 = wm * (T / 2) + t * 16 + lr, rb0 = wn * (T / 2) + t * 16 + lr;
          if constexpr (PAIR) {
            if (h == 0) {
              pa[t] = *reinterpret_cast<const d2*>(&As.at(ra0, k + 2 * lk));
              pb[t] = *reinterpret_cast<const d2*>(&Bs.at(rb0, k + 2 * lk));
            }
            a[t] = pa[t][h];
            b[t] = pb[t][h];
          } else {
            a[t] = As.at(ra0, k + 4 * h + lk);
            b[t] = Bs.at(rb0, k + 4 * h + lk);
          }
        }
#pragma unroll
        for (int i = 0; i < IW; ++i)
#pragma unroll
          for (int j = 0; j < IW; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
      }
    };
    const long nstep = nfull + (rem ? 1 : 0);
    if (nfull > 0)
      load(kbeg, std::false_type{});
    else if (rem > 0)
      load(kbeg, std::true_type{});
    for (long s = 0; s < nstep; ++s) {
      __syncthreads();
      stage_step(As, ra, tid);
      stage_step(Bs, rb, tid);
      __syncthreads();
      if (s + 1 < nfull)
        load(kbeg + (s + 1) * TK, std::false_type{});
      else if (s + 1 < nstep)
        load(kbeg + (s + 1) * TK, std::true_type{});
#pragma unroll
      for (int k = 0; k < TK; k += 8) mfma8(k);
    }


    // D[i][j] of a 16x16 f64 MFMA tile: lane = j + 16*(i%4), element i/4.
    if (kchunk > 0) {
      // split-K partial: ws[batch][chunk][m][n] (dense M x N)
      double* W = ws + (long)blockIdx.z * d.M * d.N;
#pragma unroll
      for (int i = 0; i < IW; ++i)
#pragma unroll
        for (int j = 0; j < IW; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const long m = m0 + wm * (T / 2) + i * 16 + r * 4 + lk;
            const long n = n0 + wn * (T / 2) + j * 16 + lr;
            if (m < d.M && n < d.N) W[m * d.N + n] = acc[i][j][r];
          }
      return;
    }
    // per 16-row block: C read (beta != 0) before any of the block's stores,
    // so the loads overlap instead of each waiting behind a store
    double* C = static_cast<double*>(d.C) + z * d.c_b;
#pragma unroll
    for (int i = 0; i < IW; ++i) {
      double cv[IW][4] = {};
      if (d.beta != 0.0) {  // uniform; indices clamped into C: no per-element branch
#pragma unroll
        for (int j = 0; j < IW; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const long m = min(m0 + wm * (T / 2) + i * 16 + r * 4 + lk, d.M - 1);
            const long n = min(n0 + wn * (T / 2) + j * 16 + lr, d.N - 1);
            cv[j][r] = C[m * d.c_m + n * d.c_n];
          }
      }
#pragma unroll
      for (int j = 0; j < IW; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const long m = m0 + wm * (T / 2) + i * 16 + r * 4 + lk;
          const long n = n0 + wn * (T / 2) + j * 16 + lr;
          if (m < d.M && n < d.N) {
            double v = d.alpha * acc[i][j][r];
            if (d.beta != 0.0) v += d.beta * cv[j][r];
            C[m * d.c_m + n * d.c_n] = v;
          }
        }
    }
  };
  if (ma == TM - 1 && nb == TN - 1)
    run(std::false_type{});
  else
    run(std::true_type{});
}

// C = alpha * sum_z ws[z] + beta * C (fixed summation order: deterministic).
// G groups of 256 / G threads share the z of 256 / G elements: with many
// chunks of a small C one thread per element would walk them one load
// latency after another.
template <int G>
__global__ __launch_bounds__(256) void k_splitk_reduce_f64(GemmDesc d, int nz, const double* ws) {
  constexpr int E = 256 / G;
  __shared__ double part[G][E];
  const long mn = d.M * d.N;
  ws += (long)blockIdx.y * nz * mn;
  double* C = static_cast<double*>(d.C) + (long)blockIdx.y * d.c_b;
  const int x = threadIdx.x % E, g = threadIdx.x / E;
  for (long e0 = (long)blockIdx.x * E; e0 < mn; e0 += (long)gridDim.x * E) {
    const long e = e0 + x;
    double s = 0.0;
    if (e < mn) {
#pragma unroll 4
      for (int z = g; z < nz; z += G) s += ws[(long)z * mn + e];
    }
    if constexpr (G > 1) {
      __syncthreads();  // the previous element's sums are read
      part[g][x] = s;
      __syncthreads();
    }
    if (g == 0 && e < mn) {
      if constexpr (G > 1) {
        for (int q = 1; q < G; ++q) s += part[q][x];
      }
      const long m = e / d.N, n = e - m * d.N;
      double* p = C + m * d.c_m + n * d.c_n;
      double v = d.alpha * s;
      if (d.beta != 0.0) v += d.beta * *p;
      *p = v;
    }
  }
}

namespace {
const char* const kDgemmName[2][2][2][3] = {
    {{{"k_dgemm<0,0,false,128>", "k_dgemm<0,0,false,64>", "k_dgemm<0,0,false,32>"},
      {"k_dgemm<0,0,true,128>", "k_dgemm<0,0,true,64>", "k_dgemm<0,0,true,32>"}},
     {{"k_dgemm<0,1,false,128>", "k_dgemm<0,1,false,64>", "k_dgemm<0,1,false,32>"},
      {"k_dgemm<0,1,true,128>", "k_dgemm<0,1,true,64>", "k_dgemm<0,1,true,32>"}}},
    {{{"k_dgemm<1,0,false,128>", "k_dgemm<1,0,false,64>", "k_dgemm<1,0,false,32>"},
      {"k_dgemm<1,0,true,128>", "k_dgemm<1,0,true,64>", "k_dgemm<1,0,true,32>"}},
     {{"k_dgemm<1,1,false,128>", "k_dgemm<1,1,false,64>", "k_dgemm<1,1,false,32>"},
      {"k_dgemm<1,1,true,128>", "k_dgemm<1,1,true,64>", "k_dgemm<1,1,true,32>"}}}};

bool two_level(const GemmDesc& d) { return d.Kin > 0 && d.Kin < d.K; }

template <int AM, int BM, int T>
void launch_f64(const GemmDesc& d, dim3 grid, long kchunk, int nz, double* ws, hipStream_t s) {
  const bool k2 = two_level(d);
  const unsigned magic =
      k2 ? (unsigned)std::min<unsigned long long>(0xFFFFFFFFull, (1ull << 32) / (unsigned long long)d.Kin) : 0u;
  const int id = prof_begin(kDgemmName[AM][BM][k2 ? 1 : 0][T == 128 ? 0 : (T == 64 ? 1 : 2)],
                            2.0 * d.M * d.N * d.K * d.batch, s);
  if (k2)
    CCGPU_LAUNCH((k_dgemm<AM, BM, true, T>), grid, dim3(256), 0, s, d, kchunk, nz, magic, ws);
  else
    CCGPU_LAUNCH((k_dgemm<AM, BM, false, T>), grid, dim3(256), 0, s, d, kchunk, nz, magic, ws);
  prof_end(id, s);
}

// Launch configuration of one FP64 GEMM: block tile and K chunks (1: no split).
struct F64Cfg {
  int tile = 128;
  int nz = 1;
};

constexpr long kMaxTiles = 1L << 24;

int step_k(int T) { return T == 32 ? Step<32>::TK : Step<64>::TK; }

// Estimated time (microseconds) of block tile T with K in nz chunks.  kRes
// blocks of the tile count as resident per CU (256 CUs; by registers 2, 4 to 6
// and 5 to 8, as the operand orders go); with c of them a K step
// takes kBase + kPer c cycles, and the blocks beyond whole rounds of 256 kRes
// take a round of their own.  A two-level K costs kTwoK, a split adds a launch
// and the pass over the partials, and C bounds the time from below (the
// shorter of the two adds a little: first loads and last stores are not
// overlapped).  The constants are measured (1648 runs, the products of a
// vector function for o = 5..21, v = 19..170; the configuration of least
// estimate is on average within 1% of the fastest one measured): in full
// rounds the 128 tile runs at 64 TFLOP/s, the 64 tile at 59 and the 32 tile at
// 45, but 64 x 64 and 32 x 32 tiles fill the chip, or leave it sooner, where
// 128 x 128 ones are few or mostly padding.
double cost_f64(const GemmDesc& d, int T, long nz) {
  const int q = T == 128 ? 0 : (T == 64 ? 1 : 2);
  constexpr double kBase[3] = {2400.0, 1000.0, 700.0}, kPer[3] = {3100.0, 1050.0, 650.0}, kTwoK[3] = {1.05, 1.08, 1.25};
  constexpr double kMhz = 2300.0;
  constexpr long kRes[3] = {2, 5, 8};
  const long blocks = (long)cdiv(d.M, T) * cdiv(d.N, T) * d.batch * nz, steps = cdiv(cdiv(d.K, nz), step_k(T));
  const long round = 256 * kRes[q], full = blocks / round, left = cdiv(blocks - full * round, 256);
  const double cycles = full * (kBase[q] + kPer[q] * kRes[q]) + (left > 0 ? kBase[q] + kPer[q] * left : 0.0);
  const double us = 3.8 + steps * cycles / kMhz * (two_level(d) ? kTwoK[q] : 1.0);
  const double mn = (double)d.batch * d.M * d.N, cus = 8.0 * mn * (d.beta != 0.0 ? 2.0 : 1.0) / 4.5e6;
  return std::max(us, cus) + 0.15 * std::min(us, cus) + (nz > 1 ? 2.3 + 0.02 * nz + nz * mn * 16.0 / 3.5e6 : 0.0);
}

// The configuration of least estimated time, of one tile (only) or of all.
F64Cfg plan_f64(const GemmDesc& d, int only = 0) {
  F64Cfg best;
  double bt = 1e300;
  for (int T : {128, 64, 32}) {
    if (only && T != only) continue;
    // a grid holds 2^24 blocks of 256 threads: long thin products past that
    // with the small tiles (540e6 x 1, K = 17) keep the 128 one
    if (T != 128 && (long)cdiv(d.M, T) * cdiv(d.N, T) >= kMaxTiles) continue;
    // chunks of at least two K steps; partials of at most 4 GB
    const double room = 4.0e9 / (8.0 * d.batch * (double)d.M * d.N);
    const long kmax = std::max<long>(1, std::min<long>(d.K / (2 * (step_k(T))), (long)std::min(room, 1e6)));
    for (long nz = 1; nz <= std::min<long>({kmax, 256, 65535 / d.batch}); nz = nz < 4 ? nz + 1 : nz + nz / 3) {
      const double t = cost_f64(d, T, nz);
      if (t < bt) {
        bt = t;
        best = F64Cfg{T, (int)nz};
      }
    }
  }
  return best;
}

// ---- autotuner: per GEMM shape class, the fastest configuration measured
struct ShapeKey {
  long M, N, K, Kin;
  int batch, am, bm;
  bool operator<(const ShapeKey& o) const {
    if (M != o.M) return M < o.M;
    if (N != o.N) return N < o.N;
    if (K != o.K) return K < o.K;
    if (Kin != o.Kin) return Kin < o.Kin;
    if (batch != o.batch) return batch < o.batch;
    if (am != o.am) return am < o.am;
    return bm < o.bm;
  }
};
struct Tuner {
  bool on = false;
  std::map<ShapeKey, F64Cfg> best;
  std::mutex mu;
};
Tuner& tuner() {
  static auto* t = new Tuner;
  return *t;
}
}  // namespace

void autotune_enable(bool on) { tuner().on = on; }
long autotune_entries() {
  std::lock_guard<std::mutex> lk(tuner().mu);
  return (long)tuner().best.size();
}

namespace {
long kspan(const GemmDesc& d, long s_k, long s_ko) {
  if (d.K <= 0) return -1;
  if (d.Kin > 0 && d.Kin < d.K) return ((d.K - 1) / d.Kin) * s_ko + (d.Kin - 1) * s_k;
  return (d.K - 1) * s_k;
}
}  // namespace

// Host-side bounds check of every operand span of a GEMM descriptor.
void check_gemm(const GemmDesc& d, size_t esz) {
  CCGPU_REQUIRE(d.a_m >= 0 && d.a_k >= 0 && d.a_b >= 0 && d.a_ko >= 0 && d.b_k >= 0 && d.b_n >= 0 &&
                    d.b_b >= 0 && d.b_ko >= 0 && d.c_m >= 0 && d.c_n >= 0 && d.c_b >= 0,
                "gemm: negative stride");
  if (d.M <= 0 || d.N <= 0 || d.batch <= 0) return;
  const long ka = kspan(d, d.a_k, d.a_ko), kb = kspan(d, d.b_k, d.b_ko);
  if (ka >= 0) check_span(d.A, 0, (d.M - 1) * d.a_m + ka + (d.batch - 1) * d.a_b, esz, "gemm A");
  if (kb >= 0) check_span(d.B, 0, (d.N - 1) * d.b_n + kb + (d.batch - 1) * d.b_b, esz, "gemm B");
  check_span(d.C, 0, (d.M - 1) * d.c_m + (d.N - 1) * d.c_n + (d.batch - 1) * d.c_b, esz, "gemm C");
}

namespace {
void run_f64(const GemmDesc& d, const F64Cfg& cfg, int am, int bm, hipStream_t s) {
  const int T = cfg.tile;
  const long tiles = (long)cdiv(d.M, T) * cdiv(d.N, T);
  long kchunk = 0;
  int nz = 1;
  double* ws = nullptr;
  if (cfg.nz > 1) {
    const long tk = step_k(T);  // chunks are whole K steps
    const long chunk = cdiv(cdiv(d.K, cfg.nz), tk) * tk;
    nz = (int)cdiv(d.K, chunk);
    if (nz >= 2) {
      kchunk = chunk;
      ws = grow_scratch(scratch_for(s).splitk, static_cast<size_t>(nz) * d.batch * d.M * d.N, s);
    }
  }
  CCGPU_REQUIRE((long)nz * d.batch <= 65535, "gemm: too many batches");
  CCGPU_REQUIRE(tiles < kMaxTiles, "gemm: too many tiles");
  CCGPU_REQUIRE(!two_level(d) || d.K < (1L << 32), "gemm: two-level K too long");
  dim3 grid((unsigned)tiles, 1, (unsigned)(nz * d.batch));
#define CCGPU_F64_LAUNCH(TT)                                                   \
  if (am == KFAST && bm == KFAST) launch_f64<KFAST, KFAST, TT>(d, grid, kchunk, nz, ws, s); \
  else if (am == KFAST) launch_f64<KFAST, RFAST, TT>(d, grid, kchunk, nz, ws, s);          \
  else if (bm == KFAST) launch_f64<RFAST, KFAST, TT>(d, grid, kchunk, nz, ws, s);          \
  else launch_f64<RFAST, RFAST, TT>(d, grid, kchunk, nz, ws, s);
  if (T == 32) {
    CCGPU_F64_LAUNCH(32)
  } else if (T == 64) {
    CCGPU_F64_LAUNCH(64)
  } else {
    CCGPU_F64_LAUNCH(128)
  }
#undef CCGPU_F64_LAUNCH
  CCGPU_HIPX(hipGetLastError());
  if (kchunk > 0) {
    const long mn = d.M * d.N;
    unsigned nb = static_cast<unsigned>(std::min<long>((mn + 255) / 256, 4096));
    if (nz > 4)
      CCGPU_LAUNCH(k_splitk_reduce_f64<8>, dim3((unsigned)std::min<long>((mn + 31) / 32, 8192), d.batch), dim3(256), 0, s, d, nz,
                   ws);
    else
      CCGPU_LAUNCH(k_splitk_reduce_f64<1>, dim3(nb, d.batch), dim3(256), 0, s, d, nz, ws);
    CCGPU_HIPX(hipGetLastError());
  }
}

// Times every candidate configuration of this shape (the GEMM runs for real,
// so tuning passes produce throwaway results) and returns the fastest.
F64Cfg tune_f64(const GemmDesc& d, int am, int bm, hipStream_t s) {
  // each tile with its planned chunks (an unsplit K of a million, one block
  // walking it, would take a third of a second a run)
  const F64Cfg cands[3] = {plan_f64(d, 128), plan_f64(d, 64), plan_f64(d, 32)};
  hipEvent_t e0, e1;
  CCGPU_HIP(hipEventCreate(&e0));
  CCGPU_HIP(hipEventCreate(&e1));
  F64Cfg best;
  float best_ms = 1e30f;
  for (const F64Cfg& c : cands) {
    run_f64(d, c, am, bm, s);                // warm-up (also sizes scratch)
    CCGPU_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < 2; ++r) run_f64(d, c, am, bm, s);
    CCGPU_HIP(hipEventRecord(e1, s));
    CCGPU_HIP(hipEventSynchronize(e1));
    float ms = 0.f;
    CCGPU_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (ms < best_ms) {
      best_ms = ms;
      best = c;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return best;
}
}  // namespace

namespace {
// plan_f64 through a small direct-mapped table per thread (the plan depends
// on the sizes and beta alone, and takes about as long as a launch).
F64Cfg planned(const GemmDesc& d) {
  struct Entry {
    ShapeKey key{};
    bool acc = false, set = false;
    F64Cfg cfg;
  };
  static thread_local Entry table[256];
  const bool acc = d.beta != 0.0;
  const ShapeKey key{d.M, d.N, d.K, two_level(d) ? d.Kin : 0, d.batch, 0, 0};
  unsigned long h = 1469598103934665603ul;
  for (long x : {key.M, key.N, key.K, key.Kin, (long)key.batch, acc ? 1L : 0L}) h = (h ^ (unsigned long)x) * 1099511628211ul;
  Entry& e = table[(h ^ (h >> 32)) & 255];
  if (!e.set || e.acc != acc || e.key < key || key < e.key) {
    e.key = key;
    e.acc = acc;
    e.cfg = plan_f64(d);
    e.set = true;
  }
  return e.cfg;
}
}  // namespace

void gemm_f64(const GemmDesc& d, hipStream_t s) {
  if (d.M <= 0 || d.N <= 0 || d.batch <= 0) return;
  check_gemm(d, sizeof(double));
  const int am = (d.a_m == 1 && d.a_k != 1) ? RFAST : KFAST;
  const int bm = (d.b_n == 1 && d.b_k != 1) ? RFAST : KFAST;
  F64Cfg cfg;
  Tuner& tu = tuner();
  const ShapeKey key{d.M, d.N, d.K, (d.Kin > 0 && d.Kin < d.K) ? d.Kin : 0, d.batch, am, bm};
  bool found = false;
  {
    std::lock_guard<std::mutex> lk(tu.mu);
    auto it = tu.best.find(key);
    if (it != tu.best.end()) {
      cfg = it->second;
      found = true;
    }
  }
  // Launches of 1024 or more 128 x 128 tiles fill the chip several times
  // over with the default configuration: only smaller ones are tuned.
  const long tiles128 = (long)cdiv(d.M, 128) * cdiv(d.N, 128) * d.batch;
  if (!found && tu.on && tiles128 < 1024 && !dryrun() && !capturing(s)) {
    cfg = tune_f64(d, am, bm, s);
    found = true;
    std::lock_guard<std::mutex> lk(tu.mu);
    tu.best[key] = cfg;
  }
  if (!found) cfg = planned(d);
  run_f64(d, cfg, am, bm, s);
}

void gemm_bf16x3(const GemmDesc& d, hipStream_t s);
void gemm_f32(const GemmDesc& d, hipStream_t s);
void bf16x3_scratch(ScratchNeed& n, long M, long N, long K, int batch);
void f32_scratch(ScratchNeed& n, long M, long N, long K, int batch);

void gemm_scratch(ScratchNeed& n, long M, long N, long K, int batch, double beta, GemmPrec prec) {
  if (M <= 0 || N <= 0 || batch <= 0) return;
  if (prec == GemmPrec::BF16X3) return bf16x3_scratch(n, M, N, K, batch);
  if (prec == GemmPrec::F32) return f32_scratch(n, M, N, K, batch);
  GemmDesc d;
  d.M = M;
  d.N = N;
  d.K = K;
  d.batch = std::min(batch, 65535);
  d.beta = beta;
  const int nz = planned(d).nz;  // (asked for again by the product itself)
  if (nz > 1) n.splitk = std::max(n.splitk, (size_t)nz * d.batch * M * N);
}

void gemm(const GemmDesc& d, GemmPrec prec, hipStream_t s) {
  if (prec == GemmPrec::BF16X3) {
    CCGPU_REQUIRE(d.batch <= 65535, "gemm: batch too large for the mixed-precision kernel");
    gemm_bf16x3(d, s);
    return;
  }
  if (prec == GemmPrec::F32) {
    gemm_f32(d, s);
    return;
  }
  CCGPU_REQUIRE(prec == GemmPrec::F64, "gemm: precision not available");
  if (d.batch <= 65535) {
    gemm_f64(d, s);
    return;
  }
  // grid.z is limited: issue the batch in chunks
  const size_t esz = sizeof(double);
  for (long b0 = 0; b0 < d.batch; b0 += 65535) {
    GemmDesc c = d;
    c.batch = static_cast<int>(std::min<long>(65535, d.batch - b0));
    c.A = static_cast<const char*>(d.A) + b0 * d.a_b * esz;
    c.B = static_cast<const char*>(d.B) + b0 * d.b_b * esz;
    c.C = static_cast<char*>(d.C) + b0 * d.c_b * esz;
    gemm_f64(c, s);
  }
}

void gemm_rm(bool ta, bool tb, long M, long N, long K, double alpha, const void* A, long lda,
             const void* B, long ldb, double beta, void* C, long ldc, GemmPrec prec, hipStream_t s) {
  GemmDesc d;
  d.M = M; d.N = N; d.K = K; d.alpha = alpha; d.beta = beta;
  d.A = A; d.B = B; d.C = C;
  if (!ta) { d.a_m = lda; d.a_k = 1; } else { d.a_m = 1; d.a_k = lda; }
  if (!tb) { d.b_k = ldb; d.b_n = 1; } else { d.b_k = 1; d.b_n = ldb; }
  d.c_m = ldc; d.c_n = 1;
  gemm(d, prec, s);
}

}  // namespace ccgpu
