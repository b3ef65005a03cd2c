// Mixed-precision GEMM: BF16x3 split products on gfx950 matrix cores with
// FP32 accumulation (v_mfma_f32_16x16x32_bf16).
//
// Every operand element x (stored FP64) is rounded to FP32 and split as
// x ~ hi + lo with hi = bf16(x), lo = bf16(x - hi) (round to nearest even);
// a product is formed as hi*hi + hi*lo + lo*hi, so each term carries ~16
// significant bits and the sum is accumulated in FP32.  A prologue packs
// each operand (any strides, batching, two-level K) into K-contiguous
// [batch][row][k] hi and lo arrays padded to the tile sizes; the GEMM kernel
// then streams 16-byte chunks straight into LDS.  The epilogue applies
// alpha/beta in FP64 to the FP64 output with arbitrary strides.
#include <cmath>
#include <cstdlib>
#include <map>
#include <mutex>
#include <type_traits>

#include "bf16x3_tile.h"
#include "common.h"
#include "kernels.h"

namespace ccgpu {

namespace {

// Two elements split together: packed hi and lo pairs (the conversion
// instruction rounds to nearest even).
__device__ __forceinline__ unsigned pk_bf16(float a, float b) {
  typedef float f2v __attribute__((ext_vector_type(2)));
  typedef __bf16 bf2v __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(unsigned, __builtin_convertvector(f2v{a, b}, bf2v));
}
__device__ __forceinline__ void split2(float a, float b, unsigned& hi, unsigned& lo) {
  hi = pk_bf16(a, b);
  lo = pk_bf16(a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u));
}

struct PackDesc {
  const double* src;
  long rows, K;              // logical operand: rows x K
  long s_r, s_k, s_ko, Kin;  // element (r,k) at src + r*s_r + koff(k) + b*s_b
  long s_b;
  long Rp, Kp;  // padded sizes of the packed arrays
  float scale;  // multiplies every element
};

template <bool K2>
__device__ __forceinline__ long pk_koff(const PackDesc& p, long k) {
  if (K2) {
    const long ko = k / p.Kin;
    return ko * p.s_ko + (k - ko * p.Kin) * p.s_k;
  }
  return k * p.s_k;
}

// Operand order of the source: along rows, along k with unit stride, any.
enum { PK_R = 0, PK_K1 = 1, PK_ANY = 2 };

// Tile of TR (64 or 32) rows x 64 k per block, every load before the first
// use (elements past the operand re-read one inside it and become zeros).  A
// row of the tile is one whole 128-byte line of hi and of lo, written four
// bytes a lane: with 32 x 32 tiles two blocks, on two XCDs, shared every line.
// PK_R transposes through LDS.  Bound by HBM: o=32 v=256, 22 operands of a
// vector function, 3.1 ms before, 2.7 now (12 bytes an element, 3.7 TB/s).
template <int MODE, bool K2, int TR>
__global__ __launch_bounds__(256) void k_pack_bf16x2(PackDesc p, unsigned short* __restrict__ hi,
                                                     unsigned short* __restrict__ lo) {
  constexpr int NE = TR / 8;  // pairs per thread
  __shared__ float tile[MODE == PK_R ? 64 : 1][TR + 1];
  const long r0 = (long)blockIdx.x * TR, k0 = (long)blockIdx.y * 64, b = blockIdx.z;
  const double* src = p.src + b * p.s_b;
  const int t = threadIdx.x, kp = 2 * (t % 32);
  const bool whole = r0 + TR <= p.rows && k0 + 64 <= p.K;
  float v[NE][2];
  if (p.rows <= 0 || p.K <= 0) {
#pragma unroll
    for (int i = 0; i < NE; ++i) v[i][0] = v[i][1] = 0.0f;
  } else if (MODE == PK_R) {
    float u[2 * NE];
    const long r = r0 + t % TR, k = k0 + t / TR;
    const double* s = src + min(r, p.rows - 1) * p.s_r;
    if (whole && !K2) {
      const double* q = s + k * p.s_k;
      const long st = (256 / TR) * p.s_k;
#pragma unroll
      for (int i = 0; i < 2 * NE; ++i) {
        u[i] = (float)*q;
        q += st;
      }
    } else {
#pragma unroll
      for (int i = 0; i < 2 * NE; ++i) u[i] = (float)s[pk_koff<K2>(p, min(k + (256 / TR) * i, p.K - 1))];
#pragma unroll
      for (int i = 0; i < 2 * NE; ++i)
        if (r >= p.rows || k + (256 / TR) * i >= p.K) u[i] = 0.0f;
    }
#pragma unroll
    for (int i = 0; i < 2 * NE; ++i) tile[t / TR + (256 / TR) * i][t % TR] = p.scale * u[i];  // [k][r]
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      v[i][0] = tile[kp][t / 32 + 8 * i];
      v[i][1] = tile[kp + 1][t / 32 + 8 * i];
    }
  } else {
    const long k = k0 + kp;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      const double* s = src + min(r0 + t / 32 + 8 * i, p.rows - 1) * p.s_r;
      if (MODE == PK_K1 && whole) {
        typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));
        const d2u x = *reinterpret_cast<const d2u*>(s + k);
        v[i][0] = p.scale * (float)x[0];
        v[i][1] = p.scale * (float)x[1];
      } else {
        v[i][0] = p.scale * (float)s[pk_koff<K2>(p, min(k, p.K - 1))];
        v[i][1] = p.scale * (float)s[pk_koff<K2>(p, min(k + 1, p.K - 1))];
      }
    }
    if (!whole) {
#pragma unroll
      for (int i = 0; i < NE; ++i) {
        const bool in = r0 + t / 32 + 8 * i < p.rows;
        if (!in || k >= p.K) v[i][0] = 0.0f;
        if (!in || k + 1 >= p.K) v[i][1] = 0.0f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < NE; ++i) {
    const long r = r0 + t / 32 + 8 * i;
    if (r >= p.Rp) continue;
    const long o = (b * p.Rp + r) * p.Kp + k0 + kp;
    unsigned h, l;
    split2(v[i][0], v[i][1], h, l);
    *reinterpret_cast<unsigned*>(hi + o) = h;
    *reinterpret_cast<unsigned*>(lo + o) = l;
  }
}

__device__ __forceinline__ void tile_of3(long b, long tiles_m, long tiles_n, long& tm, long& tn, long GM = 8) {
  const long nt = tiles_m * tiles_n;
  const long per = nt / 8, full = per * 8;
  const long lg = (b < full) ? (b % 8) * per + b / 8 : b;
  const long grp = lg / (GM * tiles_n);
  const long fm = grp * GM;
  const long gsz = min(tiles_m - fm, GM);
  const long r = lg - grp * GM * tiles_n;
  tm = fm + r % gsz;
  tn = r / gsz;
}

constexpr int TM = 128, TN = bf3::TN, TK = bf3::TK;

// One block per output tile over ceil(M/TMr) x ceil(N/TN) tiles (rows of a
// tile past M or N are the packed padding: read, never stored), rasterised
// by tile_of3.
template <typename OutT, int RW>
__global__ __launch_bounds__(128 * RW, 4 / RW) void k_gemm_bf16x3(BMulti p) {
  __shared__ bf3::Smem<RW> S;
  constexpr int TMr = 64 * RW;
  long tm, tn;
  tile_of3(blockIdx.x, (p.M + TMr - 1) / TMr, (p.N + TN - 1) / TN, tm, tn, p.gm);
  bf3::tile<OutT, RW>(p, tm * TMr, tn * TN, blockIdx.z, S);
}


// Large-tile kernel (the default; CCGPU_BF16X3_VARIANT=0 selects the
// 128x128 kernel above): one 256x256 tile of bf3w8::tile per block of eight
// waves, one block per CU, rasterised by tile_of3.
constexpr int DT = bf3w8::DT;

template <typename OutT>
__global__ __launch_bounds__(512, 1) void k_gemm_bf16x3_w8(BMulti p) {
  __shared__ bf3w8::Smem S;
  long tm, tn;
  tile_of3(blockIdx.x, p.Mp / DT, p.Np / DT, tm, tn, p.gm);
  bf3w8::tile<OutT>(p, tm * DT, tn * DT, blockIdx.z, S);
}

// Small-tile kernel: 64x64 tiles of bf3s::tile.
template <typename OutT>
__global__ __launch_bounds__(256, 3) void k_gemm_bf16x3_s(BMulti p) {
  __shared__ bf3s::Smem S;
  long tm, tn;
  tile_of3(blockIdx.x, (p.M + bf3s::DT - 1) / bf3s::DT, (p.N + bf3s::DT - 1) / bf3s::DT, tm, tn, p.gm);
  bf3s::tile<OutT>(p, tm * bf3s::DT, tn * bf3s::DT, blockIdx.z, S);
}

// Block-tile kernel: 1 (default) the eight-wave 256x256 direct-to-LDS
// kernel, 0 the four-wave 128x128 one (CCGPU_BF16X3_VARIANT=0).  At o=64
// v=512 the 256x256 kernel runs the mixed CCSD iteration in 2.05 s against
// 2.30 s (361 against 307 TFLOP/s per launch), bit for bit the same.
int variant() {
  static const int v = [] {
    const char* e = std::getenv("CCGPU_BF16X3_VARIANT");
    return (e && *e) ? std::atoi(e) : 1;
  }();
  return v;
}

int group_m() {
  static const int g = [] {
    const char* e = std::getenv("CCGPU_BF16X3_GM");
    const int x = e ? std::atoi(e) : 8;
    return x > 0 ? x : 8;
  }();
  return g;
}

// Block-tile kernels of a product: the four-wave 128x128 tile (two blocks
// per CU), the eight-wave 256x256 one (one block per CU; operands padded to
// 256 rows, which bf16x3_rpad gives) or the four-wave 64x64 one (three blocks
// per CU).  All accumulate every output element in the same order, so the
// choice never changes a result bit.
enum BKern { kT128 = 0, kT256 = 1, kT64 = 2 };

template <typename OutT>
void launch_kernel(int kern, const BMulti& p, int batch, hipStream_t s) {
  if (kern == kT256) {
    const long ntiles = (p.Mp / DT) * (p.Np / DT);
    CCGPU_REQUIRE(ntiles < (1L << 23), "bf16x3 gemm: grid too large");
    CCGPU_LAUNCH(k_gemm_bf16x3_w8<OutT>, dim3((unsigned)ntiles, 1, (unsigned)batch), dim3(512), 0, s, p);
  } else if (kern == kT64) {
    const long ntiles = (long)cdiv(p.M, bf3s::DT) * cdiv(p.N, bf3s::DT);
    CCGPU_REQUIRE(ntiles < (1L << 23), "bf16x3 gemm: grid too large");
    CCGPU_LAUNCH(k_gemm_bf16x3_s<OutT>, dim3((unsigned)ntiles, 1, (unsigned)batch), dim3(256), 0, s, p);
  } else {
    const long ntiles = (long)cdiv(p.M, TM) * cdiv(p.N, TN);
    CCGPU_REQUIRE(ntiles < (1L << 23), "bf16x3 gemm: grid too large");
    CCGPU_LAUNCH((k_gemm_bf16x3<OutT, 2>), dim3((unsigned)ntiles, 1, (unsigned)batch), dim3(256), 0, s, p);
  }
  CCGPU_HIPX(hipGetLastError());
}

// ---- autotuner: per product shape class, the faster block tile measured
struct BKey {
  long M, N, Mp, Np, K[4];
  int nterm, batch, flt;
  bool operator<(const BKey& o) const {
    if (M != o.M) return M < o.M;
    if (N != o.N) return N < o.N;
    if (Mp != o.Mp) return Mp < o.Mp;
    if (Np != o.Np) return Np < o.Np;
    for (int t = 0; t < 4; ++t)
      if (K[t] != o.K[t]) return K[t] < o.K[t];
    if (nterm != o.nterm) return nterm < o.nterm;
    if (batch != o.batch) return batch < o.batch;
    return flt < o.flt;
  }
};
struct BTuner {
  std::mutex mu;
  std::map<BKey, int> best;
  long timed = 0;
};
BTuner& btuner() {
  static auto* t = new BTuner;  // never destroyed (used until process exit)
  return *t;
}

// CCGPU_BF16X3_TUNE=0 disables the timing runs (the cost model decides);
// so does a NoTune scope on the calling thread (callers that must not create
// events or run extra launches).
thread_local int t_no_tune = 0;
bool tune_on() {
  static const bool on = [] {
    const char* e = std::getenv("CCGPU_BF16X3_TUNE");
    return !(e && *e && std::atoi(e) == 0);
  }();
  return on && t_no_tune == 0;
}
struct NoTune {
  NoTune() { ++t_no_tune; }
  ~NoTune() { --t_no_tune; }
};

// Products of fewer 128x128 tiles than this (four per CU, two rounds of blocks)
// may take the 64x64 one.
constexpr long kSmallTiles = 1024;
long tiles128(const BMulti& p, int batch) { return (long)cdiv(p.M, TM) * cdiv(p.N, TN) * batch; }

// Times the tiles on the product itself: an overwriting product (beta = 0)
// runs as given, since the real launch that follows rewrites the same
// values; an accumulating one runs with alpha = 0 and beta = 1, which leaves
// C as it was (up to the sign of exact zeros).
template <typename OutT>
int tune(const BMulti& p, int batch, hipStream_t s) {
  BMulti q = p;
  if (p.beta != 0.0) {
    q.alpha = 0.0;
    q.beta = 1.0;
  }
  hipEvent_t e0, e1;
  CCGPU_HIP(hipEventCreate(&e0));
  CCGPU_HIP(hipEventCreate(&e1));
  float best = 0.f;
  int kern = -1;
  for (int k : {kT128, kT256, kT64}) {
    if (k == kT256 && (p.Mp % DT != 0 || p.Np % DT != 0)) continue;
    if (k == kT64 && tiles128(p, batch) >= kSmallTiles) continue;
    float ms = 0.f;
    launch_kernel<OutT>(k, q, batch, s);  // warm-up
    CCGPU_HIP(hipEventRecord(e0, s));
    launch_kernel<OutT>(k, q, batch, s);
    CCGPU_HIP(hipEventRecord(e1, s));
    CCGPU_HIP(hipEventSynchronize(e1));
    CCGPU_HIP(hipEventElapsedTime(&ms, e0, e1));
    if (kern < 0 || ms < best) {
      best = ms;
      kern = k;
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  return kern;
}

// Without a measurement: the 256x256 tile computes M x N padded to 256,
// the 128x128 one ceil(M/128) x ceil(N/128) tiles, at 361 against 307
// TFLOP/s measured on square products; the 256 tile also needs a wave of
// tiles over the CUs to be worth its larger grain.
bool large_tile(long M, long N, long batch) {
  const double a256 = (double)bf16x3_rpad(M) * (double)bf16x3_rpad(N);
  const double a128 = (double)cdiv(M, TM) * TM * (double)cdiv(N, TN) * TN;
  const long t256 = (bf16x3_rpad(M) / DT) * (bf16x3_rpad(N) / DT) * batch;
  return a256 * 307.0 <= a128 * 361.0 && t256 >= 256;
}

template <typename OutT>
void launch_multi(BMulti p, int batch, hipStream_t s) {
  p.gm = group_m();
  CCGPU_REQUIRE(batch < 65536, "bf16x3 gemm: grid too large");
  int kern = kT128;
  if (variant() == 1 && p.Mp % DT == 0 && p.Np % DT == 0) {
    BKey key{p.M, p.N, p.Mp, p.Np, {0, 0, 0, 0}, p.nterm, batch, std::is_same<OutT, float>::value ? 1 : 0};
    for (int t = 0; t < p.nterm; ++t) key.K[t] = p.t[t].Kp;
    BTuner& tu = btuner();
    bool found = false;
    {
      std::lock_guard<std::mutex> lk(tu.mu);
      auto it = tu.best.find(key);
      if (it != tu.best.end()) {
        kern = it->second;
        found = true;
      }
    }
    if (!found) {
      if (tune_on() && !dryrun() && !capturing(s)) {
        kern = tune<OutT>(p, batch, s);
        std::lock_guard<std::mutex> lk(tu.mu);
        tu.best[key] = kern;
        ++tu.timed;
      } else {
        // without a measurement: 64x64 tiles below one 128x128 tile per CU
        kern = large_tile(p.M, p.N, batch) ? kT256 : (tiles128(p, batch) < 256 ? kT64 : kT128);
      }
    }
  }
  launch_kernel<OutT>(kern, p, batch, s);
}

}  // namespace

long bf16x3_kpad(long K) { return std::max<long>(TK, (K + TK - 1) / TK * TK); }
// Packed rows are padded to 64 columns, the 64 and 256 tiles multiply whole
// steps of 32: a term of o = 32 in the (T) passes costs one step, not two
// (64 triples at v = 256: 17.2 -> 16.6 ms).
long bf16x3_kcols(long K) { return std::max<long>(32, (K + 31) / 32 * 32); }
long bf16x3_rpad(long R) {
  const long t = variant() != 0 ? DT : TM;  // rows padded to the block tile in use
  return (R + t - 1) / t * t;
}

void bf16x3_pack(const double* src, long rows, long K, long s_r, long s_k, long s_b, int batch, long Rp, long Kp,
                 float scale, unsigned short* hi, unsigned short* lo, hipStream_t s, long s_ko, long Kin) {
  PackDesc p{src, rows, K, s_r, s_k, s_ko, Kin, s_b, Rp, Kp, scale};
  if (rows > 0 && K > 0) {
    long hiofs = (rows - 1) * s_r + (batch - 1) * s_b;
    hiofs += (Kin > 0 && Kin < K) ? ((K - 1) / Kin) * s_ko + (Kin - 1) * s_k : (K - 1) * s_k;
    check_span(src, 0, hiofs, sizeof(double), "bf16x3 pack source");
  }
  check_span(hi, 0, (long)batch * Rp * Kp - 1, 2, "bf16x3 pack hi");
  check_span(lo, 0, (long)batch * Rp * Kp - 1, 2, "bf16x3 pack lo");
  const long kt = Kp / 64;
  // 64-row tiles once they give eight blocks per CU
  const int tr = cdiv(Rp, 64) * kt * batch >= 2048 ? 64 : 32;
  CCGPU_REQUIRE(Kp % 64 == 0 && kt < 65536 && batch < 65536 && Rp < (1L << 29), "bf16x3 pack: grid too large");
  const dim3 grid(cdiv(Rp, tr), (unsigned)kt, (unsigned)batch);
  const bool k2 = Kin > 0 && Kin < K;
  const int mode = (s_r == 1 && s_k != 1) ? PK_R : (s_k == 1 && !k2 ? PK_K1 : PK_ANY);
#define CCGPU_PACK(M, Q)                                                                 \
  if (mode == M && k2 == Q) {                                                            \
    if (tr == 64)                                                                        \
      CCGPU_LAUNCH((k_pack_bf16x2<M, Q, 64>), grid, dim3(256), 0, s, p, hi, lo);          \
    else                                                                                 \
      CCGPU_LAUNCH((k_pack_bf16x2<M, Q, 32>), grid, dim3(256), 0, s, p, hi, lo);          \
  }
  CCGPU_PACK(PK_R, false)
  CCGPU_PACK(PK_R, true)
  CCGPU_PACK(PK_K1, false)
  CCGPU_PACK(PK_ANY, false)
  CCGPU_PACK(PK_ANY, true)
#undef CCGPU_PACK
  CCGPU_HIPX(hipGetLastError());
}

// Multi-term product into a float or double output (see k_gemm_bf16x3).
// Every term's packed A must cover Mp rows (per batch, at stride a_bs) and
// B Np rows, both with row length Kp; rows past M/N are read, never used.
BMulti bf16x3_desc(const BTerm* terms, int nterm, long M, long N, int batch, void* C, bool c_float, long c_m,
                   long c_n, long c_b, double alpha, double beta) {
  CCGPU_REQUIRE(nterm >= 1 && nterm <= 4, "bf16x3_multi: 1..4 terms");
  BMulti p{};
  p.nterm = nterm;
  for (int t = 0; t < nterm; ++t) {
    p.t[t] = terms[t];
    if (p.t[t].Kc == 0) p.t[t].Kc = p.t[t].Kp;
    CCGPU_REQUIRE(terms[t].Kp % TK == 0, "bf16x3_multi: Kp must be a multiple of 64");
    CCGPU_REQUIRE(p.t[t].Kc % 32 == 0 && p.t[t].Kc <= p.t[t].Kp, "bf16x3_multi: Kc must be a multiple of 32");
  }
  p.M = M; p.N = N; p.Mp = bf16x3_rpad(M); p.Np = bf16x3_rpad(N);
  p.alpha = alpha; p.beta = beta; p.C = C; p.c_m = c_m; p.c_n = c_n; p.c_b = c_b;
  const size_t esz = c_float ? sizeof(float) : sizeof(double);
  for (int t = 0; t < nterm; ++t) {
    const BTerm& T = terms[t];
    check_span(T.Ah, 0, (batch - 1) * T.a_bs + p.Mp * T.Kp - 1, 2, "bf16x3 A");
    check_span(T.Al, 0, (batch - 1) * T.a_bs + p.Mp * T.Kp - 1, 2, "bf16x3 A lo");
    check_span(T.Bh, 0, (batch - 1) * T.b_bs + p.Np * T.Kp - 1, 2, "bf16x3 B");
    check_span(T.Bl, 0, (batch - 1) * T.b_bs + p.Np * T.Kp - 1, 2, "bf16x3 B lo");
  }
  check_span(C, 0, (M - 1) * c_m + (N - 1) * c_n + (batch - 1) * c_b, esz, "bf16x3 C");
  return p;
}

void bf16x3_multi(const BTerm* terms, int nterm, long M, long N, int batch, void* C, bool c_float, long c_m,
                  long c_n, long c_b, double alpha, double beta, double flops, hipStream_t s) {
  const BMulti p = bf16x3_desc(terms, nterm, M, N, batch, C, c_float, c_m, c_n, c_b, alpha, beta);
  bf16x3_run(p, batch, c_float, flops, s);
}

void bf16x3_run(const BMulti& p, int batch, bool c_float, double flops, hipStream_t s) {
  const int id = prof_begin("k_gemm_bf16x3", flops, s);
  if (c_float)
    launch_multi<float>(p, batch, s);
  else
    launch_multi<double>(p, batch, s);
  prof_end(id, s);
}

void check_gemm(const GemmDesc& d, size_t esz);

// The packed operands of gemm_bf16x3, hi and lo of A and of B.
void bf16x3_scratch(ScratchNeed& n, long M, long N, long K, int batch) {
  const long Kp = bf16x3_kpad(K);
  const size_t na = (size_t)batch * bf16x3_rpad(M) * Kp, nb = (size_t)batch * bf16x3_rpad(N) * Kp;
  for (int q = 0; q < 4; ++q) n.pack[q] = std::max(n.pack[q], q < 2 ? na : nb);
}

void gemm_bf16x3(const GemmDesc& d, hipStream_t s) {
  if (d.M <= 0 || d.N <= 0 || d.batch <= 0) return;
  check_gemm(d, sizeof(double));
  const long Mp = bf16x3_rpad(d.M), Np = bf16x3_rpad(d.N), Kp = bf16x3_kpad(d.K);
  const long na = (long)d.batch * Mp * Kp, nb = (long)d.batch * Np * Kp;
  StreamScratch& sc = scratch_for(s);
  unsigned short* pk[4];
  for (int i = 0; i < 4; ++i) pk[i] = grow_scratch(sc.pack[i], i < 2 ? na : nb, s);
  bf16x3_pack(static_cast<const double*>(d.A), d.M, d.K, d.a_m, d.a_k, d.a_b, d.batch, Mp, Kp, 1.0f,
              pk[0], pk[1], s, d.a_ko, d.Kin);
  bf16x3_pack(static_cast<const double*>(d.B), d.N, d.K, d.b_n, d.b_k, d.b_b, d.batch, Np, Kp, 1.0f,
              pk[2], pk[3], s, d.b_ko, d.Kin);
  BTerm t{pk[0], pk[1], pk[2], pk[3], Kp, Mp * Kp, Np * Kp, bf16x3_kcols(d.K)};
  bf16x3_multi(&t, 1, d.M, d.N, d.batch, d.C, false, d.c_m, d.c_n, d.c_b, d.alpha, d.beta,
               2.0 * d.M * d.N * d.K * d.batch, s);
}

// ------------------------------------------------------ no-allocation variant
// The packed hi/lo operands of one product live in this array: one copy per
// GPU, held until the process ends, shared by every call on that GPU (the
// last call's contents stay; every element a product reads is rewritten by
// its pack kernels first).
static __device__ __attribute__((aligned(256))) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on the current device, looked up once per
// device (with that device current) and registered for the span checks.
unsigned short* noalloc_scratch() {
  int dev = 0;
  if (!dryrun()) CCGPU_HIP(hipGetDevice(&dev));
  CCGPU_REQUIRE(dev >= 0 && dev < kMaxDevices, "no-allocation scratch: device index out of range");
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    if (dryrun())
      ptr = dry_alloc(kNoAllocScratchBytes);
    else
      CCGPU_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    CCGPU_REQUIRE(ptr != nullptr, "no-allocation scratch: symbol address is null");
    register_alloc(ptr, kNoAllocScratchBytes);
    g_scratch_ptr[dev] = ptr;
  }
  return static_cast<unsigned short*>(g_scratch_ptr[dev]);
}
}  // namespace

void gemm_bf16x3_noalloc(const GemmDesc& d, hipStream_t s) {
  if (d.M <= 0 || d.N <= 0 || d.batch <= 0) return;
  check_gemm(d, sizeof(double));
  const long Mp = bf16x3_rpad(d.M), Np = bf16x3_rpad(d.N), Kp = bf16x3_kpad(d.K);
  const long na = (long)d.batch * Mp * Kp, nb = (long)d.batch * Np * Kp;
  const size_t need = 2 * sizeof(unsigned short) * (size_t)(na + nb);
  if (need > kNoAllocScratchBytes)
    throw Error(1, "no-allocation BF16x3 GEMM: the packed operands need " + std::to_string(need) +
                       " bytes, the scratch holds " + std::to_string(kNoAllocScratchBytes));
  NoTune no_tune;  // no timing runs: the block tile comes from the tuned cache or the cost model
  unsigned short* base = noalloc_scratch();
  // na and nb are multiples of 64 elements: every array starts 128-byte aligned
  unsigned short* pk[4] = {base, base + na, base + 2 * na, base + 2 * na + nb};
  bf16x3_pack(static_cast<const double*>(d.A), d.M, d.K, d.a_m, d.a_k, d.a_b, d.batch, Mp, Kp, 1.0f, pk[0], pk[1],
              s, d.a_ko, d.Kin);
  bf16x3_pack(static_cast<const double*>(d.B), d.N, d.K, d.b_n, d.b_k, d.b_b, d.batch, Np, Kp, 1.0f, pk[2], pk[3],
              s, d.b_ko, d.Kin);
  BTerm t{pk[0], pk[1], pk[2], pk[3], Kp, Mp * Kp, Np * Kp, bf16x3_kcols(d.K)};
  bf16x3_multi(&t, 1, d.M, d.N, d.batch, d.C, false, d.c_m, d.c_n, d.c_b, d.alpha, d.beta,
               2.0 * d.M * d.N * d.K * d.batch, s);
}

}  // namespace ccgpu

namespace ccgpu {
// V+/-_{ab,cd} = Y[(a,c),(b,d)] +/- Y[(a,d),(b,c)] of one ladder a-batch,
// from the FP32 Y block straight into the split-bf16 operand layout of the
// S GEMM: hi/lo[s][r][p] (s = 0: V+, 1: V-; p = d(d+1)/2 + c), row length
// Kp; the K padding p in [npv, Kp) is written as zeros by the first tile
// pair of each row.
//
// Block: row r = (a,b), 32 columns d and 128 c (c <= d), both orders of Y
// staged in LDS (16-byte loads where rows of Y are 16-byte aligned, V4); every
// d is one run of the packed row, written two bf16 (4 bytes) a lane, the odd
// elements at its ends alone.  Bound by HBM (16 bytes a pair): o=32 v=256
// 7.2 ms a vector function with 32 x 32 tiles, 2-byte stores and the tiles of a
// row spread over the XCDs, 4.7 now (3.7 TB/s).
template <bool V4>
__global__ __launch_bounds__(256) void k_ladder_vpm_pack(unsigned short* __restrict__ hi,
                                                         unsigned short* __restrict__ lo, const float* __restrict__ Y,
                                                         long ldY, int a0, int v, long rows, long Rp, long Kp) {
  constexpr int CT = 128;
  __shared__ float Mcd[CT][33], Mdc[32][CT + 1];
  // the tiles of a row run one after the other on one XCD (block b runs on XCD
  // b % 8), whose L2 joins their part lines of Y and of the packed row
  const int nct = (v + CT - 1) / CT, ntile = nct * ((v + 31) / 32), idx = blockIdx.x / 8, tile = idx % ntile;
  const int c0 = (tile % nct) * CT, d0 = (tile / nct) * 32;
  const long r = (long)(idx / ntile) * 8 + blockIdx.x % 8;
  if (r >= rows) return;
  const int t = threadIdx.x;
  unsigned short* const row[4] = {hi + r * Kp, lo + r * Kp, hi + (Rp + r) * Kp, lo + (Rp + r) * Kp};
  if (tile == 0) {  // K padding
    const long npv = (long)v * (v + 1) / 2;
    for (long p = npv + t; p < Kp; p += 256)
      for (int q = 0; q < 4; ++q) row[q][p] = 0;
  }
  if (c0 > d0 + 31) return;
  int a, b;
  batch_row_decode(r, a0, v, a, b);
  const float* Ya = Y + (long)(a - a0) * v * ldY + (long)(b - a0) * v;  // M[c][d] = Ya[c*ldY + d]
  // all loads before the LDS stores, rows and columns clamped into the block
  // (elements past the triangle or v are staged and not used)
  const int cm = min(v - 1, d0 + 31);
  if constexpr (V4) {
    f4 mcd[4], mdc[4];  // v is a multiple of four here: groups of four columns do not straddle it
    const int dc = min(d0 + 4 * (t % 8), v - 4), cc = min(c0 + 4 * (t % 32), cm & ~3);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      mcd[k] = *reinterpret_cast<const f4*>(Ya + (long)min(c0 + t / 8 + 32 * k, cm) * ldY + dc);
#pragma unroll
    for (int k = 0; k < 4; ++k)
      mdc[k] = *reinterpret_cast<const f4*>(Ya + (long)min(d0 + t / 32 + 8 * k, v - 1) * ldY + cc);
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int h = 0; h < 4; ++h) Mcd[t / 8 + 32 * k][4 * (t % 8) + h] = mcd[k][h];
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int h = 0; h < 4; ++h) Mdc[t / 32 + 8 * k][4 * (t % 32) + h] = mdc[k][h];
  } else {
    float mcd[16], mdc[16];
    const int dc = min(d0 + t % 32, v - 1), cc = min(c0 + t % CT, cm);
#pragma unroll
    for (int k = 0; k < 16; ++k) mcd[k] = Ya[(long)min(c0 + t / 32 + 8 * k, cm) * ldY + dc];
#pragma unroll
    for (int k = 0; k < 16; ++k) mdc[k] = Ya[(long)min(d0 + t / CT + 2 * k, v - 1) * ldY + cc];
#pragma unroll
    for (int k = 0; k < 16; ++k) Mcd[t / 32 + 8 * k][t % 32] = mcd[k];
#pragma unroll
    for (int k = 0; k < 16; ++k) Mdc[t / CT + 2 * k][t % CT] = mdc[k];
  }
  __syncthreads();
  const int lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
#pragma unroll 2
  for (int k = 0; k < 8; ++k) {
    const int dl = wave + 4 * k, d = d0 + dl;
    if (d >= v) break;
    const long p0 = (long)d * (d + 1) / 2 + c0;
    const int n = min(CT, d - c0 + 1);  // elements of this run: c0 .. c0 + n - 1
    const int sh = (int)(p0 & 1);
    for (int e = 2 * lane - sh; e < n; e += CT) {  // the aligned pair of elements e, e + 1
      const int e0 = max(e, 0), e1 = min(e + 1, CT - 1);
      const float x0 = Mcd[e0][dl], x1 = Mcd[e1][dl], y0 = Mdc[dl][e0], y1 = Mdc[dl][e1];
      unsigned w[4];
      split2(x0 + y0, x1 + y1, w[0], w[1]);
      split2(x0 - y0, x1 - y1, w[2], w[3]);
      if (e >= 0 && e + 1 < n) {
#pragma unroll
        for (int q = 0; q < 4; ++q) *reinterpret_cast<unsigned*>(row[q] + p0 + e) = w[q];
      } else if (e >= 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) row[q][p0 + e] = (unsigned short)w[q];
      } else if (n > 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) row[q][p0] = (unsigned short)(w[q] >> 16);
      }
    }
  }
}

__global__ void k_fill_u16(unsigned short* p, long n) {
  for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) p[e] = 0;
}

void ladder_vpm_pack(unsigned short* hi, unsigned short* lo, const float* Y, long ldY, int a0, int a1, int v,
                     long Rp, long Kp, hipStream_t st) {
  long rows = 0;
  for (int a = a0; a < a1; ++a) rows += v - a;
  const long npv = (long)v * (v + 1) / 2;
  CCGPU_REQUIRE(rows < 65536 && rows <= Rp && npv <= Kp, "ladder_vpm_pack: bad batch");
  check_span(hi, 0, 2 * Rp * Kp - 1, sizeof(unsigned short), "ladder_vpm_pack hi");
  check_span(lo, 0, 2 * Rp * Kp - 1, sizeof(unsigned short), "ladder_vpm_pack lo");
  check_span(Y, 0, ((long)(a1 - a0) * v - 1) * ldY + (long)(v - a0) * v - 1, sizeof(float), "ladder_vpm_pack Y");
  CCGPU_REQUIRE(ldY >= (long)(v - a0) * v, "ladder_vpm_pack: ldY too small");
  CCGPU_REQUIRE(v < 32 * 65536, "ladder_vpm_pack: virtual space too large");
  const long nblk = (long)cdiv(v, 128) * cdiv(v, 32) * cdiv(rows, 8) * 8;
  CCGPU_REQUIRE(nblk < (1L << 24), "ladder_vpm_pack: grid too large");
  const dim3 grid((unsigned)nblk);
  if (v % 4 == 0 && ldY % 4 == 0 && reinterpret_cast<uintptr_t>(Y) % 16 == 0)
    CCGPU_LAUNCH(k_ladder_vpm_pack<true>, grid, dim3(256), 0, st, hi, lo, Y, ldY, a0, v, rows, Rp, Kp);
  else
    CCGPU_LAUNCH(k_ladder_vpm_pack<false>, grid, dim3(256), 0, st, hi, lo, Y, ldY, a0, v, rows, Rp, Kp);
  // padding rows of both halves
  const long pad = (Rp - rows) * Kp;
  if (pad > 0) {
    const unsigned nb = (unsigned)std::min<long>(4096, (pad + 255) / 256);
    for (int s = 0; s < 2; ++s) {
      CCGPU_LAUNCH(k_fill_u16, dim3(nb), dim3(256), 0, st, hi + (s * Rp + rows) * Kp, pad);
      CCGPU_LAUNCH(k_fill_u16, dim3(nb), dim3(256), 0, st, lo + (s * Rp + rows) * Kp, pad);
    }
  }
  CCGPU_HIPX(hipGetLastError());
}
}  // namespace ccgpu
