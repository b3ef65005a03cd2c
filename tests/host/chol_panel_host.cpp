// Host build of the pivoted Cholesky's column pass: one block of 256 threads,
// LDS as statics (which keep what the last block left in them, as LDS does),
// barriers that count exited threads as arrived.  The threads are released in
// waves, and the stop flag is raised between two of them, as block 0 of a
// launch may raise it while a later block of the same launch is starting.
#include <cmath>
#include <condition_variable>
#include <cstdio>
#include <mutex>
#include <thread>
#include <vector>

#define __global__
#define __device__
#define __forceinline__ inline
#define __launch_bounds__(n)
#define __shared__ static

namespace {
struct Dim {
  int x = 0;
};
thread_local Dim threadIdx;
thread_local Dim blockIdx;
const Dim blockDim{256}, gridDim{8};

// A group of threads that meet; one that has left counts as arrived.
struct Meet {
  std::mutex mu;
  std::condition_variable cv;
  int alive = 0, in = 0;
  long round = 0;
  void open() {
    if (in < alive || alive == 0) return;
    in = 0;
    ++round;
    cv.notify_all();
  }
  void wait() {
    std::unique_lock<std::mutex> lk(mu);
    ++in;
    const long r = round;
    open();
    cv.wait(lk, [&] { return round != r; });
  }
  void leave() {
    std::lock_guard<std::mutex> lk(mu);
    --alive;
    open();
  }
};
Meet block_meet, wave_meet[4];
double lane_val[256];

void __syncthreads() { block_meet.wait(); }
template <typename T>
T exchange(T v, int from) {
  Meet& m = wave_meet[threadIdx.x / 64];
  reinterpret_cast<T*>(lane_val)[threadIdx.x] = v;
  m.wait();
  const T r = reinterpret_cast<T*>(lane_val)[threadIdx.x / 64 * 64 + from % 64];
  m.wait();
  return r;
}
template <typename T>
T __shfl_xor(T v, int off, int) {
  return exchange(v, threadIdx.x % 64 ^ off);
}
template <typename T>
T __shfl_down(T v, int off, int) {
  return exchange(v, threadIdx.x % 64 + off < 64 ? threadIdx.x % 64 + off : threadIdx.x % 64);
}
}  // namespace

#include "chol_panel.h"

namespace {
constexpr long M = 512;
struct State {
  std::vector<double> L, d, R, pin, pout;
  long st[2] = {0, 0};
};
State make(double big, double small) {  // 8 partials per block, the largest diagonal in the last one
  State s;
  s.L.assign(64 * M, 0.25);
  s.d.assign(M, small);
  s.R.assign(M * M, 0.5);
  s.pin.assign(2 * 256, 0.0);
  for (int q = 0; q < 256; ++q) {
    s.pin[2 * q] = q == 255 ? big : small;
    s.pin[2 * q + 1] = 2 * q;
  }
  s.pout.assign(2 * 8, -7.0);
  return s;
}
// One block of the pass; the waves whose bit in first is set start (and run up
// to the block's barrier or the end) before the flag is raised, the others after.
void run(State& s, int block, unsigned first, bool raise, double thr) {
  block_meet.alive = 256;
  block_meet.in = 0;
  std::mutex mu;
  std::condition_variable cv;
  int phase = 0, ended[2] = {0, 0}, n[2] = {0, 0};
  for (Meet& m : wave_meet) m.alive = 64, m.in = 0;
  std::vector<std::thread> th;
  for (int t = 0; t < 256; ++t) {
    const int ph = first >> (t / 64) & 1 ? 1 : 2;
    ++n[ph - 1];
    th.emplace_back([&, t, ph] {
      {
        std::unique_lock<std::mutex> lk(mu);
        cv.wait(lk, [&] { return phase >= ph; });
      }
      threadIdx.x = t;
      blockIdx.x = block;
      ccgpu::k_chol_panel_col(s.L.data(), s.d.data(), s.R.data(), s.pin.data(), 256, s.st, M, 0, 3, thr,
                              s.pout.data());
      wave_meet[t / 64].leave();
      block_meet.leave();
      std::lock_guard<std::mutex> lk(mu);
      ++ended[ph - 1];
    });
  }
  auto go = [&](int ph) {
    std::lock_guard<std::mutex> lk(mu);
    phase = ph;
    cv.notify_all();
  };
  go(1);
  while (true) {  // every wave of the first set has ended or waits for the others
    std::lock_guard<std::mutex> lk(mu);
    std::lock_guard<std::mutex> lb(block_meet.mu);
    if (ended[0] + block_meet.in == n[0] || ended[0] == n[0]) break;
  }
  if (raise) s.st[0] = 1;
  go(2);
  for (auto& x : th) x.join();
}
}  // namespace

int main() {
  const double thr = 1e-6;
  int bad = 0;
  for (unsigned first = 0; first < 16; ++first) {
    State live = make(5.0, 0.5);  // a step that runs leaves its pivot in LDS
    run(live, 0, 15, false, thr);
    if (live.st[1] != 4 || live.pout[0] < 0.0) {
      std::printf("running step: vectors %ld partial %g\n", live.st[1], live.pout[0]);
      return 1;
    }
    State s = make(1e-9, 1e-10), ref = make(1e-9, 1e-10);  // nothing above the threshold: the stop
    run(s, 5, first, true, thr);
    const bool same = s.L == ref.L && s.d == ref.d && s.pout == ref.pout && s.st[1] == 0;
    if (!same) {
      std::printf("waves %x before the flag: the step after the stop ran with pivot value of the last step\n", first);
      ++bad;
    }
  }
  std::printf("%d of 16 orders wrong\n", bad);
  return bad ? 1 : 0;
}
