// prep_selec_wave on the CPU: 64 lanes as coroutines that meet at every sync and ballot, against prep_selec
// on arrays with many ties, infinities, NaN and sorted runs.  Prints the number of differing cases.
#include <ucontext.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#define __host__
#define __device__
#include "selec.hpp"

namespace {
constexpr int kLanes = 64;
ucontext_t main_ctx, ctx[kLanes];
std::vector<char> stacks[kLanes];
int current;
bool finished[kLanes];
unsigned long long votes[2];
struct Call {
  int k, n;
  float* arr;
  int *ls, *rs;
  float out[kLanes];
} call;

// Every lane runs up to its next meeting point, lane after lane, in ascending or descending order in turn.
struct HostWave {
  mutable int round = 0;
  int lane() const { return current; }
  void sync() const { swapcontext(&ctx[current], &main_ctx); }
  unsigned long long ballot(bool b) const {
    unsigned long long& v = votes[round++ & 1];
    if (b) v |= 1ull << current;
    sync();
    const unsigned long long got = v;
    votes[round & 1] = 0;        // the next ballot's, before any lane can vote in it
    sync();
    return got;
  }
};
void lane_main() {
  HostWave w;
  call.out[current] = pfk::prep_selec_wave(w, call.k, call.n, call.arr, call.ls, call.rs);
  finished[current] = true;
}
// false: lanes disagree about the meeting points or the result
bool run(bool& done_together) {
  votes[0] = votes[1] = 0;
  for (int l = 0; l < kLanes; ++l) {
    finished[l] = false;
    getcontext(&ctx[l]);
    ctx[l].uc_stack.ss_sp = stacks[l].data();
    ctx[l].uc_stack.ss_size = stacks[l].size();
    ctx[l].uc_link = &main_ctx;
    makecontext(&ctx[l], lane_main, 0);
  }
  for (int step = 0;; ++step) {
    int done = 0;
    for (int i = 0; i < kLanes; ++i) {
      current = step & 1 ? kLanes - 1 - i : i;
      swapcontext(&main_ctx, &ctx[current]);
      done += finished[current];
    }
    if (done) {
      done_together = done == kLanes;
      break;
    }
  }
  for (int l = 1; l < kLanes; ++l)
    if (memcmp(&call.out[l], &call.out[0], 4)) return false;
  return done_together;
}
}  // namespace

int main(int, char** argv) {
  const int cases = atoi(argv[1]);
  for (auto& s : stacks) s.resize(64 << 10);
  std::mt19937 rng(1);
  auto below = [&](int n) { return (int)(rng() % (unsigned)n); };
  long bad = 0;
  for (int it = 0; it < cases; ++it) {
    const int n = 4 + 2 * below(it % 10 == 0 ? 250 : 60), mode = it % 6, k = n / 2;
    std::vector<float> a(n);
    for (float& v : a) {
      if (mode == 0) v = (float)rng() / 4294967296.0f;
      else if (mode == 1) v = (float)below(3);
      else if (mode == 2) v = (float)below(8);
      else if (mode == 3) v = below(20) == 0 ? NAN : (float)below(50);
      else if (mode == 4) v = below(10) == 0 ? (below(2) ? INFINITY : -INFINITY) : (float)below(100) - 50.0f;
      else v = 1.0f;
    }
    if (below(10) == 0) std::sort(a.begin(), a.end(), [](float x, float y) { return x < y; });
    std::vector<float> b = a;
    std::vector<int> ls(n), rs(n);
    const float x = pfk::prep_selec(k, n, a.data());
    call = Call{k, n, b.data(), ls.data(), rs.data(), {}};
    bool together = false;
    const bool same = run(together);
    if (!same || memcmp(&x, &call.out[0], 4) || memcmp(a.data(), b.data(), 4 * (size_t)n)) ++bad;
  }
  printf("%ld of %d differ\n", bad, cases);
  return bad != 0;
}
