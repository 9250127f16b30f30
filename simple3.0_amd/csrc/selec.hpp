// selec.hpp - the reference's quickselect, by one thread and by one wavefront.
#pragma once

namespace pfk {

// selec (simple_math.f90:2204-2261), restated step for step on an LDS array (1-based indices as
// the reference's; arr permuted in place).  Its final test compares ir - 1 with 1.
__host__ __device__ inline float prep_selec(int k, int n, float* arr) {
  int l = 1, ir = n;
  auto A = [&](int i) -> float& { return arr[i - 1]; };
  for (;;) {
    if (ir - l <= 1) {
      if (ir - 1 == 1 && A(ir) < A(l)) {
        const float t = A(l);
        A(l) = A(ir);
        A(ir) = t;
      }
      return A(k);
    }
    const int mid = (l + ir) / 2;
    float t = A(mid);
    A(mid) = A(l + 1);
    A(l + 1) = t;
    if (A(l) > A(ir)) { t = A(l); A(l) = A(ir); A(ir) = t; }
    if (A(l + 1) > A(ir)) { t = A(l + 1); A(l + 1) = A(ir); A(ir) = t; }
    if (A(l) > A(l + 1)) { t = A(l); A(l) = A(l + 1); A(l + 1) = t; }
    int i = l + 1, j = ir;
    const float a = A(l + 1);
    for (;;) {
      do { ++i; } while (A(i) < a);
      do { --j; } while (A(j) > a);
      if (j < i) break;
      t = A(i);
      A(i) = A(j);
      A(j) = t;
    }
    A(l + 1) = A(j);
    A(j) = a;
    if (j >= k) ir = j - 1;
    if (j <= k) l = i;
  }
}

// The same selection by one wavefront, with the same array afterwards: a partition's scans become
// two lists of the positions where they stop, ascending from the left (!(A < a)) and descending from
// the right (!(A > a)), and its exchanges the pairs of list entries that have not crossed.  The
// scans' last stops are the next entries of their lists, or positions that an exchange has filled
// if those come first.  ls, rs: n ints each.  wave: its lanes call this together (lane, ballot over the
// lanes, sync: the lanes' writes are seen).
template <typename Wave>
__host__ __device__ inline float prep_selec_wave(const Wave& wave, int k, int n, float* arr, int* ls, int* rs) {
  const int lane = wave.lane();
  const unsigned long long below = (1ull << lane) - 1;
  int l = 1, ir = n;
  float* A = arr - 1;
  for (;;) {
    wave.sync();
    if (ir - l <= 1) {
      if (ir - 1 == 1) {
        const float x = A[l], y = A[ir];
        wave.sync();
        if (y < x && lane == 0) {
          A[l] = y;
          A[ir] = x;
        }
        wave.sync();
      }
      return A[k];
    }
    const int mid = (l + ir) / 2;
    const float vm = A[mid], v1 = A[l + 1];
    float x0 = A[l], x1 = vm, x2 = A[ir], t;
    if (x0 > x2) { t = x0; x0 = x2; x2 = t; }
    if (x1 > x2) { t = x1; x1 = x2; x2 = t; }
    if (x0 > x1) { t = x0; x0 = x1; x1 = t; }
    const float a = x1;
    wave.sync();
    if (lane == 0) {
      A[mid] = v1;
      A[l] = x0;
      A[l + 1] = x1;
      A[ir] = x2;
    }
    wave.sync();
    int nl = 0, nr = 0;
    for (int b = l + 2; b <= ir; b += 64) {
      const int p = b + lane;
      const bool stop = p <= ir && !(A[p <= ir ? p : ir] < a);
      const unsigned long long m = wave.ballot(stop);
      if (stop) ls[nl + __builtin_popcountll(m & below)] = p;
      nl += __builtin_popcountll(m);
    }
    for (int b = ir - 1; b > l; b -= 64) {
      const int p = b - lane;
      const bool stop = p > l && !(A[p > l ? p : l + 1] > a);
      const unsigned long long m = wave.ballot(stop);
      if (stop) rs[nr + __builtin_popcountll(m & below)] = p;
      nr += __builtin_popcountll(m);
    }
    wave.sync();
    const int nm = nl < nr ? nl : nr;
    int T = 0;                               // exchanges: entries that have not crossed
    for (int b = 0; b < nm; b += 64) {
      const int q = b + lane;
      T += __builtin_popcountll(wave.ballot(q < nm && ls[q < nl ? q : nl - 1] <= rs[q < nr ? q : nr - 1]));
    }
    for (int b = 0; b < T; b += 64) {
      const int q = b + lane;
      if (q < T) {
        const float x = A[ls[q]], y = A[rs[q]];
        A[ls[q]] = y;
        A[rs[q]] = x;
      }
    }
    int i = ls[T], j = rs[T];
    const int q = T > 0 && ls[T - 1] == rs[T - 1] ? T - 2 : T - 1;
    if (q >= 0) {
      i = rs[q] < i ? rs[q] : i;
      j = ls[q] > j ? ls[q] : j;
    }
    wave.sync();
    if (lane == 0) {
      A[l + 1] = A[j];
      A[j] = a;
    }
    if (j >= k) ir = j - 1;
    if (j <= k) l = i;
  }
}

}  // namespace pfk
