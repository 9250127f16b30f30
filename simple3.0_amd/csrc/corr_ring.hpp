// corr_ring.hpp - the plain FP32 correlation search with two-pass ring transforms.
//
// One work-group correlates one particle with F (reference, shift) pairs, shell by shell.  The
// packed length-N transform of a pair's shell runs as N = A B (ring_fft.hpp):
//  * pass 1 (radix A, A = 2 H): butterfly t3 builds q = ref x |CTF| [x shift] [x shell scale] at its
//    H pairs (q[2h], q[2h+1]), h = t1 B + t3, and leaves output k1 at LDS position (k1, t3);
//  * last pass (radix B) on the mirrored rows g and A - g, in one thread (RP = 2) or in two
//    neighbouring lanes that exchange their outputs (RP = 1, half the registers): bin m = g + A t of
//    row g and bin N - m of row A - g meet there, where the real-FFT split and the product with the
//    particle's spectrum accumulate over the shells.
// The split is folded into the staged particle spectrum: with Z the transform of the halved sums
// (dft_even_odd), conj(V[m]) W[m] = conj(Z[m]) conj(A') W + Z[N-m] conj(B') W, A' = 1 - i w_m,
// B' = 1 + i w_m, w_m = exp(-i pi m / N): 8 FMAs per bin and pair.
// The mirrored row of g = 0 is row 0 transformed with the twiddles of row A: that shifts its outputs
// by one, so bin N - m sits at the same place as in every other group (and its last output is the
// Nyquist bin); no lane takes a branch in the shell loop.
// Two barriers per shell: the shell's spectra are written beside pass 1 (the previous last pass has
// finished), the next shell's reference rows or |CTF| beside the last pass.
// Bound: VALU issue and the LDS exchange beside it, three wavefronts per SIMD hiding the latency; HBM
// traffic is small.  Against four to six LDS passes of radix 4 to 11 (radix-4 first, one barrier
// each) the two register passes take a third of the LDS accesses: 256 particles x 100 references
// x 49 shifts at n 308, 59 shells: 40.2 -> 32.3 ms; 200 x 1500 at n 400, 79 shells: 24.0 -> 13.5 ms
// (VALU busy 0.89, 1.03 at n 220); against runtime-size passes 200 x 50 x 25 at n 220, 44
// shells: 26.1 -> 2.9 ms, and 150 x 500 (Euclid) at n 364, 71 shells: 17.3 -> 3.9 ms.
#pragma once
#include <type_traits>

#include "corr_args.hpp"
#include "ring_fft.hpp"

namespace pfk {

// Loads from an array at a uniform base by a 32-bit byte offset, which lets the load take the
// base from scalar registers: ld16 reads elements elem and elem + 1 of a float2 array.
__device__ __forceinline__ float4 ld16(const float2* __restrict__ base, unsigned int elem) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(base) + (elem << 3));
}
__device__ __forceinline__ float2 ld8(const float2* __restrict__ base, unsigned int elem) {
  return *reinterpret_cast<const float2*>(reinterpret_cast<const char*>(base) + (elem << 3));
}
// 16 bytes at a uniform base plus a 32-bit byte offset plus a constant: one instruction, no address
// arithmetic per load.
__device__ __forceinline__ float4 ld16b(const void* __restrict__ base, unsigned int off, int imm) {
  return *reinterpret_cast<const float4*>(static_cast<const char*>(base) + off + imm);
}
__device__ __forceinline__ float ldf(const float* __restrict__ base, unsigned int elem) {
  return *reinterpret_cast<const float*>(reinterpret_cast<const char*>(base) + (elem << 2));
}

// Ring lengths that had compile-time kernels before the table of lengths (ring_table.hpp).  Results
// recorded with them stay as they are: their sums (ring_apart), their callback's order of operations
// (rings.hip) and their FP16 spectra in the FP8 coarse pass (mfma_group).
constexpr bool ring_first(int n) {
  for (int m : {16, 24, 32, 40, 48, 64, 100, 192, 240, 308, 400, 500, 600})
    if (n == m) return true;
  return false;
}

// Whether a shell's product is formed on its own and then added to the sum over the shells, as the
// runtime-size kernel does, instead of by multiply-adds onto the sum: one rounding of the sum per shell
// and component instead of four, for two additions per bin.  Relative error of 5760 correlation vectors
// against FP64: n 220 3.5e-7 -> 2.3e-7 (runtime-size kernel 2.5e-7), n 450 4.9e-7 -> 2.8e-7 (3.0e-7); the first
// lengths' kernels always added onto the sum (n 400 4.5e-7).  200 particles x 50 references x 25 shifts
// at n 220: 2.81 -> 2.92 ms; 150 x 500 at n 364: 4.04 -> 4.02 ms.
constexpr bool ring_apart(int n) { return !ring_first(n); }

// conj(Z) w1 + Zn w2, the split and the product conj(V) W of one bin with the split's m-dependent
// factors folded into w1 = conj(A') W and w2 = conj(B') W: onto acc (APART: formed apart and added).
template <bool APART>
__device__ __forceinline__ void acc_w12(float2& acc, float2 Z, float2 Zn, float4 w) {
  float2 p = APART ? make_float2(Z.x * w.x, Z.x * w.y) : make_float2(fmaf(Z.x, w.x, acc.x), fmaf(Z.x, w.y, acc.y));
  p.x = fmaf(Z.y, w.y, p.x);
  p.y = fmaf(-Z.y, w.x, p.y);
  p.x = fmaf(Zn.x, w.z, p.x);
  p.x = fmaf(-Zn.y, w.w, p.x);
  p.y = fmaf(Zn.x, w.w, p.y);
  p.y = fmaf(Zn.y, w.z, p.y);
  acc = APART ? cadd(acc, p) : p;
}

// (w1, w2) of acc_w12 at a bin with spectrum value w, shell weight wk and t = exp(-i pi m / N).
__device__ __forceinline__ float4 spec_w12(float2 w, float wk, float2 t) {
  const float2 wh = make_float2(wk * w.x, wk * w.y);
  const float2 w1 = cmul(make_float2(1.f + t.y, t.x), wh), w2 = cmul(make_float2(1.f - t.y, -t.x), wh);
  return make_float4(w1.x, w1.y, w2.x, w2.y);
}

// Particle's share of the normalisation: the sum of squares, or (Euclid) of the weighted shells'.
__device__ __forceinline__ float ring_pscal(const CorrArgs& a, int ip) {
  if (a.mode != 1) return a.sqsums[ip];
  float s = 0.f;
  for (int kk = 0; kk < a.kcorr; ++kk) s += a.shellw[(size_t)ip * a.nk + kk] * a.sqsums_k[(size_t)ip * a.nk + kk];
  return s;
}

// Y[m] of the inverse real FFT from X[m] and X[N-m]; e = exp(+i pi m / N).  Returns conj(Y).
__device__ __forceinline__ float2 unsplit_bin_conj(float2 X, float2 Xn, float2 e) {
  const float2 s = make_float2(X.x + Xn.x, X.y - Xn.y);
  const float2 d = make_float2(X.x - Xn.x, X.y + Xn.y);
  const float2 ed = cmul(e, d);
  return make_float2(s.x - ed.y, -(s.y + ed.x));
}

// Geometry of a two-pass transform N = A B and its LDS layout: position (k1, t3) at k1 SB + t3.
// SB is odd, so that the lanes of the last pass (consecutive rows) spread over the banks.
template <int N, int A>
struct RingGeom {
  static constexpr int B = N / A, H = A / 2, SB = B | 1, S = A * SB, G = H + 1;
  static constexpr int TW = (B - 1) * (A + 1);   // last-pass twiddles tw[t - 1][k1] = exp(-2 pi i k1 t / N), k1 <= A
  static_assert(A * B == N && A % 2 == 0, "N = A B with A even");
  // Good-Thomas form (A, B coprime), used where the operands can be stored in its order: input
  // u = (B t1 + A t3) mod N, output m = k1 mod A = k3 mod B, no twiddles between the passes.
  static constexpr bool coprime = cx_gcd(A, B) == 1;
  static constexpr int IA = cx_modinv(A % B, B), IB = cx_modinv(B % A, A);
  // slot of the q pair (q[2h], q[2h+1]): pass-1 lane order t1 B + t3 with t1 < H.  neg: z[u], z[u + N/2]
  // come in the other order, so the difference changes sign: the pair is stored conjugated.
  static __host__ __device__ __forceinline__ int pfa_slot(int h, bool& neg) {
    const int t1 = (h * IB) % A, t3 = (h * IA) % B;
    neg = t1 >= H;
    return (neg ? t1 - H : t1) * B + t3;
  }
  static __device__ __forceinline__ int pfa_bin(int k1, int k3) { return (k1 * B * IB + k3 * A * IA) % N; }
  // staged spectrum bin m: [k3][A + 1], the Nyquist bin at k1 = A, k3 = 0
  static __device__ __forceinline__ int pfa_wpos(int m) { return m == N ? A : (m % B) * (A + 1) + m % A; }
};

// Reference rows a tile of the staged-reference variant may span (their prefetch takes registers,
// twice as many past N = 256), and the fewest shifts with which its F pairs span no more.
constexpr int ring_rows(int N, int F, int RP) {
  const int most = N <= 256 ? 5 : RP == 2 ? 3 : 4, use = 1 + (F + 3) / 4;
  return use < most ? use : most;
}
constexpr int ring_min_shifts(int N, int F, int RP) {
  return (F + ring_rows(N, F, RP) - 2) / (ring_rows(N, F, RP) - 1);
}

template <int N, int A, int NT>
__device__ __forceinline__ void ring_twiddles(float2* __restrict__ tw, const float2* __restrict__ tw2g, int tid) {
  using R = RingGeom<N, A>;
  for (int i = tid; i < R::TW; i += NT) {
    const int t = i / (A + 1) + 1, k1 = i % (A + 1);
    tw[i] = tw2g[2 * k1 * t];      // k1 t <= A (B - 1) < N
  }
}

// Value of the neighbouring lane (lanes 2 i and 2 i + 1 swap).
__device__ __forceinline__ float lane_swap(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0xB1, 0xf, 0xf, true));   // quad_perm [1, 0, 3, 2]
}
__device__ __forceinline__ float2 lane_swap(float2 v) { return make_float2(lane_swap(v.x), lane_swap(v.y)); }

// acc_w12 with Zn the neighbouring lane's Zm, read by the multiply-adds themselves (a quad permutation
// of their first operand) instead of by two moves: 80 of 977 instructions of a shell at n 400.  The
// leading wait covers the hazard between the instruction that wrote Zm and the first that permutes it.
template <bool APART>
__device__ __forceinline__ void acc_w12_swap(float2& acc, float2 Z, float2 Zm, float4 w) {
  float2 p = APART ? make_float2(Z.x * w.x, Z.x * w.y) : make_float2(fmaf(Z.x, w.x, acc.x), fmaf(Z.x, w.y, acc.y));
  p.x = fmaf(Z.y, w.y, p.x);
  p.y = fmaf(-Z.y, w.x, p.y);
  asm("s_nop 1\n\t"
      "v_fmac_f32_dpp %0, %2, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %2, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %0, -%3, %5 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t"
      "v_fmac_f32_dpp %1, %3, %4 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf"
      : "+v"(p.x), "+v"(p.y)
      : "v"(Zm.x), "v"(Zm.y), "v"(w.z), "v"(w.w));
  acc = APART ? cadd(acc, p) : p;
}

// Row k1 (0 .. A, row A being row 0 with its outputs shifted by one) of one transform (buf at the
// transform's base) through the last pass (PFA: no twiddles).
template <int N, int A, bool PFA>
__device__ __forceinline__ void ring_last_row(const float2* __restrict__ buf, const float2* __restrict__ tw, int row,
                                              float2 (&y)[N / A]) {
  using R = RingGeom<N, A>;
  const float2* r = buf + (row == A ? 0 : row) * R::SB;
  static_for<0, R::B>([&](auto t) { y[decltype(t)::value] = r[decltype(t)::value]; });
  if constexpr (!PFA)
    static_for<1, R::B>([&](auto t) {
      constexpr int T = decltype(t)::value;
      y[T] = cmul(y[T], tw[(T - 1) * (A + 1) + row]);
    });
  RDft<R::B>::run(y);
}

// Last-pass tasks of a transform: RP = 2: G = A / 2 + 1 tasks, rows g and A - g each; RP = 1: 2 G tasks,
// row g in lane 2 g and row A - g in lane 2 g + 1.
template <int A, int RP>
__device__ __forceinline__ int ring_row(int r) {
  return RP == 2 ? r : (r & 1) ? A - (r >> 1) : (r >> 1);
}

// Output of one pair's transform: normalised values to cc_out, the best (cc, first position) into key.
struct RingEmit {
  float scale, off;
  int n;
  __device__ __forceinline__ RingEmit(const CorrArgs& a, int n, float sq, float o, float ps) : off(o + ps), n(n) {
    const float inv4n = 1.0f / (4.0f * (float)n);
    scale = a.mode == 1 ? inv4n : inv4n / sqrtf(sq * ps);
  }
  // output m of particle slot pi's pair P: rotations 2 m and 2 m + 1
  __device__ __forceinline__ void operator()(const CorrArgs& a, int pi, int npairs, int P, int m, float2 y,
                                             unsigned long long& key) const {
    float x0 = y.x, x1 = -y.y;
    if (a.mode == 1) {
      x0 = 2.f * x0 * scale - off;
      x1 = 2.f * x1 * scale - off;
    } else {
      x0 *= scale;
      x1 *= scale;
    }
    if (a.cc_out) reinterpret_cast<float2*>(a.cc_out + ((size_t)pi * npairs + P) * (2 * n))[m] = make_float2(x0, x1);
    if (a.best) {
      const unsigned int lin0 = (unsigned int)P * (unsigned int)(2 * n) + 2u * m;
      const unsigned long long k0 = ((unsigned long long)ordered_bits(x0) << 32) | (0xFFFFFFFFu - lin0);
      const unsigned long long k1 = ((unsigned long long)ordered_bits(x1) << 32) | (0xFFFFFFFFu - lin0 - 1u);
      key = k0 > key ? k0 : key;
      key = k1 > key ? k1 : key;
    }
  }
};

// The work-group's best key into *best: wavefront maxima, then the wavefronts' in a fixed order.
template <int NT>
__device__ __forceinline__ void ring_best(unsigned long long* best, unsigned long long key, unsigned long long* red,
                                          int tid) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long v = __shfl_xor(key, o);
    key = v > key ? v : key;
  }
  if ((tid & 63) == 0) red[tid >> 6] = key;
  __syncthreads();
  if (tid == 0) {
    unsigned long long m = red[0];
    for (int w = 1; w < NT / 64; ++w) m = red[w] > m ? red[w] : m;
    atomicMax(best, m);
  }
}

// Inverse real transform of F accumulated spectra held as acc[slot][RP B] by the tasks of the last
// pass: emit(f, m, y) gets output m, rotations 2m (y.x) and
// 2m + 1 (-y.y).  buf is free; every thread of the work-group calls it.
template <int N, int A, int F, int NT, int RP, int TPTL, bool PFA, typename Emit>
__device__ __forceinline__ void ring_inverse(const float2 (&acc)[TPTL][RP * (N / A)], float2* __restrict__ buf,
                                             const float2* __restrict__ tw, const float2* __restrict__ tw2g, int tid,
                                             Emit&& emit) {
  using R = RingGeom<N, A>;
  constexpr int B = R::B, TF = RP == 2 ? R::G : 2 * R::G, TL = F * TF;
  auto put = [&](int f, int m, float2 X, float2 Xn) {
    if (m == 0) {
      X.y = 0.f;
      Xn.y = 0.f;
    }
    buf[f * R::S + (m / B) * R::SB + m % B] = unsplit_bin_conj(X, Xn, cconj(tw2g[m]));
  };
  auto bin = [&](int row, int t) { return PFA ? R::pfa_bin(row, t) : row + A * t; };
#pragma unroll
  for (int c = 0; c < TPTL; ++c) {
    const int task = tid + c * NT;
    if (!(TL % NT == 0 || task < TL)) continue;
    const int f = task / TF, row = ring_row<A, RP>(task % TF);
    // mirror of output t: PFA (-k1, -k3), else (A - k1, B - 1 - k3).  PFA row 0: mirrored within
    // itself, but for the Nyquist bin, which row A holds
    static_for<0, B>([&](auto t) {
      constexpr int T = decltype(t)::value, TM = PFA ? (B - T) % B : B - 1 - T;
      float2 Xn;
      if constexpr (RP == 2) Xn = acc[c][B + TM];
      else Xn = lane_swap(acc[c][TM]);
      if constexpr (PFA && T != 0) Xn = make_float2(row == 0 ? acc[c][TM].x : Xn.x, row == 0 ? acc[c][TM].y : Xn.y);
      if (RP == 2 || row != A) put(f, bin(row, T), acc[c][T], Xn);
    });
    if constexpr (RP == 2)
      if (row != 0)
        static_for<0, B>([&](auto t) {
          constexpr int T = decltype(t)::value, TM = PFA ? (B - T) % B : B - 1 - T;
          put(f, bin(A - row, T), acc[c][B + T], acc[c][TM]);
        });
  }
  __syncthreads();
  for (int task = tid; task < F * B; task += NT) {
    const int f = task / B, t3 = task % B;
    float2* p = buf + f * R::S + t3;
    float2 v[A];
    static_for<0, A>([&](auto t) { v[decltype(t)::value] = p[decltype(t)::value * R::SB]; });
    RDft<A>::run(v);
    static_for<0, A>([&](auto t) { p[decltype(t)::value * R::SB] = v[decltype(t)::value]; });
  }
  __syncthreads();
  for (int task = tid; task < F * A; task += NT) {
    const int f = task / A, row = task % A;
    float2 y[B];
    ring_last_row<N, A, false>(buf + f * R::S, tw, row, y);
    static_for<0, B>([&](auto t) { emit(f, row + A * decltype(t)::value, y[decltype(t)::value]); });
  }
}

// A search whose shells are split over work-groups: they leave every shell's transform, zrow
// [pair][kcorr][B][A + 1] (row A as in ring_last_row), and (per-pair variant) its slots' sums |q|^2,
// es [pair][shells][B]; k_ring_finish multiplies and sums them in the order of the unsplit kernel, so a
// pair's result does not depend on the launch.  pair = particle slot x (nr ns) + P.
struct RingSplit {
  int nsplit;                  // shell chunks (1: not split)
  int kper;                    // shells per chunk
  float2* zrow;
  float* es;
};

// The staged-reference kernel takes the Good-Thomas form where it can: its operands (staged rows,
// shift table) are stored in that order.
template <int N, int A, bool RST>
constexpr bool ring_pfa() { return RST && RingGeom<N, A>::coprime; }

// float4 entries of the staged spectra
template <int N, int A, bool RST>
constexpr int ring_wlen() { return ring_pfa<N, A, RST>() ? RingGeom<N, A>::B * (A + 1) : N + 1; }

// rows: staged reference rows (RST): as many as a tile of F pairs can span with ns shifts, so that a
// search with many shifts leaves LDS for more work-groups per CU.
constexpr int ring_span(int F, int ns) { return 1 + (F - 1 + ns - 1) / ns; }
template <int N, int A, int F, int NT, bool RST>
constexpr size_t ring_lds_bytes(int rows) {
  using R = RingGeom<N, A>;
  return 16 * (size_t)ring_wlen<N, A, RST>() +
         8 * (size_t)((F * R::S + (ring_pfa<N, A, RST>() ? 0 : R::TW) + 1) / 2 * 2 + (RST ? rows * N : (N + 1) / 2));
}

// W: minimum wavefronts per SIMD the register allocation must allow.
// RST: shifted CC search without shell normalisation whose tiles span at most ring_rows
// references: the shell's CTF-weighted reference rows are staged once per work-group in LDS and each
// reference's norm is summed from them (|ref x CTF x shmat|^2 = |ref x CTF|^2), instead of per pair.
// PRF (per-pair variant): pass 1 loads its reference values a shell ahead.
// SPLIT: only the transforms, of the shells of one chunk (RingSplit).
template <int N, int A, int F, int NT, int W, int RP, bool RST, bool PRF, bool SPLIT>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(W))) k_corr_ring(CorrArgs a, RingSplit sp) {
  static_assert(!(RST && PRF), "the staged variant loads its shift phases where it uses them");
  using R = RingGeom<N, A>;
  constexpr int B = R::B, H = R::H, S = R::S;
  constexpr int T1 = F * B, TPT1 = (T1 + NT - 1) / NT;
  constexpr int TF = RP == 2 ? R::G : 2 * R::G;     // last-pass tasks per transform
  constexpr int TL = F * TF, TPTL = (TL + NT - 1) / NT;
  constexpr bool PFA = ring_pfa<N, A, RST>(), APART = ring_apart(N);
  constexpr int WL = ring_wlen<N, A, RST>(), RR = RST ? ring_rows(N, F, RP) : 1;
  constexpr int WS = PFA ? A + 1 : A;        // stride of a row's staged bins
  extern __shared__ __align__(16) float2 smem[];
  float4* Wk4 = reinterpret_cast<float4*>(smem);                       // [WL] (W1, W2)
  float2* buf = reinterpret_cast<float2*>(Wk4 + WL);                   // [F][S]
  float2* tw = PFA ? smem : buf + F * S;     // PFA: for the inverse only, over the spectra
  float2* rck = buf + (F * S + (PFA ? 0 : R::TW) + 1) / 2 * 2;         // RST: [<= RR][N] ref x |CTF|
  float* ctfk = reinterpret_cast<float*>(rck);                         // else: [N] |CTF|
  __shared__ float sq[F], off[F], pscal;
  __shared__ double rsq[RR][NT / 64];
  __shared__ unsigned long long red[NT / 64];
  static_assert(2 * T1 <= 4 * WL && R::TW <= 2 * WL, "norm sums and twiddles fit the spectra's space");

  // Passes whose tasks do not fill the work-group leave its last wavefront short of work, and the
  // wavefronts of every work-group go to the SIMDs in the same order: work-groups that share a CU
  // start their tasks at different wavefronts.
  const int tid = (threadIdx.x + 64 * (blockIdx.x >> 8)) % NT;
  // each XCD takes a contiguous range of the logical order; within it, the tiles of a group of 16
  // particles are interleaved, so that the work-groups resident together share reference and
  // shift rows in their L2
  constexpr int GRP = 16;
  const int t = xcd_remap(blockIdx.x, gridDim.x);
  const int grp = t / (GRP * a.ntiles);
  const int gsz = min(GRP, a.np - grp * GRP);
  const int rem = t - grp * GRP * a.ntiles;
  const int tile = rem / gsz;
  const int pi = grp * GRP + (rem - tile * gsz);
  const int ip = a.plist[pi];
  const bool even = a.iseven[ip] != 0;
  const float2* refs = even ? a.refs_even : a.refs_odd;
  const int npairs = a.nr * a.ns;
  const int nk = a.nk;
  // tasks of the tile's pairs: the wavefronts past the last pair of a part-filled tile do no work
  // (1000 particles x 50 references at n 192, tiles of 21: 710 -> 660 us)
  const int live = min(F, npairs - tile * F), t1 = live * B, tl = live * TF;
  const bool EUC = !RST && a.mode == 1;
  const int kloop = a.kcorr > a.knorm ? a.kcorr : a.knorm;
  const int kb = SPLIT ? (int)blockIdx.y * sp.kper : 0;
  const int ke = SPLIT ? min(kloop, kb + sp.kper) : kloop;

  if constexpr (!PFA) ring_twiddles<N, A, NT>(tw, a.tw2g, tid);

  // RST: the references the tile spans (uniform: row bases in scalar registers) and this thread's
  // share of their norms
  const int rr0 = RST ? (tile * F) / a.ns : 0;
  const int nrow = RST ? min(a.nr - 1, (min(npairs, (tile + 1) * F) - 1) / a.ns) - rr0 + 1 : 0;
  const float2* rs[RR];
  double rsum[RR];
#pragma unroll
  for (int r = 0; r < RR; ++r) {
    rsum[r] = 0.0;
    const int ir = min(rr0 + r, a.nr - 1);
    rs[r] = refs;
    if constexpr (RST) rs[r] += (size_t)__builtin_amdgcn_readfirstlane(a.rlist ? a.rlist[ir] : ir) * nk * N;
  }
  // pass-1 slots: byte offsets (32 bits) of the pair's reference and shift rows, fixed for all
  // shells
  float sqp[TPT1], offp[TPT1];
  unsigned int roff[TPT1], soff[TPT1];
  int slotref[TPT1];
#pragma unroll
  for (int c = 0; c < TPT1; ++c) {
    const int task = tid + c * NT;
    const int f = task / B, t3 = task % B;
    const int P = tile * F + f;
    sqp[c] = 0.f;
    offp[c] = 0.f;
    roff[c] = (RST ? 2u : 16u) * t3;
    soff[c] = (RST ? 2u : 16u) * t3;
    slotref[c] = 0;
    if (task < T1 && P < npairs) {
      const int ir = P / a.ns, is = P % a.ns;
      const int iref = a.rlist ? a.rlist[(size_t)pi * a.rlist_ld + ir] : ir;
      slotref[c] = iref;
      if constexpr (RST) roff[c] += (unsigned int)((ir - rr0) * N);
      else roff[c] += (unsigned int)iref * (unsigned int)(nk * N * 8);
      soff[c] += (unsigned int)is * (unsigned int)(nk * N * (RST ? 1 : 8));
    }
  }
  float2 acc[TPTL][RP * B];
#pragma unroll
  for (int c = 0; c < TPTL; ++c)
#pragma unroll
    for (int b = 0; b < RP * B; ++b) acc[c][b] = make_float2(0.f, 0.f);

  // the staging operands of the next shell: |CTF| and (RST) two reference rows; the particle's
  // spectrum, with the split's factors (constant over the shells) in registers
  constexpr int JP = (N + NT - 1) / NT, MP = (N + NT) / NT;
  float pcv[JP];
  float2 prr[RR][JP], pwm[MP], twm[MP];
  unsigned int jpos[JP];                     // staged position of element j (bit 31: conjugated)
  const float* ctfp = a.ctf ? a.ctf + (size_t)ip * nk * N : nullptr;
  const float2* memop = a.memo + (size_t)ip * nk * (N + 1);
#pragma unroll
  for (int u = 0; u < MP; ++u) {
    const int m = tid + u * NT;
    twm[u] = a.tw2g[m <= N ? m : 0];
  }
#pragma unroll
  for (int u = 0; u < JP; ++u) {
    const int j = min(tid + u * NT, N - 1);
    bool neg = false;
    jpos[u] = PFA ? 2 * R::pfa_slot(j >> 1, neg) + (j & 1) : j;
    if (neg) jpos[u] |= 0x80000000u;
  }
  auto fetch_rows = [&](int k) {
#pragma unroll
    for (int u = 0; u < JP; ++u) {
      const int j = tid + u * NT;
      if (N % NT == 0 || j < N) {
        pcv[u] = ctfp ? ldf(ctfp, (unsigned int)(k * N + j)) : 1.0f;
        if constexpr (RST)
#pragma unroll
          for (int r = 0; r < RR; ++r)
            if (r < nrow) prr[r][u] = ld8(rs[r], (unsigned int)(k * N + j));
      }
    }
  };
  auto fetch_spec = [&](int k) {
    if (!SPLIT && k < a.kcorr)
#pragma unroll
      for (int u = 0; u < MP; ++u) {
        const int m = tid + u * NT;
        if (m <= N) pwm[u] = ld8(memop, (unsigned int)(k * (N + 1) + m));
      }
  };
  auto stage_rows = [&]() {
#pragma unroll
    for (int u = 0; u < JP; ++u) {
      const int j = tid + u * NT;
      if (N % NT == 0 || j < N) {
        if constexpr (RST) {
          // these searches' norms cover every shell
          const float cv = pcv[u];
          const unsigned int sgn = jpos[u] & 0x80000000u;
          const unsigned int jp = jpos[u] & 0x7fffffffu;
#pragma unroll
          for (int r = 0; r < RR; ++r)
            if (r < nrow) {
              const float2 q = make_float2(prr[r][u].x * cv, prr[r][u].y * cv);
              rck[r * N + jp] = make_float2(q.x, __uint_as_float(__float_as_uint(q.y) ^ sgn));
              rsum[r] += (double)fmaf(q.y, q.y, q.x * q.x);
            }
        } else {
          ctfk[j] = pcv[u];
        }
      }
    }
  };
  float4 pre[PRF ? TPT1 : 1][PRF ? H : 1];
  if (kb < ke) {
    fetch_rows(kb);
    fetch_spec(kb);
    if constexpr (PRF)
#pragma unroll
      for (int c = 0; c < TPT1; ++c)
        if (tid + c * NT < t1)
#pragma unroll
          for (int h = 0; h < H; ++h) pre[c][h] = ld16b(refs + (size_t)kb * N, roff[c], 16 * h * B);
    stage_rows();
  }
  __syncthreads();
  for (int kk = kb; kk < ke; ++kk) {
    const bool docorr = kk < a.kcorr;
    const bool donorm = RST || kk < a.knorm;
    const float wk = (EUC && docorr) ? a.shellw[(size_t)ip * nk + kk] : 1.0f;
    if (!SPLIT && docorr)
#pragma unroll
      for (int u = 0; u < MP; ++u) {
        const int m = tid + u * NT;
        if (m <= N) Wk4[PFA ? R::pfa_wpos(m) : m] = spec_w12(pwm[u], wk, twm[u]);
      }
    if (kk + 1 < ke) {
      fetch_rows(kk + 1);
      fetch_spec(kk + 1);
    }
    // ---- pass 1 ----
    // this shell's rows and the next one's (the last shell loads its own again)
    const size_t kN = (size_t)kk * N, kX = (size_t)min(kk + 1, ke - 1) * N;
    const bool filter = a.refinv && docorr;
#pragma unroll
    for (int c = 0; c < TPT1; ++c) {
      const int task = tid + c * NT;
      if (task >= t1) continue;
      const int f = task / B, t3 = task % B;
      float4 q[RST ? 1 : H];                 // pairs (q[2h], q[2h+1])
      float2 E[H], O[H];
      static_for<0, H>([&](auto tt) {
        constexpr int T = decltype(tt)::value;
        if constexpr (RST) {
          const float4 r = *reinterpret_cast<const float4*>(rck + roff[c] + 2 * T * B);
          const float4 s = ld16(a.shtab, soff[c] + (unsigned int)kN + 2 * T * B);
          const float2 q0 = cmul(make_float2(r.x, r.y), make_float2(s.x, s.y));
          const float2 q1 = cmul(make_float2(r.z, r.w), make_float2(s.z, s.w));
          E[T] = make_float2(q0.x, q1.x);
          O[T] = make_float2(q0.y, q1.y);
        } else {
          float4 r;
          if constexpr (PRF) r = pre[c][T];
          else r = ld16b(refs + kN, roff[c], 16 * T * B);
          const float2 cv = *reinterpret_cast<const float2*>(ctfk + 2 * t3 + 2 * T * B);
          q[T] = make_float4(r.x * cv.x, r.y * cv.x, r.z * cv.y, r.w * cv.y);
        }
      });
      if constexpr (!RST)
        if (a.shtab)
          static_for<0, H>([&](auto tt) {
            constexpr int T = decltype(tt)::value;
            const float4 s = ld16b(a.shtab + kN, soff[c], 16 * T * B);
            const float2 q0 = cmul(make_float2(q[T].x, q[T].y), make_float2(s.x, s.y));
            const float2 q1 = cmul(make_float2(q[T].z, q[T].w), make_float2(s.z, s.w));
            q[T] = make_float4(q0.x, q0.y, q1.x, q1.y);
          });
      if constexpr (PRF)
        static_for<0, H>([&](auto tt) {
          constexpr int T = decltype(tt)::value;
          pre[c][T] = ld16b(refs + kX, roff[c], 16 * T * B);
        });
      float e2 = 0.f;
      if constexpr (!RST) {
        if (filter) {
          const int iref = slotref[c];
          const int row = a.optrow ? a.optrow[ip] : iref;
          const float sc = a.ofac[(size_t)row * a.kcorr + kk] *
                           a.refinv[((size_t)(even ? 0 : 1) * a.nrefs + iref) * a.kcorr + kk];
          static_for<0, H>([&](auto tt) {
            constexpr int T = decltype(tt)::value;
            q[T] = make_float4(q[T].x * sc, q[T].y * sc, q[T].z * sc, q[T].w * sc);
          });
        }
        static_for<0, H>([&](auto tt) {
          constexpr int T = decltype(tt)::value;
          e2 = fmaf(q[T].x, q[T].x, e2);
          e2 = fmaf(q[T].y, q[T].y, e2);
          e2 = fmaf(q[T].z, q[T].z, e2);
          e2 = fmaf(q[T].w, q[T].w, e2);
          E[T] = make_float2(q[T].x, q[T].z);
          O[T] = make_float2(q[T].y, q[T].w);
        });
      }
      if constexpr (!RST) {
        if constexpr (SPLIT) sp.es[(((size_t)pi * npairs + tile * F + f) * kloop + kk) * B + t3] = e2;
        if (donorm) sqp[c] += e2;
        if (EUC && docorr) offp[c] = fmaf(wk, e2, offp[c]);
      }
      if (docorr) {
        float2* p = buf + f * S + t3;
        dft_even_odd<A>(E, O, [&](auto k, float2 v) { p[decltype(k)::value * R::SB] = v; });
      }
    }
    __syncthreads();
    if (kk + 1 < ke) stage_rows();
    // ---- last pass, split and product ----
    if (docorr)
#pragma unroll
      for (int c = 0; c < TPTL; ++c) {
        const int task = tid + c * NT;
        if (task >= tl) continue;
        const int f = task / TF, row = ring_row<A, RP>(task % TF);
        float2 y1[B];
        ring_last_row<N, A, PFA>(buf + f * S, tw, row, y1);
        const float4* wa = Wk4 + row;
        if constexpr (SPLIT) {
          static_assert(RP == 1, "a row per task");
          float2* z = sp.zrow + (((size_t)pi * npairs + tile * F + f) * a.kcorr + kk) * (B * (A + 1)) + row;
          static_for<0, B>([&](auto tt) { z[decltype(tt)::value * (A + 1)] = y1[decltype(tt)::value]; });
        } else if constexpr (RP == 2) {
          float2 y2[B];
          ring_last_row<N, A, PFA>(buf + f * S, tw, A - row, y2);
          const float4* wb = Wk4 + A - row;
          static_for<0, B>([&](auto tt) {
            constexpr int T = decltype(tt)::value, TM = PFA ? (B - T) % B : B - 1 - T;
            acc_w12<APART>(acc[c][T], y1[T], y2[TM], wa[WS * T]);
            acc_w12<APART>(acc[c][B + T], y2[T], y1[TM], wb[WS * T]);
          });
        } else {
          static_for<0, B>([&](auto tt) {
            constexpr int T = decltype(tt)::value, TM = PFA ? (B - T) % B : B - 1 - T;
            acc_w12_swap<APART>(acc[c][T], y1[T], y1[TM], wa[WS * T]);
          });
        }
      }
    __syncthreads();
  }
  if constexpr (SPLIT) return;
  // ---- normalisation sums (fixed order) ----
  float* sqs = reinterpret_cast<float*>(Wk4);
  float* offs = sqs + T1;
  if constexpr (RST) {
#pragma unroll
    for (int r = 0; r < RR; ++r) {
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) rsum[r] += __shfl_xor(rsum[r], o);
      if ((tid & 63) == 0) rsq[r][tid >> 6] = rsum[r];
    }
  } else {
#pragma unroll
    for (int c = 0; c < TPT1; ++c) {
      const int task = tid + c * NT;
      if (task < T1) {
        sqs[task] = sqp[c];
        offs[task] = offp[c];
      }
    }
  }
  __syncthreads();
  for (int f = tid; f < F; f += NT) {
    double s0 = 0.0, s1 = 0.0;
    if constexpr (RST) {
      const int row = min((tile * F + f) / a.ns - rr0, nrow - 1);
      for (int w = 0; w < NT / 64; ++w) s0 += rsq[row][w];
    } else {
      for (int u = 0; u < B; ++u) {
        s0 += sqs[f * B + u];
        s1 += offs[f * B + u];
      }
    }
    sq[f] = (float)s0;
    off[f] = (float)s1;
  }
  if (tid == 0) pscal = ring_pscal(a, ip);
  if constexpr (PFA) ring_twiddles<N, A, NT>(tw, a.tw2g, tid);   // the spectra are no longer read
  // ---- inverse transform of every pair, normalisation, output ----
  unsigned long long bestkey = 0ull;
  ring_inverse<N, A, F, NT, RP, TPTL, PFA>(acc, buf, tw, a.tw2g, tid, [&](int f, int m, float2 y) {
    const int P = tile * F + f;
    if (P < npairs) RingEmit(a, N, sq[f], off[f], pscal)(a, pi, npairs, P, m, y, bestkey);
  });
  if (a.best) ring_best<NT>(a.best + pi, bestkey, red, tid);
}

// Finishes a search whose shells were split over work-groups: the work-group of a pair (particle slot x
// npairs + P) runs the products, sums, inverse transform, normalisation and output of k_corr_ring on the
// transforms left in sp, in the same order of operations (row A's bins, the mirror of row 0, have
// sums of their own there and here).  RST: the reference's norm is summed from its rows, as there.
// Bound: the latency of the loads, so a thread owns MB bins and keeps UB shells of each in flight, and UK
// shells of the norm's operands (100 pairs, 9 shifts at n 600: 177 us with the norm's loads one by one,
// 106).  160 pairs x 47 shells at n 240: 56 us per call; 152 us unsplit through the kernels before.
template <int N, int A, bool RST, int NT>
__global__ void __launch_bounds__(NT) k_ring_finish(CorrArgs a, RingSplit sp, int npairs) {
  using R = RingGeom<N, A>;
  constexpr int B = R::B, S = R::S, A1 = A + 1, ZL = A1 * B, MB = (ZL + NT - 1) / NT, UB = 16 / MB;
  constexpr bool PFA = ring_pfa<N, A, RST>(), APART = ring_apart(N);
  static_assert(A <= NT && B <= NT && NT % 64 == 0, "one task per thread");
  extern __shared__ __align__(16) float2 smem[];
  float2* buf = smem;                        // [S]
  float2* tw = buf + S;
  float2* Z = tw + R::TW;                    // [ZL]
  __shared__ float sqs[B], offs[B], norm[3]; // norm: sum |q|^2, Euclid offset, particle scale
  __shared__ double rsq[NT / 64];
  __shared__ unsigned long long red[NT / 64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int pair = blockIdx.x, pi = pair / npairs, P = pair - pi * npairs;
  const int ip = a.plist[pi], nk = a.nk, kc = a.kcorr, kloop = kc > a.knorm ? kc : a.knorm;
  ring_twiddles<N, A, NT>(tw, a.tw2g, tid);
  if constexpr (RST) {
    constexpr int JP = (N + NT - 1) / NT;
    const int ir = P / a.ns, iref = a.rlist ? a.rlist[ir] : ir;
    const float2* ref = (a.iseven[ip] ? a.refs_even : a.refs_odd) + (size_t)iref * nk * N;
    const float* ctf = a.ctf ? a.ctf + (size_t)ip * nk * N : nullptr;
    constexpr int UK = 16 / JP;
    double s = 0.0;
    for (int k0 = 0; k0 < kloop; k0 += UK) {
      float2 r[UK][JP];
      float cv[UK][JP];
#pragma unroll
      for (int v = 0; v < UK; ++v)
#pragma unroll
        for (int u = 0; u < JP; ++u) {
          const int e = min(k0 + v, kloop - 1) * N + min(tid + u * NT, N - 1);
          r[v][u] = ref[e];
          cv[v][u] = ctf ? ctf[e] : 1.0f;
        }
#pragma unroll
      for (int v = 0; v < UK; ++v)
#pragma unroll
        for (int u = 0; u < JP; ++u)
          if (k0 + v < kloop && (N % NT == 0 || tid + u * NT < N)) {
            const float2 q = make_float2(r[v][u].x * cv[v][u], r[v][u].y * cv[v][u]);
            s += (double)fmaf(q.y, q.y, q.x * q.x);
          }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) rsq[tid >> 6] = s;
  } else if (tid < B) {
    const float* e = sp.es + (size_t)pair * kloop * B + tid;
    constexpr int UK = 16;
    float s = 0.f, o = 0.f;
    for (int k0 = 0; k0 < kloop; k0 += UK) {
      float e2[UK], wk[UK];
#pragma unroll
      for (int v = 0; v < UK; ++v) {
        const int k = min(k0 + v, kloop - 1);
        e2[v] = e[k * B];
        wk[v] = a.mode == 1 ? a.shellw[(size_t)ip * nk + min(k, kc - 1)] : 0.f;
      }
#pragma unroll
      for (int v = 0; v < UK; ++v) {
        if (k0 + v < a.knorm) s += e2[v];
        if (k0 + v < kc) o = fmaf(wk[v], e2[v], o);
      }
    }
    sqs[tid] = s;
    offs[tid] = o;
  }
  if (tid == NT - 1) norm[2] = ring_pscal(a, ip);
  {
    const float2* z = sp.zrow + (size_t)pair * kc * ZL;
    const float2* memo = a.memo + (size_t)ip * nk * (N + 1);
    int iz[MB], in[MB], im[MB];
    float2 acc[MB], tm[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) {
      const int i = min(tid + b * NT, ZL - 1), T = i / A1, row = i - T * A1;
      iz[b] = i;
      in[b] = (PFA ? (B - T) % B : B - 1 - T) * A1 + A - row;
      im[b] = row == A ? (PFA ? N : A * (T + 1)) : PFA ? R::pfa_bin(row, T) : row + A * T;
      acc[b] = make_float2(0.f, 0.f);
      tm[b] = a.tw2g[im[b]];
    }
    for (int k0 = 0; k0 < kc; k0 += UB) {
      float2 v[UB][MB], vn[UB][MB], w[UB][MB];
#pragma unroll
      for (int u = 0; u < UB; ++u)
#pragma unroll
        for (int b = 0; b < MB; ++b) {
          const int k = min(k0 + u, kc - 1);
          v[u][b] = z[k * ZL + iz[b]];
          vn[u][b] = z[k * ZL + in[b]];
          w[u][b] = memo[k * (N + 1) + im[b]];
        }
#pragma unroll
      for (int u = 0; u < UB; ++u)
        if (k0 + u < kc) {
          const float wk = a.mode == 1 ? a.shellw[(size_t)ip * nk + k0 + u] : 1.0f;
#pragma unroll
          for (int b = 0; b < MB; ++b) acc_w12<APART>(acc[b], v[u][b], vn[u][b], spec_w12(w[u][b], wk, tm[b]));
        }
    }
#pragma unroll
    for (int b = 0; b < MB; ++b)
      if (tid + b * NT < ZL) Z[tid + b * NT] = acc[b];
  }
  __syncthreads();
  if (tid == 0) {
    double s0 = 0.0, s1 = 0.0;
    if constexpr (RST) {
      for (int w = 0; w < NT / 64; ++w) s0 += rsq[w];
    } else {
      for (int u = 0; u < B; ++u) {
        s0 += sqs[u];
        s1 += offs[u];
      }
    }
    norm[0] = (float)s0;
    norm[1] = (float)s1;
  }
  for (int i = tid; i < N; i += NT) {
    const int T = i / A, row = i - T * A, TM = PFA ? (B - T) % B : B - 1 - T;
    const int m = PFA ? R::pfa_bin(row, T) : row + A * T;
    float2 X = Z[T * A1 + row], Xn = Z[TM * A1 + (PFA && row == 0 && T != 0 ? 0 : A - row)];
    if (m == 0) {
      X.y = 0.f;
      Xn.y = 0.f;
    }
    buf[(m / B) * R::SB + m % B] = unsplit_bin_conj(X, Xn, cconj(a.tw2g[m]));
  }
  __syncthreads();
  if (tid < B) {
    float2* p = buf + tid;
    float2 v[A];
    static_for<0, A>([&](auto t) { v[decltype(t)::value] = p[decltype(t)::value * R::SB]; });
    RDft<A>::run(v);
    static_for<0, A>([&](auto t) { p[decltype(t)::value * R::SB] = v[decltype(t)::value]; });
  }
  __syncthreads();
  unsigned long long bestkey = 0ull;
  if (tid < A) {
    float2 y[B];
    ring_last_row<N, A, false>(buf, tw, tid, y);
    const RingEmit e(a, N, norm[0], norm[1], norm[2]);
    static_for<0, B>([&](auto t) {
      e(a, pi, npairs, P, tid + A * decltype(t)::value, y[decltype(t)::value], bestkey);
    });
  }
  if (a.best) ring_best<NT>(a.best + pi, bestkey, red, tid);
}

// Ring spectra (memoize_ffts :848-877): dst[i][kk][m] = rfft_2n(Re p + Im p | Re p - Im p)[m] of ring
// rows src[list ? list[i] : i][kk], F rings per work-group, the same two-pass transform.
// Bound: 16 bytes of HBM per ring element.
template <int N, int A, int F, int NT>
__global__ void __launch_bounds__(NT) k_ring_spec(const float2* __restrict__ src, const int* __restrict__ list,
                                                  int count, int nk, const float2* __restrict__ tw2g,
                                                  float2* __restrict__ dst) {
  using R = RingGeom<N, A>;
  constexpr int B = R::B, H = R::H, S = R::S, G = R::G;
  extern __shared__ __align__(16) float2 smem[];
  float2* buf = smem;                        // [F][S]
  float2* tw = buf + F * S;
  const int tid = threadIdx.x;
  const long long nitems = (long long)count * nk, item0 = (long long)blockIdx.x * F;
  ring_twiddles<N, A, NT>(tw, tw2g, tid);
  for (int task = tid; task < F * B; task += NT) {
    const int f = task / B, t3 = task % B;
    const long long item = item0 + f;
    if (item >= nitems) continue;
    const int i = (int)(item / nk), kk = (int)(item % nk);
    const float2* p = src + ((size_t)(list ? list[i] : i) * nk + kk) * N + 2 * t3;
    float2 E[H], O[H];
    static_for<0, H>([&](auto tt) {
      constexpr int T = decltype(tt)::value;
      const float4 q = *reinterpret_cast<const float4*>(p + 2 * T * B);
      E[T] = make_float2(q.x, q.z);
      O[T] = make_float2(q.y, q.w);
    });
    float2* o = buf + f * S + t3;
    dft_even_odd<A>(E, O, [&](auto k, float2 v) { o[decltype(k)::value * R::SB] = v; });
  }
  __syncthreads();
  for (int task = tid; task < F * G; task += NT) {
    const int f = task / G, g = task % G;
    const long long item = item0 + f;
    if (item >= nitems) continue;
    float2 y1[B], y2[B];
    ring_last_row<N, A, false>(buf + f * S, tw, g, y1);
    ring_last_row<N, A, false>(buf + f * S, tw, A - g, y2);
    float2* o = dst + (size_t)item * (N + 1);
    // V[m] = (Z[m] + conj Z[N-m]) - i w_m (Z[m] - conj Z[N-m]) of the halved transform
    auto put = [&](int m, float2 Z, float2 Zn) {
      const float2 sum = make_float2(Z.x + Zn.x, Z.y - Zn.y), dif = make_float2(Z.x - Zn.x, Z.y + Zn.y);
      const float2 wd = cmul(tw2g[m], dif);
      o[m] = make_float2(sum.x + wd.y, sum.y - wd.x);
    };
    static_for<0, B>([&](auto tt) {
      constexpr int T = decltype(tt)::value;
      put(g + A * T, y1[T], y2[B - 1 - T]);
      if (g != H && (g != 0 || T == B - 1)) put(A - g + A * T, y2[T], y1[B - 1 - T]);
    });
  }
}

}  // namespace pfk
