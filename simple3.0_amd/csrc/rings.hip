// rings.hip - instantiations of the kernels with a compile-time ring length (ring_ops.hpp).
//
// Compiled once per PFTCC_RING_GROUP (0 .. PFTCC_RING_GROUPS - 1), so that the groups build in
// parallel.  The lengths are the FFT-friendly ones of the reference's table that a mask radius can
// lead to (simple_magic_boxes.f90:14-19) up to 600, and small ones.
#include "corr_items.hpp"
#include "ring_ops.hpp"

using namespace pfk;

#ifndef PFTCC_RING_GROUP
#define PFTCC_RING_GROUP 0
#endif
#define PFTCC_RING_SIZES(X) \
  X(0, 16) X(1, 24) X(2, 32) X(3, 36) X(4, 40) X(5, 48) X(6, 52) X(7, 56) X(0, 64) X(1, 66) X(2, 70) X(3, 72)     \
  X(4, 80) X(5, 84) X(6, 88) X(7, 100) X(0, 104) X(1, 108) X(2, 112) X(3, 120) X(4, 128) X(5, 130) X(6, 132)      \
  X(7, 140) X(0, 144) X(1, 150) X(2, 160) X(3, 162) X(4, 168) X(5, 176) X(6, 180) X(7, 182) X(0, 192) X(1, 200)    \
  X(2, 208) X(3, 216) X(4, 220) X(5, 224) X(6, 240) X(7, 256) X(0, 264) X(1, 288) X(2, 300) X(3, 308) X(4, 320)    \
  X(5, 324) X(6, 336) X(7, 338) X(0, 352) X(1, 364) X(2, 384) X(3, 400) X(4, 420) X(5, 432) X(6, 448) X(7, 450)    \
  X(0, 462) X(1, 480) X(2, 486) X(3, 500) X(4, 504) X(5, 512) X(6, 520) X(7, 528) X(0, 546) X(1, 560) X(2, 576)    \
  X(3, 588) X(4, 600)

namespace {

// Radix and tile of the plain search at one ring length (N = A B).
struct RingCfg {
  int A;      // radix of pass 1
  int F;      // pairs per work-group
  int W;      // wavefronts per SIMD the registers must allow
  int RP;     // rows per last-pass task
  bool PRF = false;   // per-pair: reference values loaded a shell ahead
};
struct RingRow {
  int n;
  RingCfg pair, staged;        // per-pair and staged-reference variants
  int za;                      // radix A of the inverse stage
};
#include "ring_table.hpp"
constexpr RingRow kRingTable[] = {PFTCC_RING_TABLE};
constexpr RingRow ring_row_of(int n) {
  for (const RingRow& r : kRingTable)
    if (r.n == n) return r;
  return RingRow{-1, {}, {}, 0};
}

template <int N>
struct Ring {
  static constexpr int NT = 256;
  static constexpr RingCfg P = ring_row_of(N).pair, S = ring_row_of(N).staged;
  static void corr(bool rst, dim3 grid, hipStream_t s, const CorrArgs& a, const RingSplit& sp) {
    const size_t lds_r = ring_lds_bytes<N, S.A, S.F, NT, true>(ring_span(S.F, a.ns));
    constexpr size_t lds = ring_lds_bytes<N, P.A, P.F, NT, false>(0);
    if (rst && sp.nsplit > 1)
      hipLaunchKernelGGL((k_corr_ring<N, S.A, S.F, NT, 2, 1, true, false, true>), grid, dim3(NT), lds_r, s, a, sp);
    else if (rst)
      hipLaunchKernelGGL((k_corr_ring<N, S.A, S.F, NT, S.W, S.RP, true, false, false>), grid, dim3(NT), lds_r, s, a, sp);
    else if (sp.nsplit > 1)
      hipLaunchKernelGGL((k_corr_ring<N, P.A, P.F, NT, 2, 1, false, false, true>), grid, dim3(NT), lds, s, a, sp);
    else
      hipLaunchKernelGGL((k_corr_ring<N, P.A, P.F, NT, P.W, P.RP, false, P.PRF, false>), grid, dim3(NT), lds, s, a, sp);
  }
  template <int A>
  static constexpr int zrow() { return (A + 1) * (N / A); }
  template <int A, bool RST>
  static void finish_go(int total, int npairs, hipStream_t s, const CorrArgs& a, const RingSplit& sp) {
    using R = RingGeom<N, A>;
    hipLaunchKernelGGL((k_ring_finish<N, A, RST, NT>), dim3((unsigned)total), dim3(NT),
                       8 * (size_t)(R::S + R::TW + zrow<A>()), s, a, sp, npairs);
  }
  static void finish(bool rst, int total, int npairs, hipStream_t s, const CorrArgs& a, const RingSplit& sp) {
    if (rst) finish_go<S.A, true>(total, npairs, s, a, sp);
    else finish_go<P.A, false>(total, npairs, s, a, sp);
  }
  // shift-search items: shells per work-group pass (LDS for four work-groups per CU), and threads
  static constexpr int IF = N <= 400 ? 8 : 4, IT = N <= 64 ? 64 : 256;
  // the other lengths' callback keeps the runtime-size kernel's order of operations
  static constexpr bool has_items() { return ring_first(N); }
  static void items(hipStream_t s, const CorrArgs& a) {
    if constexpr (has_items())
      hipLaunchKernelGGL((k_corr_items<N, IF, IT>), dim3((unsigned)a.np), dim3(IT),
                         (corr_items_lds<N, IF>()), s, a);
  }
  // inverse stage: 8 pairs per two wavefronts
  static constexpr int ZA = ring_row_of(N).za, ZF = 8, ZT = 128;
  static void zifft(int cnt, int nr, hipStream_t s, const ZifftArgs& a) {
    const dim3 grid((unsigned)((size_t)((cnt + ZF - 1) / ZF) * nr));
    if (a.Z16)
      hipLaunchKernelGGL((k_ring_zifft<N, ZA, ZF, ZT, true>), grid, dim3(ZT), (ring_zifft_lds<N, ZA, ZF>()), s, a);
    else
      hipLaunchKernelGGL((k_ring_zifft<N, ZA, ZF, ZT, false>), grid, dim3(ZT), (ring_zifft_lds<N, ZA, ZF>()), s, a);
  }
  static constexpr int XF = 8;               // rings per work-group of the spectra
  static void spec(const float2* src, const int* list, int count, int nk, const float2* tw2g, float2* dst,
                   hipStream_t s) {
    using R = RingGeom<N, P.A>;
    hipLaunchKernelGGL((k_ring_spec<N, P.A, XF, 128>), dim3((unsigned)(((size_t)count * nk + XF - 1) / XF)), dim3(128),
                       8 * (size_t)(XF * R::S + R::TW), s, src, list, count, nk, tw2g, dst);
  }
  static constexpr RingOps ops{N, P.F, S.F, ring_min_shifts(N, S.F, S.RP), ring_pfa<N, S.A, true>() ? S.A : 0,
                               zrow<P.A>(), zrow<S.A>(), N / P.A, corr, finish,
                               has_items() ? items : nullptr, zifft, spec};
};

}  // namespace

#define RING_FN2(g) ring_ops_group##g
#define RING_FN(g) RING_FN2(g)

const RingOps* RING_FN(PFTCC_RING_GROUP)(int n) {
#define X(G, N)                         \
  if constexpr (G == PFTCC_RING_GROUP) { \
    if (n == N) return &Ring<(G == PFTCC_RING_GROUP ? N : 16)>::ops; \
  }
  PFTCC_RING_SIZES(X)
#undef X
  return nullptr;
}
