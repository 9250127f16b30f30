// ring_ops.hpp - the kernels with a compile-time ring length, by ring length.
//
// rings.hip instantiates them (in several translation units, each holding a group of lengths);
// ring_ops(n) gives the launchers of ring length n, or null where n has none and the runtime-size
// kernels run.
#pragma once
#include "corr_ring.hpp"
#include "zifft.hpp"

struct RingOps {
  int n;
  int tile, tile_rst;          // pairs per work-group of the plain search (per-pair / staged references)
  int min_shifts;              // fewest shifts with which the staged-reference variant runs
  int pfa_a;                   // its radix A where it takes the Good-Thomas form (shift table in that order), else 0
  // a split search's memory per pair: values per shell of its transform (per-pair / staged variant), and
  // the per-pair variant's sums |q|^2 per shell
  int zrow, zrow_rst, slots;
  // plain search: grid (particle slots x tiles, shell chunks)
  void (*corr)(bool rst, dim3 grid, hipStream_t s, const pfk::CorrArgs& a, const pfk::RingSplit& sp);
  // finishes a search split over shell chunks: total pairs, npairs per particle slot
  void (*finish)(bool rst, int total, int npairs, hipStream_t s, const pfk::CorrArgs& a, const pfk::RingSplit& sp);
  // shift-search items (a.np items, a.shtab their phases), or null: the runtime-size kernel takes them
  void (*items)(hipStream_t s, const pfk::CorrArgs& a);
  // inverse stage of the precision form: cnt particles against nr operand rows (a.Z16: FP16 spectra)
  void (*zifft)(int cnt, int nr, hipStream_t s, const pfk::ZifftArgs& a);
  // ring spectra of count rows of nk rings (list: their rows in src, null: 0 ..), dst [count][nk][n+1]
  void (*spec)(const float2* src, const int* list, int count, int nk, const float2* tw2g, float2* dst, hipStream_t s);
};

const RingOps* ring_ops(int n);
