// Shared by the prefill grouped-GEMM kernels (hx_prefill*.hip): the M tile of a
// workgroup and the matrix-core vector types.
#pragma once
#include "hx_internal.h"

namespace hx {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int PM = HX_TILE_M;     // rows of an M tile

// the M tile of a workgroup (expert, first permuted row, rows): from the
// dispatch list, or for a shared-expert-only launch computed from T; false if
// the workgroup has no tile (past the end, or a tile the launch skips). TS is
// the launch's tile selection (HX_TILES_*), a template parameter so that each
// selection is a kernel of its own name in traces and counter runs.
// m: the rows of the expert's call (the reference's arm: m <= HX_QUANT_M
// quantised activations, else f16)
template <int TS>
HX_DEV bool get_tile(const ExpertArgs& a, int tile, int& e, int& p0, int& rows, int& m) {
  if (TS == HX_TILES_SHARED) {
    const int m0 = tile * PM;
    if (m0 >= a.T) return false;
    e = a.E;
    p0 = a.F + m0;
    rows = min(PM, a.T - m0);
    m = a.T;
    return true;
  }
  // the record's address needs no count (the grid is rounded up past the list's
  // last record). The compiler reads it behind the count's branch all the same;
  // held together with the count it changed nothing (512 tokens Q4_K_M 210.8 /
  // 210.7 us, 2048 Q8_0 434 / 433)
  const int4 rec = *(const int4*)(a.tiles + 4 * min(tile, a.max_tiles - 1));
  const int n = a.counts[1];
  m = rec.x;
  e = rec.y;
  p0 = rec.z;
  rows = rec.w;
  return tile < n && !(TS == HX_TILES_ROUTED && e == a.E);
}

}  // namespace hx
