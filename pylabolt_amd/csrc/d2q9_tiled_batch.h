// Batched tiled sweep: the tiles of many lattices in one launch of several
// steps (d2q9_tiled.h).  A workgroup takes one item -- a tile of one lattice
// -- and dispatches on that lattice's collision model and forcing.  Items are
// in lattice and row order and each XCD takes a contiguous run of them, so
// that neighbouring tiles meet in one L2.
#pragma once
#include "d2q9_tiled.h"

namespace d2q9 {
namespace tiled {

struct BatchLaunch {
  const d2q9_tiled_entry* entries;
  const d2q9_tiled_item* items;
  int n_items, rows, width, tile_c, K, collide_first, parity, write_mom, planes;
  hipStream_t stream;
};

template <int S, int W>
__global__ __launch_bounds__(MAX_CELLS, S == D2Q9_STORE_F64 ? 4 : 8) void k_tiled_batch(
    const d2q9_tiled_entry* __restrict__ entries, const d2q9_tiled_item* __restrict__ items,
    int n_items, int K, int rows, int tile_c, int collide_first, int parity, int write_mom) {
  using C = Codec<S>;
  extern __shared__ __align__(16) char smem[];
  const d2q9_tiled_item it = items[xcd_remap((int)blockIdx.x, n_items)];
  const d2q9_tiled_entry& E = entries[it.lattice];
  const d2q9_lattice L = E.L;
  const d2q9_tiled_desc D = E.D;
  auto fs = static_cast<const typename C::raw*>(E.f[parity]);
  auto fd = static_cast<typename C::raw*>(E.f[1 - parity]);
  auto ms = static_cast<const typename C::T*>(E.mom[parity]);
  auto md = static_cast<typename C::T*>(E.mom[1 - parity]);
#define D2Q9_TILED_ITEM(KEY, M, F)                                                         \
  case KEY:                                                                                \
    run_tile<S, M, F, W, false>(L, D, smem, 1 + it.ti * (rows - 2 * K), 1 + it.tj * tile_c,       \
                         tile_c, K, rows, collide_first, fs, fd, ms, md, write_mom,        \
                         nullptr, 0);                                                      \
    break;
  switch (L.collision * 3 + L.forcing) {
    D2Q9_TILED_ITEM(0, D2Q9_BGK, D2Q9_FORCING_NONE)
    D2Q9_TILED_ITEM(1, D2Q9_BGK, D2Q9_GUO_LINEAR)
    D2Q9_TILED_ITEM(2, D2Q9_BGK, D2Q9_GUO_SECOND_ORDER)
    D2Q9_TILED_ITEM(3, D2Q9_MRT, D2Q9_FORCING_NONE)
    D2Q9_TILED_ITEM(4, D2Q9_MRT, D2Q9_GUO_LINEAR)
    D2Q9_TILED_ITEM(5, D2Q9_MRT, D2Q9_GUO_SECOND_ORDER)
  }
#undef D2Q9_TILED_ITEM
}

template <int S, int W>
hipError_t launch_batch_one(const BatchLaunch& A) {
  auto kern = k_tiled_batch<S, W>;
  static PerDevice limit;
  if (const hipError_t e = allow_lds(limit, kern)) return e;
  const int area = A.rows * W;
  const size_t lds = (size_t)((area * A.planes + 3) & ~3) * sizeof(typename Codec<S>::T) +
                     MAX_ELEMS * sizeof(d2q9_bc_elem);
  hipLaunchKernelGGL(kern, dim3((unsigned)A.n_items), dim3((unsigned)((area + 63) / 64 * 64)),
                     lds, A.stream, A.entries, A.items, A.n_items, A.K, A.rows, A.tile_c,
                     A.collide_first, A.parity, A.write_mom);
  return hipGetLastError();
}

template <int S>
hipError_t launch_batch(const BatchLaunch& A);

#define D2Q9_TILED_BATCH_DEFINE(SV)                      \
  template <>                                            \
  hipError_t launch_batch<SV>(const BatchLaunch& A) {    \
    switch (A.width) {                                   \
      case 16: return launch_batch_one<SV, 16>(A);       \
      case 32: return launch_batch_one<SV, 32>(A);       \
      case 64: return launch_batch_one<SV, 64>(A);       \
    }                                                    \
    return hipErrorInvalidValue;                         \
  }
template <>
hipError_t launch_batch<D2Q9_STORE_F64>(const BatchLaunch& A);
template <>
hipError_t launch_batch<D2Q9_STORE_F32>(const BatchLaunch& A);

}  // namespace tiled
}  // namespace d2q9
