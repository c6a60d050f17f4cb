// Strip sweep: up to STRIP_STEPS fused time steps per pass over the plain
// interior of a large lattice.
//
// A workgroup sweeps a chunk -- a strip of 64 - 2 STRIP_STEPS output columns
// by a run of rows -- row by row, one wave per time step: in every iteration
// wave s - 1 computes one row of step s, two rows behind the wave before it,
// so that the three rows it pulls from are there.  Steps hand rows on through
// LDS rings that hold what is still to be pulled: three rows of the
// directions pulled from the same or the next row, four of those pulled from
// the row before.  The first wave pulls from the lattice (a row ahead, in
// registers), the last stores to the other one.
//
// Compared with a tile held in LDS, cells are computed twice only at the sides
// of a strip (64 lanes for 56 columns) and at the ends of a chunk, and loads,
// arithmetic and stores of different rows overlap.  Per K steps the lattice is
// read 64 / 56 times and written once.
//
// Chunks hold plain cells only, but for a straight zero-gradient or
// bounce-back wall in the lattice's first or last column; every other cell
// is in a tile of the tiled sweep, run by the same launch's first workgroups:
// both read the source lattice alone and write different cells.  The
// arithmetic per cell is the single step's; 16-bit storage rounds every step
// (or, when asked, the last of a launch only).
#pragma once
#include "d2q9_tiled.h"

namespace d2q9 {
namespace strip {

constexpr int STEPS = 4;                     // most steps of a launch
constexpr int LANES = 64;
constexpr int COLS = LANES - 2 * STEPS;      // output columns of a strip
constexpr int THREADS = 64 * STEPS;
constexpr int TILE_W = 16;                   // region width of the tiles
constexpr int TILE = TILE_W - 2 * STEPS;     // their output rows and columns
constexpr int PITCH = LANES + 2;
// dir-rows of a ring: 3 rows of directions 0,2,4, 3 of 3,6,7, 4 of 1,5,8
constexpr int RING_B = 9, RING_C = 18, RING = 30;

// Place of direction k in its group of three, and the group's first dir-row.
__device__ constexpr int SLOT[9] = {0, 0, 1, 0, 2, 1, 1, 2, 2};
__device__ constexpr int BASE[9] = {0, RING_C, 0, RING_B, 0, RING_C, RING_B, RING_B, RING_C};

// One stored element as an integer (non-temporal stores take no half types).
template <size_t BYTES> struct Word;
template <> struct Word<2> { using type = unsigned short; };
template <> struct Word<4> { using type = uint32_t; };
template <> struct Word<8> { using type = uint64_t; };

template <int S>
__host__ __device__ constexpr size_t ring_bytes(int steps) {
  return (size_t)(steps - 1) * RING * PITCH * sizeof(typename Codec<S>::T);
}

template <int S, int MODEL, int FORCING>
__device__ __forceinline__ void run_strip(
    const d2q9_lattice& L, char* __restrict__ smem, const d2q9_strip_chunk ch, int K,
    const typename Codec<S>::raw* __restrict__ fsrc, typename Codec<S>::raw* __restrict__ fdst,
    typename Codec<S>::T* __restrict__ mdst, int write_mom, int round_last) {
  using C = Codec<S>;
  using T = typename C::T;
  using R = typename C::raw;
  constexpr int B = 64 * C::CPL;
  const int lane = (int)threadIdx.x & 63;
  const int st = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) + 1;  // this wave's step
  const Consts<T> Kc = load_consts<T>(L);
  const int lo = ch.walls & 3, hi = (ch.walls >> 2) & 3;
  // the lane's column, its neighbours' places in a row
  auto column = [&](int j) {
    if (L.y_periodic) {
      if (j < 1) j += L.ny;
      else if (j > L.ny) j -= L.ny;
    }
    return min(max(j, 0), L.ny + 1);
  };
  auto place = [&](int j) {
    const unsigned jj = (unsigned)(j + B - 1);
    return ((jj / B) * (9u * B) + jj % B) * (unsigned)sizeof(R);
  };
  const int ju = ch.j_first - K + lane, j = column(ju);
  const bool out = lane >= K && lane < K + ch.cols;
  const bool wall_lo = lo != 0 && ju == 1, wall_hi = hi != 0 && ju == L.ny;
  const bool zg = (wall_lo && lo == 1) || (wall_hi && hi == 1);
  const bool bb = (wall_lo && lo == 2) || (wall_hi && hi == 2);
  const unsigned p0 = place(j);
  // zero-gradient: the unknown directions are what the inner neighbour pulls,
  // from the wall cell's own column
  const unsigned pm = place(zg && wall_lo ? j : column(ju - 1));
  const unsigned pp = place(zg && wall_hi ? j : column(ju + 1));
  auto wrap = [&](int i) { return L.x_periodic ? (i < 1 ? i + L.nx : i > L.nx ? i - L.nx : i) : i; };
  auto row_at = [&](int i) {
    return (uint64_t)((unsigned)wrap(i) * (unsigned)L.nbj) * (9u * B * (unsigned)sizeof(R));
  };
  auto load = [&](int i, int k, unsigned at) {
    return *reinterpret_cast<const R*>(reinterpret_cast<const char*>(fsrc + k * B) + row_at(i) +
                                       at);
  };
  // step `st` computes rows i_first - (K - st) .. i_first + rows - 1 + (K - st)
  const int begin = 3 * (st - 1), count = ch.rows + 2 * (K - st);
  const int total = ch.rows + 3 * (K - 1);
  int i = ch.i_first - (K - st);
  T* const to = reinterpret_cast<T*>(smem) + (st - 1) * RING * PITCH + 1 + lane;
  const T* const from = to - RING * PITCH;
  // the first step's row, a row ahead; the wall's own opposite populations
  R raw[9], back[3];
  auto fetch = [&](int row) {
#pragma unroll
    for (int k = 0; k < 9; ++k)
      raw[k] = load(row - CX[k], k, CY[k] == 0 ? p0 : CY[k] > 0 ? pm : pp);
    if (lo == 2 || hi == 2) {
      if (wall_lo) {
        back[0] = load(row, 4, p0);
        back[1] = load(row, 7, p0);
        back[2] = load(row, 8, p0);
      }
      if (wall_hi) {
        back[0] = load(row, 2, p0);
        back[1] = load(row, 5, p0);
        back[2] = load(row, 6, p0);
      }
    }
  };
  if (st == 1) fetch(i);
  int a3 = 0, a4 = 0;   // ring slots this row is written to (row number mod 3 and 4)
#pragma unroll 1
  for (int t = 0; t < total; ++t) {
    if (st <= K && t >= begin && t < begin + count) {
      T g[9];
      if (st == 1) {
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = C::dec(raw[k], k, Kc);
        if (lo == 2 || hi == 2) {
          if (bb) {
            // directions 2, 5, 6 from 4, 7, 8 (low wall), 4, 7, 8 from 2, 5, 6
            if (wall_lo) {
              g[2] = C::dec(back[0], 4, Kc);
              g[5] = C::dec(back[1], 7, Kc);
              g[6] = C::dec(back[2], 8, Kc);
            } else {
              g[4] = C::dec(back[0], 2, Kc);
              g[7] = C::dec(back[1], 5, Kc);
              g[8] = C::dec(back[2], 6, Kc);
            }
          }
        }
        if (t + 1 < begin + count) fetch(i + 1);
      } else {
        // rows i (number n + 1 of the step before), i + 1 (n + 2), i - 1 (n)
        const int same = (a3 + 1 >= 3 ? a3 - 2 : a3 + 1) * 3;
        const int next = RING_B + (a3 + 2 >= 3 ? a3 - 1 : a3 + 2) * 3;
        const int prev = RING_C + a4 * 3;
        const T* const r0 = from + same * PITCH;
        const T* const rb = from + next * PITCH;
        const T* const rc = from + prev * PITCH;
#pragma unroll
        for (int k = 0; k < 9; ++k)
          g[k] = (CX[k] == 0 ? r0 : CX[k] < 0 ? rb : rc)[SLOT[k] * PITCH - CY[k]];
        if (lo | hi) {
          if (zg) {
#pragma unroll
            for (int k = 1; k < 9; ++k)
              if (CY[k] == 1 ? wall_lo : CY[k] == -1 ? wall_hi : false)
                g[k] = (CX[k] == 0 ? r0 : CX[k] < 0 ? rb : rc)[SLOT[k] * PITCH];
          } else if (bb) {
            const T* const own_b = from + (RING_B + same) * PITCH;
            const T* const own_c = from + (RING_C + (a4 + 1 & 3) * 3) * PITCH;
#pragma unroll
            for (int k = 1; k < 9; ++k)
              if (CY[k] == 1 ? wall_lo : CY[k] == -1 ? wall_hi : false)
                g[k] = (CX[INV[k]] == 0 ? r0 : CX[INV[k]] < 0 ? own_b
                                                              : own_c)[SLOT[INV[k]] * PITCH];
          }
        }
      }
      const int iw = wrap(i);
      const int cell = L.origin + iw * L.pitch + j;
      T ffx = (T)0, ffy = (T)0;
      if (FORCING != D2Q9_FORCING_NONE && L.force_source == D2Q9_FSRC_FIELD) {
        const T* ff = static_cast<const T*>(L.force_field);
        ffx = ff[cell];
        ffy = ff[L.plane + cell];
      }
      T drho, rho, ux, uy, fx, fy, px, py;
      moments<T, FORCING, C::dev>(g, L, Kc, ffx, ffy, drho, rho, ux, uy, fx, fy, px, py);
      collide<T, MODEL, FORCING, C::dev>(g, Kc, drho, rho, ux, uy, fx, fy, px, py);
      const uint32_t key = sizeof(R) == 2 ? cell_key((uint32_t)cell) : 0u;
      if (st < K) {
        T* const w0 = to + a3 * 3 * PITCH;
        T* const wc = to + (RING_C + a4 * 3) * PITCH;
        if (sizeof(R) == 2 && !round_last) {
#pragma unroll
          for (int k = 0; k < 9; ++k) g[k] = tiled::through_storage<S>(g[k], k, key, Kc);
        }
#pragma unroll
        for (int k = 0; k < 9; ++k)
          (CX[k] == 0 ? w0 : CX[k] < 0 ? w0 + RING_B * PITCH : wc)[SLOT[k] * PITCH] = g[k];
      } else if (out) {
        char* const d = reinterpret_cast<char*>(fdst) + row_at(i);
#pragma unroll
        for (int k = 0; k < 9; ++k) {
          using W = typename Word<sizeof(R)>::type;
          const R v = C::encs(g[k], k, key, Kc);
          W w;
          __builtin_memcpy(&w, &v, sizeof(W));
          store_nt(w, reinterpret_cast<W*>(d + (size_t)(k * B) * sizeof(R) + p0));
        }
        if (write_mom) {
          mdst[cell] = rho;
          mdst[L.plane + cell] = ux;
          mdst[2 * L.plane + cell] = uy;
        }
      }
      ++i;
      a3 = a3 == 2 ? 0 : a3 + 1;
      a4 = (a4 + 1) & 3;
    }
    __syncthreads();
  }
}

template <int S, int FORCING>
constexpr int waves_per_simd() {
  return S == D2Q9_STORE_F64 ? 4 : 6;
}

// Workgroups [0, n_tiles): tiles of TILE x TILE cells; the others: chunks.
template <int S, int MODEL, int FORCING>
__global__ __launch_bounds__(THREADS, (waves_per_simd<S, FORCING>())) void k_strip(
    const d2q9_lattice L, const d2q9_tiled_desc D, const d2q9_strip_desc P, int K,
    const typename Codec<S>::raw* __restrict__ fsrc, typename Codec<S>::raw* __restrict__ fdst,
    const typename Codec<S>::T* __restrict__ msrc, typename Codec<S>::T* __restrict__ mdst,
    int write_mom, int round_last) {
  extern __shared__ __align__(16) char smem[];
  const int b = (int)blockIdx.x;
  if (b < P.n_tiles) {
    const d2q9_strip_tile it = P.tiles[b];
    tiled::run_tile<S, MODEL, FORCING, TILE_W>(L, D, smem, it.i_first, it.j_first, TILE, K,
                                               TILE + 2 * K, 0, fsrc, fdst, msrc, mdst,
                                               write_mom, nullptr, 0);
    return;
  }
  run_strip<S, MODEL, FORCING>(L, smem, P.chunks[xcd_remap(b - P.n_tiles, P.n_chunks)], K, fsrc,
                               fdst, mdst, write_mom, round_last);
}

struct Launch {
  int K, write_mom, round_last;
  const void* fsrc;
  void* fdst;
  const void* msrc;
  void* mdst;
  hipStream_t stream;
};

template <int S, int MODEL, int FORCING>
hipError_t launch_one(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                      const Launch& A) {
  using C = Codec<S>;
  auto kern = k_strip<S, MODEL, FORCING>;
  static const hipError_t limit =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                          hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
  if (limit != hipSuccess) return limit;
  size_t lds = ring_bytes<S>(A.K);
  if (P->n_tiles > 0) {
    const size_t t = tiled::lds_bytes(*D, (TILE + 2 * A.K) * TILE_W, sizeof(typename C::T));
    if (t > lds) lds = t;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(P->n_tiles + P->n_chunks)), dim3(THREADS), lds,
                     A.stream, *L, *D, *P, A.K, static_cast<const typename C::raw*>(A.fsrc),
                     static_cast<typename C::raw*>(A.fdst),
                     static_cast<const typename C::T*>(A.msrc),
                     static_cast<typename C::T*>(A.mdst), A.write_mom, A.round_last);
  return hipGetLastError();
}

template <int S>
hipError_t launch(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                  const Launch& A);

template <int S>
hipError_t launch_model(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                        const Launch& A) {
  switch (L->collision * 3 + L->forcing) {
    case 0: return launch_one<S, D2Q9_BGK, D2Q9_FORCING_NONE>(L, D, P, A);
    case 1: return launch_one<S, D2Q9_BGK, D2Q9_GUO_LINEAR>(L, D, P, A);
    case 2: return launch_one<S, D2Q9_BGK, D2Q9_GUO_SECOND_ORDER>(L, D, P, A);
    case 3: return launch_one<S, D2Q9_MRT, D2Q9_FORCING_NONE>(L, D, P, A);
    case 4: return launch_one<S, D2Q9_MRT, D2Q9_GUO_LINEAR>(L, D, P, A);
    case 5: return launch_one<S, D2Q9_MRT, D2Q9_GUO_SECOND_ORDER>(L, D, P, A);
  }
  return hipErrorInvalidValue;
}

#define D2Q9_STRIP_DECLARE(SV)                                                 \
  template <>                                                                  \
  hipError_t launch<SV>(const d2q9_lattice* L, const d2q9_tiled_desc* D,       \
                        const d2q9_strip_desc* P, const Launch& A);
D2Q9_STRIP_DECLARE(D2Q9_STORE_F64)
D2Q9_STRIP_DECLARE(D2Q9_STORE_F32)
D2Q9_STRIP_DECLARE(D2Q9_STORE_F16DEV)
D2Q9_STRIP_DECLARE(D2Q9_STORE_BF16DEV)
#undef D2Q9_STRIP_DECLARE

}  // namespace strip
}  // namespace d2q9
