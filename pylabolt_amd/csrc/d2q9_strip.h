// Strip sweep: up to STEPS fused time steps per pass over the plain interior
// of a large lattice.
//
// A workgroup sweeps a chunk -- a strip of columns by a run of rows -- row by
// row, one wave per time step: in every iteration wave s - 1 computes one row
// of step s, two rows behind the wave before it, so that the three rows it
// pulls from are there.  Steps hand rows on through LDS rings that hold what
// is still to be pulled: three rows of the directions pulled from the same or
// the next row, four of those pulled from the row before.  The first wave
// pulls from the lattice (a row or two ahead, in registers), the last stores
// to the other one.  A lane holds one cell, so a row is 64 cells wide, STEPS of them on
// either side for the neighbouring strips' sake only.  (Two cells a lane for the
// float forms halve the waves a CU holds: FP32 2999x1111 22 us per step against
// 18, 8192x2048 97 against 91.)
//
// Compared with a tile held in LDS, cells are computed twice only at the sides
// of a strip (64 for 56 columns) and at the ends of a chunk, and loads,
// arithmetic and stores of different rows overlap.  Per STEPS steps the lattice
// is read 1.15 times in FP64 and about 1.45 in FP32 and 16 bits, and written 1.0
// to 1.05 times (counters: FP64 8192x2048, FP32 2999x1111, BF16 4096x1024).
//
// What bounds it (same launches): FP64 without a force and FP32 HBM at 4.5 TB/s
// and vector issue in 0.6 of the cycles at once; BF16 vector issue (0.77).
// FP64 MRT + Guo, 4096x1024, is at neither limit, 2.6 TB/s and 0.51: 298
// vector instructions per cell and step with the 12 waves per CU that the
// rings leave room for.
//
// Chunks hold plain cells only, but for a straight zero-gradient or
// bounce-back wall in the lattice's first or last column; every other cell
// is in a tile of the tiled sweep, run by the same launch's first workgroups:
// both read the source lattice alone and write different cells.  The
// arithmetic per cell is the single step's; 16-bit storage rounds every step
// (when asked, the last of a launch only, or as the two-step sweep: chunks then
// hold cells of its deep tiles, rounded after every second step).
#pragma once
#include "d2q9_tiled.h"

namespace d2q9 {
namespace strip {

constexpr int STEPS = 4;                     // most steps of a launch
constexpr int THREADS = 64 * STEPS;
constexpr int COLS = 64 - 2 * STEPS;         // output columns of a strip
constexpr int TILE_W = 16;                   // region width of the tiles
constexpr int TILE = TILE_W - 2 * STEPS;     // their output rows and columns
static_assert(STEPS % 2 == 0, "launches take whole pairs of steps");
// Rows of a ring, three directions each: 3 of 0,2,4, 3 of 3,6,7, 4 of 1,5,8.
constexpr int RING_B = 9, RING_C = 18, RING = 30;

// Place of direction k in its group of three.
__device__ constexpr int SLOT[9] = {0, 0, 1, 0, 2, 1, 1, 2, 2};

constexpr int PITCH = 64 + 2;                // values of an LDS row
template <int S>
constexpr size_t ring_bytes(int steps) {
  return (size_t)(steps - 1) * RING * PITCH * sizeof(typename Codec<S>::T);
}

// Barrier of the workgroup that waves may reach at different places of the
// code, with the LDS traffic before it done: s_barrier counts arrivals.
__device__ __forceinline__ void workgroup_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// A row's values: the loaded ones themselves, or room for them decoded.
template <typename R, typename T>
__device__ __forceinline__ T (&values_of(R (&raw)[9], T (&apart)[9]))[9] {
  if constexpr (std::is_same<R, T>::value)
    return raw;
  else
    return apart;
}

template <int S, int MODEL, int FORCING, bool PAIRS>
__device__ __forceinline__ void run_strip(
    const d2q9_lattice& L, char* __restrict__ smem, const d2q9_strip_chunk ch, int K,
    const typename Codec<S>::raw* __restrict__ fsrc, typename Codec<S>::raw* __restrict__ fdst,
    typename Codec<S>::T* __restrict__ mdst, int write_mom, bool round_last) {
  using C = Codec<S>;
  using T = typename C::T;
  using R = typename C::raw;
  constexpr int B = 64 * C::CPL;
  const int lane = (int)threadIdx.x & 63;
  const int st = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) + 1;  // this wave's step
  const Consts<T> Kc = load_consts<T>(L);
  const int lo = ch.walls & 3, hi = (ch.walls >> 2) & 3;
  // the lane's column; columns past a periodic side are their images, other
  // ones outside the lattice are clamped and never used
  const int ju = ch.j_first - STEPS + lane;
  auto column = [&](int j) {
    if (L.y_periodic) {
      if (j < 1) j += L.ny;
      else if (j > L.ny) j -= L.ny;
    }
    return min(max(j, 0), L.ny + 1);
  };
  auto place = [&](int j) {   // in a row of the lattice
    const unsigned jj = (unsigned)(j + B - 1);
    return ((jj / B) * (9u * B) + jj % B) * (unsigned)sizeof(R);
  };
  const int j = column(ju);
  const bool out = lane >= STEPS && lane < STEPS + ch.cols;
  const bool wall_lo = lo != 0 && ju == 1, wall_hi = hi != 0 && ju == L.ny;
  const bool zg = (wall_lo && lo == 1) || (wall_hi && hi == 1);
  // the lane beside a bounce-back wall's cell loads that cell's own outward
  // populations for it: the diagonals of row i itself, where the other lanes'
  // come from rows i -+ 1
  const bool helper = (lo == 2 && ju == 0) || (hi == 2 && ju == L.ny + 1);
  const unsigned p0 = place(j);
  // zero-gradient: the unknown directions are what the inner neighbour pulls,
  // from the wall cell's own column
  const unsigned pm = place(zg && wall_lo ? j : column(ju - 1));
  const unsigned pp = place(zg && wall_hi ? j : column(ju + 1));
  auto wrap = [&](int i) { return L.x_periodic ? (i < 1 ? i + L.nx : i > L.nx ? i - L.nx : i) : i; };
  auto row_at = [&](int i) {
    return (unsigned)wrap(i) * (unsigned)L.nbj * (9u * B * (unsigned)sizeof(R));
  };
  // step `st` computes rows i_first - (K - st) .. i_first + rows - 1 + (K - st)
  const int begin = 3 * (st - 1), count = ch.rows + 2 * (K - st);
  const int total = ch.rows + 3 * (K - 1);
  int i = ch.i_first - (K - st);
  T* const to = reinterpret_cast<T*>(smem) + (st - 1) * RING * PITCH + 1 + lane;
  const T* const from = to - RING * PITCH;
  auto fetch = [&](R (&r)[9], int row) {
    const unsigned r0 = row_at(row), rp = row_at(row + 1), rm = row_at(row - 1);
    const unsigned dp = helper ? r0 : rp, dm = helper ? r0 : rm;
#pragma unroll
    for (int k = 0; k < 9; ++k) {
      const unsigned at = CX[k] == 0 ? r0 : CX[k] < 0 ? (k > 4 ? dp : rp) : (k > 4 ? dm : rm);
      r[k] = *reinterpret_cast<const R*>(reinterpret_cast<const char*>(fsrc + k * B) +
                                         (at + (CY[k] == 0 ? p0 : CY[k] > 0 ? pm : pp)));
    }
  };
  int a3 = 0, a4 = 0;   // ring slots this row is written to (row number mod 3 and 4)
  // One row of step `st`, from its pulled populations on: moments, collision,
  // and the row's way on.
  auto finish = [&](T (&g)[9], auto stores) {
    const int cell = L.origin + wrap(i) * L.pitch + j;
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
    if (!decltype(stores)::value || st < K) {
      T* const w0 = to + a3 * 3 * PITCH;
      T* const wc = to + (RING_C + a4 * 3) * PITCH;
      if (sizeof(R) == 2 && (PAIRS ? !(st & 1) : !round_last)) {
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = tiled::through_storage<S>(g[k], k, key, Kc);
      }
#pragma unroll
      for (int k = 0; k < 9; ++k)
        (CX[k] == 0 ? w0 : CX[k] < 0 ? w0 + RING_B * PITCH : wc)[SLOT[k] * PITCH] = g[k];
    } else if (out) {
      // plain stores: a strip's segments end inside cache lines that the
      // next strip completes (non-temporal: FP32 8192x2048 91 us against 83)
      const unsigned at = row_at(i) + p0;
#pragma unroll
      for (int k = 0; k < 9; ++k)
        *reinterpret_cast<R*>(reinterpret_cast<char*>(fdst + k * B) + at) =
            C::encs(g[k], k, key, Kc);
      if (write_mom) {
        mdst[cell] = rho;
        mdst[L.plane + cell] = ux;
        mdst[2 * L.plane + cell] = uy;
      }
    }
    ++i;
    a3 = a3 == 2 ? 0 : a3 + 1;
    a4 = (a4 + 1) & 3;
  };
  auto barriers = [&](int n) {
#pragma unroll 1
    for (int q = 0; q < n; ++q) workgroup_barrier();
  };
  // The first step: rows from the lattice, in two sets of registers.  Where
  // storage and compute type agree a row is computed in its set while the next
  // row's loads fill the other; 16-bit rows are decoded first and their set
  // takes the row after the next.  (More rows in flight: no faster.)  Every
  // row fetches, the last ones the last row again, and nothing here stores to
  // memory, so that the compiler can wait for one row and leave the later one
  // in flight: in a loop that all steps shared it waited for all loads, and
  // copied each row (us per step before / after: FP64 8192x2048 149 / 142,
  // 4096x1024 MRT + Guo 62.5 / 57, FP32 4096x1024 MRT + Guo 28.6 / 24.4,
  // 2999x1111 17.2 / 16.5; FP32 8192x2048 72 / 74).
  auto first = [&](auto stores) {
    constexpr bool SAME = std::is_same<R, T>::value;
    constexpr int AHEAD = SAME ? 1 : 2;
    R raw[2][9];
    const int last = i + count - 1;
#pragma unroll
    for (int q = 0; q < AHEAD; ++q) fetch(raw[q], min(i + q, last));
    auto row = [&](auto set) {
      constexpr int u = decltype(set)::value;
      T apart[9];
      T (&g)[9] = values_of(raw[u], apart);
      if constexpr (!SAME) {
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = C::dec(raw[u][k], k, Kc);
      }
      fetch(raw[SAME ? 1 - u : u], min(i + AHEAD, last));
      if (lo == 2) {
        const T b4 = wave_from_prev(g[4]), b7 = wave_from_prev(g[7]), b8 = wave_from_prev(g[8]);
        if (wall_lo) {
          g[2] = b4;
          g[5] = b7;
          g[6] = b8;
        }
      }
      if (hi == 2) {
        const T b2 = wave_from_next(g[2]), b5 = wave_from_next(g[5]), b6 = wave_from_next(g[6]);
        if (wall_hi) {
          g[4] = b2;
          g[7] = b5;
          g[8] = b6;
        }
      }
      finish(g, stores);
      workgroup_barrier();
    };
    // no way out between the rows of a turn: with one the compiler moves the
    // sets at the loop's end, and waits for them
    int left = count;
#pragma unroll 1
    for (; left > 1; left -= 2) {
      row(std::integral_constant<int, 0>{});
      row(std::integral_constant<int, 1>{});
    }
    if (left > 0) row(std::integral_constant<int, 0>{});
    barriers(total - count);
  };
  // The steps after it.
  auto later = [&]() {
    barriers(begin);
#pragma unroll 1
    for (int t = 0; t < count; ++t) {
      T g[9];
      // rows i (number n + 1 of the step before), i + 1 (n + 2), i - 1 (n)
      const int same = (a3 == 2 ? 0 : a3 + 1) * 3;
      const int next = RING_B + (a3 == 0 ? 2 : a3 - 1) * 3;
      const T* const r0 = from + same * PITCH;
      const T* const rb = from + next * PITCH;
      const T* const rc = from + (RING_C + a4 * 3) * PITCH;
#pragma unroll
      for (int k = 0; k < 9; ++k)
        g[k] = (CX[k] == 0 ? r0 : CX[k] < 0 ? rb : rc)[SLOT[k] * PITCH - CY[k]];
      if ((lo | hi) && (wall_lo || wall_hi)) {
        const T* const own_b = from + (RING_B + same) * PITCH;
        const T* const own_c = from + (RING_C + ((a4 + 1) & 3) * 3) * PITCH;
#pragma unroll
        for (int k = 1; k < 9; ++k) {
          if (CY[k] == 0 || (CY[k] == 1 ? !wall_lo : !wall_hi)) continue;
          const int o = INV[k];
          g[k] = zg ? (CX[k] == 0 ? r0 : CX[k] < 0 ? rb : rc)[SLOT[k] * PITCH]
                    : (CX[o] == 0 ? r0 : CX[o] < 0 ? own_b : own_c)[SLOT[o] * PITCH];
        }
      }
      finish(g, std::true_type{});
      workgroup_barrier();
    }
    barriers(total - begin - count);
  };
  // every wave passes `total` barriers, in whichever loop
  if (st > K)
    barriers(total);
  else if (st > 1)
    later();
  else if (K > 1)
    first(std::false_type{});
  else
    first(std::true_type{});
}

// Waves per SIMD the registers must allow: the rings of three FP64 chunks
// (47.5 KB each) or six float ones fill a CU's LDS.
template <int S>
constexpr int waves_per_simd() {
  return S == D2Q9_STORE_F64 ? 4 : 6;
}

// Workgroups [0, n_tiles): tiles of TILE x TILE cells; the others: chunks.
template <int S, int MODEL, int FORCING, bool PAIRS>
__global__ __launch_bounds__(THREADS, waves_per_simd<S>()) void k_strip(
    const d2q9_lattice L, const d2q9_tiled_desc D, const d2q9_strip_desc P, int K,
    const typename Codec<S>::raw* __restrict__ fsrc, typename Codec<S>::raw* __restrict__ fdst,
    const typename Codec<S>::T* __restrict__ msrc, typename Codec<S>::T* __restrict__ mdst,
    int write_mom) {
  extern __shared__ __align__(16) char smem[];
  const int b = (int)blockIdx.x;
  if (b < P.n_tiles) {
    const d2q9_strip_tile it = P.tiles[b];
    tiled::run_tile<S, MODEL, FORCING, TILE_W, PAIRS>(L, D, smem, it.i_first, it.j_first, TILE,
                                                      K, TILE + 2 * K, 0, fsrc, fdst, msrc, mdst,
                                                      write_mom, nullptr, 0);
    return;
  }
  run_strip<S, MODEL, FORCING, PAIRS>(L, smem, P.chunks[xcd_remap(b - P.n_tiles, P.n_chunks)], K,
                                      fsrc, fdst, mdst, write_mom, D.round_last != 0);
}

struct Launch {
  int K, write_mom;
  const void* fsrc;
  void* fdst;
  const void* msrc;
  void* mdst;
  hipStream_t stream;
};

template <int S, int MODEL, int FORCING, bool PAIRS>
hipError_t launch_one(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                      const Launch& A) {
  using C = Codec<S>;
  auto kern = k_strip<S, MODEL, FORCING, PAIRS>;
  static PerDevice limit;
  if (const hipError_t e = tiled::allow_lds(limit, kern)) return e;
  size_t lds = ring_bytes<S>(A.K);
  if (P->n_tiles > 0) {
    const size_t t = tiled::lds_bytes<PAIRS>(*D, (TILE + 2 * A.K) * TILE_W, sizeof(typename C::T));
    if (t > lds) lds = t;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(P->n_tiles + P->n_chunks)), dim3(THREADS), lds,
                     A.stream, *L, *D, *P, A.K, static_cast<const typename C::raw*>(A.fsrc),
                     static_cast<typename C::raw*>(A.fdst),
                     static_cast<const typename C::T*>(A.msrc),
                     static_cast<typename C::T*>(A.mdst), A.write_mom);
  return hipGetLastError();
}

template <int S>
hipError_t launch(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                  const Launch& A);

template <int S, bool PAIRS>
hipError_t launch_kind(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                       const Launch& A) {
  switch (L->collision * 3 + L->forcing) {
    case 0: return launch_one<S, D2Q9_BGK, D2Q9_FORCING_NONE, PAIRS>(L, D, P, A);
    case 1: return launch_one<S, D2Q9_BGK, D2Q9_GUO_LINEAR, PAIRS>(L, D, P, A);
    case 2: return launch_one<S, D2Q9_BGK, D2Q9_GUO_SECOND_ORDER, PAIRS>(L, D, P, A);
    case 3: return launch_one<S, D2Q9_MRT, D2Q9_FORCING_NONE, PAIRS>(L, D, P, A);
    case 4: return launch_one<S, D2Q9_MRT, D2Q9_GUO_LINEAR, PAIRS>(L, D, P, A);
    case 5: return launch_one<S, D2Q9_MRT, D2Q9_GUO_SECOND_ORDER, PAIRS>(L, D, P, A);
  }
  return hipErrorInvalidValue;
}

template <int S>
hipError_t launch_model(const d2q9_lattice* L, const d2q9_tiled_desc* D, const d2q9_strip_desc* P,
                        const Launch& A) {
  if constexpr (sizeof(typename Codec<S>::raw) == 2) {
    if (D->pairs) return launch_kind<S, true>(L, D, P, A);
  }
  return launch_kind<S, false>(L, D, P, A);
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
