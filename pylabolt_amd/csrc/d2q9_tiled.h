// Tiled sweep: several fused time steps of a whole lattice per launch, for
// lattices that the caches hold.
//
// A workgroup owns an output tile of rows x cols cells.  It loads the
// post-collision populations of the tile grown by K cells on every side into
// LDS once, then runs K steps on them -- each step pulls from LDS,
// collides and writes back in place between two barriers, on a region that
// shrinks by one cell per step -- and stores the tile after the last.  The
// grown cells are computed by several workgroups with the same bits.
//
// Every kind of cell is swept here, so a launch has no second kernel and no
// fork and join: the nine values of a cell come from nine LDS positions
// that are set up once per launch.  For a plain cell they are its pull
// neighbours; at solids, bounce-back and zero-gradient walls the host
// resolves the rule to another position (a record of eight codes per
// special cell), and only moving walls and fixed-pressure nodes add
// arithmetic of their own, in the order of apply_bc.  Periodic sides are
// images in the grown region.  The arithmetic per cell is that of the
// single step and 16-bit storage rounds every step (the last of a launch
// only, or as the two-step sweep, when asked), so the result is bitwise that of
// K single steps in every storage form.
//
// What bounds it: for small lattices the latency of a launch (about 4 us
// of load, collide, store and hand-over) which the K steps share; for larger
// ones the work on the grown cells, (rows + 2K)(cols + 2K) / (rows cols) at
// the first step.  16-bit storage rounded in pairs (FP16 cylinder 900x700 7.4 us
// per step; 14.5 by the two-step sweep): where there is a rim, a second copy of
// the nine values in LDS, rounded after the first step of a pair in the cells
// that a rim cell pulls from, leaves two workgroups of 1024 cells per CU.
#pragma once
#include <hip/hip_runtime.h>

#include "d2q9_per_device.h"
#include "d2q9_sweep.h"

namespace d2q9 {
namespace tiled {

constexpr int MAX_ELEMS = 32;
constexpr int MAX_CELLS = 1024;   // of a region, one per thread

// Planes of LDS values besides the nine populations: rho where a cell is a
// moving wall's, u where one is at fixed pressure, and the rounded populations
// for the rim's cells (pairs == 2).  PAIRS: of a kernel that rounds pairs.
template <bool PAIRS>
__host__ __device__ inline int lds_planes(const d2q9_tiled_desc& D) {
  return 9 + (D.has_vel ? 1 : 0) + (D.has_pres ? 2 : 0) + (PAIRS && D.pairs == 2 ? 9 : 0);
}
template <bool PAIRS>
__host__ __device__ inline int lds_values(const d2q9_tiled_desc& D, int area) {
  return (area * lds_planes<PAIRS>(D) + 3) & ~3;
}
// LDS of a launch: the planes of every cell of the region and the boundary
// elements.
template <bool PAIRS>
__host__ __device__ inline size_t lds_bytes(const d2q9_tiled_desc& D, int area, size_t elem) {
  return (size_t)lds_values<PAIRS>(D, area) * elem + MAX_ELEMS * sizeof(d2q9_bc_elem);
}

// Value as the storage form keeps it from one step to the next.
template <int S>
__device__ __forceinline__ typename Codec<S>::T through_storage(
    typename Codec<S>::T v, int k, uint32_t key, const Consts<typename Codec<S>::T>& K) {
  if constexpr (sizeof(typename Codec<S>::raw) == 2)
    return Codec<S>::dec(Codec<S>::encs(v, k, key, K), k, K);
  else
    return v;
}

// Directions with arithmetic of their own: moving walls and fixed-pressure
// nodes (fluid_boundary_kernels.py:28-152), in the operation order of
// apply_bc.  `arith` names up to two boundary elements of a cell and their
// directions d (see d2q9_tiled_desc), for which g holds the cell's own
// outward population g_o, o = INV[d].  The term of direction d depends on
// c_o only through c_o . v, so a cell has four of them up to the sign
// (exactly), evaluated in registers.
//
// Moving walls: g_o - 2 w_o rho cs^-2 (c_o . U).
template <typename T>
__device__ __forceinline__ void apply_vel(const Consts<T>& K, uint32_t mask,
                                          const d2q9_bc_elem& el, T (&g)[9], T rho) {
  const T vx = (T)el.vec[0], vy = (T)el.vec[1];
  const T a1 = (((T)2 * K.w[1]) * rho) * K.ics2, a5 = (((T)2 * K.w[5]) * rho) * K.ics2;
  // by outward direction 1, 2, 5, 6; the opposite ones have the other sign
  const T t[4] = {a1 * vx, a1 * vy, a5 * (vx + vy), a5 * (-vx + vy)};
#pragma unroll
  for (int d = 1; d < 9; ++d) {
    const int o = INV[d], n = (o - 1) % 2 + (o > 4 ? 2 : 0);
    const bool neg = o == 3 || o == 4 || o == 7 || o == 8;
    if ((mask >> (d - 1)) & 1u) g[d] = g[d] - (neg ? -t[n] : t[n]);
  }
}

// Fixed pressure: -g_o + 2 w_o rho_b (1 + (c_o . u_e)^2 / (2 cs^4) - u_e^2 /
// (2 cs^2)), u_e extrapolated from the cell and its inward neighbour.
template <int S>
__device__ __forceinline__ void apply_pres(const Consts<typename Codec<S>::T>& K, uint32_t mask,
                                           const d2q9_bc_elem& el, typename Codec<S>::T (&g)[9],
                                           typename Codec<S>::T vx, typename Codec<S>::T vy,
                                           typename Codec<S>::T nx, typename Codec<S>::T ny) {
  using T = typename Codec<S>::T;
  const T ex = vx + (T)0.5 * (vx - nx);
  const T ey = vy + (T)0.5 * (vy - ny);
  const T u2 = ex * ex + ey * ey;
  const T h4 = (T)0.5 * K.ics4, hu = ((T)0.5 * K.ics2) * u2;
  const T rb = (T)el.scalar;
  const T cu[4] = {ex, ey, ex + ey, -ex + ey};
  T t[4];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
    const T w = K.w[n < 2 ? 1 : 5];
    if constexpr (Codec<S>::dev) {
      const T drb = (T)(el.scalar - 1.0);
      t[n] = ((T)2 * w) * (drb + rb * (h4 * cu[n] * cu[n] - hu));
    } else {
      t[n] = (((T)2 * w) * rb) * (((T)1 + h4 * cu[n] * cu[n]) - hu);
    }
  }
#pragma unroll
  for (int d = 1; d < 9; ++d) {
    const int o = INV[d], n = (o - 1) % 2 + (o > 4 ? 2 : 0);
    if ((mask >> (d - 1)) & 1u) g[d] = -g[d] + t[n];
  }
}

// K steps of the output tile of (rows - 2 K) x tile_c cells from (i_first,
// j_first) on, tile_c <= W - 2 K: region of `rows` x W cells, a wave holding 64 /
// W rows, one cell per thread.  LDS element of direction k of region
// cell e: 9 e + k (an odd stride: no bank conflicts, and every neighbour at
// a constant distance).  mom_steps, when not null, receives rho/u of every
// owned cell after every step (step s at mom_steps + s * mom_stride), and
// mdst is not written.  With collide_first the first step is moments and
// collision of the loaded populations alone (no streaming).  PAIRS: D.pairs is
// not 0 (a kernel of its own: in one with the other forms BF16 1024x256 took
// 3.86 us per step with every step rounded, 3.72 without).
template <int S, int MODEL, int FORCING, int W, bool PAIRS>
__device__ __forceinline__ void run_tile(
    const d2q9_lattice& L, const d2q9_tiled_desc& D, char* __restrict__ smem, int i_first,
    int j_first, int tile_c, int K, int rows, int collide_first, const typename Codec<S>::raw* __restrict__ fsrc,
    typename Codec<S>::raw* __restrict__ fdst, const typename Codec<S>::T* __restrict__ msrc,
    typename Codec<S>::T* __restrict__ mdst, int write_mom,
    typename Codec<S>::T* __restrict__ mom_steps, int64_t mom_stride) {
  using C = Codec<S>;
  using T = typename C::T;
  using R = typename C::raw;
  constexpr int B = 64 * C::CPL;
  const int e = (int)threadIdx.x;
  const int area = rows * W;
  T* const s = reinterpret_cast<T*>(smem);
  T* const srho = s + 9 * area;
  T* const su = srho + (D.has_vel ? area : 0);
  T* const srim = su + (D.has_pres ? 2 * area : 0);   // as s, 16-bit rims only
  d2q9_bc_elem* const elems = reinterpret_cast<d2q9_bc_elem*>(s + lds_values<PAIRS>(D, area));
  const Consts<T> Kc = load_consts<T>(L);
  const int i0 = i_first - K, j0 = j_first - K;   // the region's first cell
  // the whole region lies in the lattice: nothing to wrap or to leave out
  const bool inside = i0 > 0 && i0 + rows <= L.nx + 1 && j0 > 0 && j0 + W <= L.ny + 1;
  if (D.has_vel || D.has_pres)
    for (int n = e; n < D.n_elems * (int)(sizeof(d2q9_bc_elem) / 4); n += (int)blockDim.x)
      reinterpret_cast<uint32_t*>(elems)[n] = reinterpret_cast<const uint32_t*>(L.bc_elems)[n];
  // the cell's state through the steps
  int depth = 0;            // number of steps it takes part in
  bool own = false;         // the tile stores it
  bool keep = false;        // its moments are read by the next step
  uint32_t pop = 0;         // byte offset of its direction 0
  int32_t cell = 0;         // index in the side planes
  uint32_t from[4] = {};    // special cells: LDS elements to read, two a word
  uint32_t arith = 0;       // special cells: directions with arithmetic
  T ffx = (T)0, ffy = (T)0;
  // 16-bit storage: every step is rounded, or every second one
  const bool each = !PAIRS && sizeof(R) == 2 && !D.round_last;
  bool rim = false, near_rim = false;
  {
    const int r = e / W, c = e % W;
    int i = i0 + r, j = j0 + c;
    own = i <= L.nx && j <= L.ny && c < K + tile_c;
    if (!inside) {
      if (L.x_periodic) {
        while (i < 1) i += L.nx;
        while (i > L.nx) i -= L.nx;
      }
      if (L.y_periodic) {
        while (j < 1) j += L.ny;
        while (j > L.ny) j -= L.ny;
      }
    }
    if (r < rows && (unsigned)i <= (unsigned)L.nx + 1u && (unsigned)j <= (unsigned)L.ny + 1u) {
      const unsigned jj = (unsigned)(j + B - 1);
      pop = (((unsigned)i * (unsigned)L.nbj + jj / B) * (9u * B) + jj % B) * (unsigned)sizeof(R);
      cell = L.origin + i * L.pitch + j;
      // all loads of a plain cell are independent of one another
      R raw[9];
#pragma unroll
      for (int k = 0; k < 9; ++k)
        raw[k] = *reinterpret_cast<const R*>(reinterpret_cast<const char*>(fsrc + k * B) + pop);
      const uint32_t info = D.cells[cell];
      if (D.has_vel) srho[e] = msrc[cell];
      if (D.has_pres) {
        su[e] = msrc[L.plane + cell];
        su[area + e] = msrc[2 * L.plane + cell];
      }
      if (info & D2Q9_CELL_FLUID) {
        depth = min(min(r, rows - 1 - r), min(c, W - 1 - c));
        keep = (info & D2Q9_CELL_STORE_MOM) != 0;
        if (PAIRS && D.pairs == 2) {
          rim = (info & D2Q9_TILED_RIM) != 0;
          near_rim = (info & D2Q9_TILED_NEAR_RIM) != 0;
        }
        if (FORCING != D2Q9_FORCING_NONE && L.force_source == D2Q9_FSRC_FIELD) {
          const T* ff = static_cast<const T*>(L.force_field);
          ffx = ff[cell];
          ffy = ff[L.plane + cell];
        }
        if (info & (D2Q9_CELL_NEAR_SOLID | D2Q9_CELL_BC)) {
          // a wall or solid: where its rules take each direction from
          const uint4 v = reinterpret_cast<const uint4*>(D.codes)[info >> 8];
          arith = v.z;
#pragma unroll
          for (int d = 1; d < 9; ++d) {
            const uint32_t w = ((d < 5 ? v.x : v.y) >> (8 * ((d - 1) & 3))) & 0xffu;
            const uint32_t at = ((w & 3u) * W + ((w >> 2) & 3u)) * 9u + (w >> 4);
            from[(d - 1) >> 1] |= at << (16 * ((d - 1) & 1));
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 9; ++k) s[e * 9 + k] = C::dec(raw[k], k, Kc);
      if (PAIRS && D.pairs == 2) {
        // cells that are not fluid keep these
#pragma unroll
        for (int k = 0; k < 9; ++k) srim[e * 9 + k] = C::dec(raw[k], k, Kc);
      }
    }
    own = own && depth >= K;
  }
#pragma unroll 1
  for (int st = 1; st <= K; ++st) {
    __syncthreads();
    T g[9];
    if (depth >= st) {
      if (collide_first && st == 1) {
#pragma unroll
        for (int k = 0; k < 9; ++k) g[k] = s[e * 9 + k];
      } else {
        // the cell's neighbourhood
        const T* const p = (rim && !(st & 1) ? srim : s) + (e - W - 1) * 9;
        g[0] = p[(W + 1) * 9];
        if (from[0] == 0) {
#pragma unroll
          for (int d = 1; d < 9; ++d) g[d] = p[((1 - CX[d]) * W + 1 - CY[d]) * 9 + d];
        } else {
#pragma unroll
          for (int d = 1; d < 9; ++d)
            g[d] = p[(from[(d - 1) >> 1] >> (16 * ((d - 1) & 1))) & 0xffffu];
          if (arith) {
#pragma unroll 1
            for (int n = 0; n < 2; ++n) {
              const uint32_t sel = (arith >> 8) & 0xffu;
              const uint32_t mask = (n ? sel : ~sel) & arith & 0xffu;
              if (!mask) continue;
              const d2q9_bc_elem& el = elems[(arith >> (n ? 24 : 16)) & 0xffu];
              if (el.type == D2Q9_RULE_VEL) {
                apply_vel<T>(Kc, mask, el, g, srho[e]);
              } else {
                const int nb = e + el.normal[0] * W + el.normal[1];
                apply_pres<S>(Kc, mask, el, g, su[e], su[area + e], su[nb], su[area + nb]);
              }
            }
          }
        }
      }
    }
    __syncthreads();
    if (depth < st) continue;
    T drho, rho, ux, uy, fx, fy, px, py;
    moments<T, FORCING, C::dev>(g, L, Kc, ffx, ffy, drho, rho, ux, uy, fx, fy, px, py);
    collide<T, MODEL, FORCING, C::dev>(g, Kc, drho, rho, ux, uy, fx, fy, px, py);
    const uint32_t key = sizeof(R) == 2 ? cell_key((uint32_t)cell) : 0u;
    if (st < K) {
      const bool round = PAIRS ? !(st & 1) : each;
#pragma unroll
      for (int k = 0; k < 9; ++k)
        s[e * 9 + k] = round ? through_storage<S>(g[k], k, key, Kc) : g[k];
      if (near_rim && (st & 1)) {
#pragma unroll
        for (int k = 0; k < 9; ++k) srim[e * 9 + k] = through_storage<S>(g[k], k, key, Kc);
      }
      if (keep) {
        if (D.has_vel) srho[e] = rho;
        if (D.has_pres) {
          su[e] = ux;
          su[area + e] = uy;
        }
      }
    } else if (own) {
#pragma unroll
      for (int k = 0; k < 9; ++k)
        *reinterpret_cast<R*>(reinterpret_cast<char*>(fdst + k * B) + pop) =
            C::encs(g[k], k, key, Kc);
    }
    if (mom_steps || st == K) {
      if (own && (mom_steps || write_mom || keep)) {
        T* const m = (mom_steps ? mom_steps + (int64_t)(st - 1) * mom_stride : mdst) + cell;
        m[0] = rho;
        m[L.plane] = ux;
        m[2 * L.plane] = uy;
      }
    }
  }
}

// Waves per SIMD the registers must allow.  Floats fit eight (two workgroups
// of 1024 threads per CU); unforced FP64 takes 78 VGPRs, six waves, two
// workgroups of 768; with a force it would spill at that (1024x256 BGK +
// Guo 7.5 us per step against 6.6) and keeps one workgroup of up to 1024.
template <int S, int FORCING>
constexpr int waves_per_simd() {
  return S != D2Q9_STORE_F64 ? 8 : FORCING == D2Q9_FORCING_NONE ? 6 : 4;
}

template <int S, int MODEL, int FORCING, int W, bool PAIRS>
__global__ __launch_bounds__(MAX_CELLS, (waves_per_simd<S, FORCING>())) void k_tiled(
    const d2q9_lattice L, const d2q9_tiled_desc D, int ntiles, int ntj, int K, int rows,
    int collide_first, const typename Codec<S>::raw* __restrict__ fsrc,
    typename Codec<S>::raw* __restrict__ fdst, const typename Codec<S>::T* __restrict__ msrc,
    typename Codec<S>::T* __restrict__ mdst, int write_mom,
    typename Codec<S>::T* __restrict__ mom_steps, int64_t mom_stride) {
  extern __shared__ __align__(16) char smem[];
  const int tile = xcd_remap((int)blockIdx.x, ntiles);
  run_tile<S, MODEL, FORCING, W, PAIRS>(
      L, D, smem, 1 + (tile / ntj) * (rows - 2 * K), 1 + (tile % ntj) * (W - 2 * K), W - 2 * K, K,
      rows, collide_first, fsrc, fdst, msrc, mdst, write_mom, mom_steps, mom_stride);
}

// The checks of a descriptor every entry point makes (d2q9_tiled.hip): 0, or
// a D2Q9_E_* code with the error text set.
int check_desc(const d2q9_lattice* L, const d2q9_tiled_desc* D);

// Lets a kernel have all LDS of a CU on the current device, where more than
// 64 KB has to be asked for.
template <typename K>
hipError_t allow_lds(PerDevice& done, K* kern) {
  int device = 0;
  if (const hipError_t e = hipGetDevice(&device)) return e;
  return static_cast<hipError_t>(done.once(device, [kern] {
    return static_cast<int>(hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                                160 * 1024));
  }));
}

// Arguments of one launch.
struct Launch {
  int K, collide_first, write_mom;
  const void* fsrc;
  void* fdst;
  const void* msrc;
  void* mdst;
  void* mom_steps;
  int64_t mom_stride;
  hipStream_t stream;
};

// One launch of up to D->steps steps; instantiated once per storage form in
// its own translation unit (d2q9_tiled_<form>.hip).
template <int S>
hipError_t launch(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A);

template <int S, int MODEL, int FORCING, int W, bool PAIRS>
hipError_t launch_one(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A) {
  using C = Codec<S>;
  auto kern = k_tiled<S, MODEL, FORCING, W, PAIRS>;
  static PerDevice limit;
  if (const hipError_t e = allow_lds(limit, kern)) return e;
  // the region loses the rows a shorter launch does not need
  const int rows = D->rows - 2 * (D->steps - A.K);
  const int tr = rows - 2 * A.K, tc = W - 2 * A.K;
  const int ntj = (L->ny + tc - 1) / tc, tiles = (L->nx + tr - 1) / tr * ntj;
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles), dim3((unsigned)((rows * W + 63) / 64 * 64)),
                     lds_bytes<PAIRS>(*D, rows * W, sizeof(typename C::T)),
                     A.stream, *L, *D, tiles,
                     ntj, A.K, rows, A.collide_first, static_cast<const typename C::raw*>(A.fsrc),
                     static_cast<typename C::raw*>(A.fdst),
                     static_cast<const typename C::T*>(A.msrc),
                     static_cast<typename C::T*>(A.mdst), A.write_mom,
                     static_cast<typename C::T*>(A.mom_steps), A.mom_stride);
  return hipGetLastError();
}

template <int S, int MODEL, int FORCING, bool PAIRS>
hipError_t launch_width(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A) {
  switch (D->width) {
    case 16: return launch_one<S, MODEL, FORCING, 16, PAIRS>(L, D, A);
    case 32: return launch_one<S, MODEL, FORCING, 32, PAIRS>(L, D, A);
    case 64: return launch_one<S, MODEL, FORCING, 64, PAIRS>(L, D, A);
  }
  return hipErrorInvalidValue;
}

template <int S, int MODEL, int FORCING>
hipError_t launch_shape(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A) {
  if constexpr (sizeof(typename Codec<S>::raw) == 2) {
    if (D->pairs) return launch_width<S, MODEL, FORCING, true>(L, D, A);
  }
  return launch_width<S, MODEL, FORCING, false>(L, D, A);
}

template <int S>
hipError_t launch_model(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A) {
  switch (L->collision * 3 + L->forcing) {
    case 0: return launch_shape<S, D2Q9_BGK, D2Q9_FORCING_NONE>(L, D, A);
    case 1: return launch_shape<S, D2Q9_BGK, D2Q9_GUO_LINEAR>(L, D, A);
    case 2: return launch_shape<S, D2Q9_BGK, D2Q9_GUO_SECOND_ORDER>(L, D, A);
    case 3: return launch_shape<S, D2Q9_MRT, D2Q9_FORCING_NONE>(L, D, A);
    case 4: return launch_shape<S, D2Q9_MRT, D2Q9_GUO_LINEAR>(L, D, A);
    case 5: return launch_shape<S, D2Q9_MRT, D2Q9_GUO_SECOND_ORDER>(L, D, A);
  }
  return hipErrorInvalidValue;
}

#define D2Q9_TILED_DECLARE(SV) \
  template <>                  \
  hipError_t launch<SV>(const d2q9_lattice* L, const d2q9_tiled_desc* D, const Launch& A);
D2Q9_TILED_DECLARE(D2Q9_STORE_F64)
D2Q9_TILED_DECLARE(D2Q9_STORE_F32)
D2Q9_TILED_DECLARE(D2Q9_STORE_F16DEV)
D2Q9_TILED_DECLARE(D2Q9_STORE_BF16DEV)
#undef D2Q9_TILED_DECLARE

}  // namespace tiled
}  // namespace d2q9
