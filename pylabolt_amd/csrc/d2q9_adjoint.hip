// Reverse-mode (adjoint) step of the FP64 D2Q9 BGK time step with Guo
// forcing and a fixed per-cell force field.
//
// Forward step at a fluid cell y (post-collision state p -> p'):
//   g = S(p)[y]                       pull streaming + bounce-back rules
//   rho = sum g,  u = (sum c g + F/2) / rho
//   p'_k = (1 - om) g_k + om feq_k(rho, u) + (1 - om/2) Fbar_k(u, F)
// The collision depends on g only through (rho, u), so with
//   lam' = dL/dp'  and  G_u = dL/du of this step (the loss seed),
//   A_rho = om sum_k lam'_k dfeq_k/drho
//   A_u   = sum_k lam'_k (om dfeq_k/du + (1 - om/2) dFbar_k/du) + G_u
//   mu_k  = dL/dg_k = (1 - om) lam'_k + A_rho + inv (c_k - u) . A_u
//   dL/dF += (1 - om/2) sum_k lam'_k dFbar_k/dF + (inv / 2) A_u
// with inv = 1 / (rho + float_min); then lam = S^T mu.  Streaming with
// bounce-back walls, periodic wraps and static solids is a permutation of
// the fluid populations, so S^T is a scatter in which every target is
// written exactly once: mu_d of cell y goes to the population it was pulled
// from -- (y - c_d, d) wrapped, or (y, inv(d)) where a bounce-back rule or a
// solid neighbour supplied it.  The caller guarantees that precondition
// (no moving walls, pressure or zero-gradient rules, no moving solids).
//
// The constants (inv_cs_2, inv_cs_4, weights) are the forward pass's, so the
// gradient is the exact derivative of the discrete FP64 map.
#include <hip/hip_runtime.h>

#include <string>

#include "d2q9_tiled.h"

using namespace d2q9;

namespace {

int afail(int code, const char* what) {
  set_error(what);
  return code;
}

constexpr int B64 = 64;

// The collision's transpose at one cell, in place: lam' -> mu, and this step's
// contribution to dL/dF.  The sums over k reduce to the weighted moments of
// lam' up to second order (w_k lam'_k against 1, c, cc), since feq and Fbar
// are quadratic in c: about 110 FP64 operations against 390 direction by
// direction.
struct AdjointConsts {
  double om, a, i4, fmin, w0, w1, w5;
};

__device__ __forceinline__ AdjointConsts adjoint_consts(const d2q9_lattice& L) {
  return {L.omega, L.inv_cs_2, L.inv_cs_4, L.float_min, L.w[0], L.w[1], L.w[5]};
}

template <int FORCING>
__device__ __forceinline__ void collide_transpose(const AdjointConsts& K, double (&g)[9],
                                                  double rho, double ux, double uy, double fx,
                                                  double fy, double seed_x, double seed_y,
                                                  double& gfx, double& gfy) {
  const double om = K.om, a = K.a, i4 = K.i4;
  const double inv = 1.0 / (rho + K.fmin);
  const double s13 = g[1] + g[3], s24 = g[2] + g[4], d13 = g[1] - g[3], d24 = g[2] - g[4];
  const double s57 = g[5] + g[7], s68 = g[6] + g[8], d57 = g[5] - g[7], d68 = g[6] - g[8];
  const double diag = K.w5 * (s57 + s68);
  const double mxx = K.w1 * s13 + diag, myy = K.w1 * s24 + diag, mxy = K.w5 * (s57 - s68);
  const double m0 = K.w0 * g[0] + (K.w1 * (s13 + s24) + diag);
  const double mx = K.w1 * d13 + K.w5 * (d57 - d68), my = K.w1 * d24 + K.w5 * (d57 + d68);
  // c . u against c, twice over: sum w lam (c . u) c
  const double cux = ux * mxx + uy * mxy, cuy = ux * mxy + uy * myy;
  const double a_rho =
      om * (m0 * (1.0 - (0.5 * a) * (ux * ux + uy * uy)) + a * (ux * mx + uy * my) +
            (0.5 * i4) * (ux * cux + uy * cuy));
  const double omr = om * rho, cf = 1.0 - 0.5 * om;
  double aux = omr * (a * (mx - ux * m0) + i4 * cux);
  double auy = omr * (a * (my - uy * m0) + i4 * cuy);
  gfx = gfy = 0.0;
  if constexpr (FORCING == D2Q9_GUO_LINEAR) {
    gfx = cf * (a * mx);
    gfy = cf * (a * my);
  } else if constexpr (FORCING == D2Q9_GUO_SECOND_ORDER) {
    aux += cf * (i4 * (fx * mxx + fy * mxy) - a * (fx * m0));
    auy += cf * (i4 * (fx * mxy + fy * myy) - a * (fy * m0));
    gfx = cf * (a * (mx - ux * m0) + i4 * cux);
    gfy = cf * (a * (my - uy * m0) + i4 * cuy);
  }
  aux += seed_x;
  auy += seed_y;
  const double ax = inv * aux, ay = inv * auy;
  gfx += 0.5 * ax;
  gfy += 0.5 * ay;
  const double base = a_rho - (ux * ax + uy * ay);
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    double v = base;
    if (CX[k] != 0) v = CX[k] > 0 ? v + ax : v - ax;
    if (CY[k] != 0) v = CY[k] > 0 ? v + ay : v - ay;
    g[k] = (1.0 - om) * g[k] + v;
  }
}

template <int FORCING, bool SCATTER>
__global__ __launch_bounds__(256) void k_adjoint(
    const d2q9_lattice L, const double* __restrict__ lam_src,
    double* __restrict__ lam_dst, const double* __restrict__ mom,
    const double* __restrict__ seed_u, double* __restrict__ grad_f) {
  const int64_t n = (int64_t)L.nx * L.ny;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int i = 1 + (int)(e / L.ny), j = 1 + (int)(e % L.ny);
  const int64_t c = cell_index(L, i, j);
  const uint8_t fl = L.flags[c];
  if (!(fl & D2Q9_CELL_FLUID)) return;
  const int64_t P = L.plane;
  const double* F = static_cast<const double*>(L.force_field);
  double mu[9];
#pragma unroll
  for (int k = 0; k < 9; ++k) mu[k] = lam_src[pop_index<B64>(L, i, j, k)];
  double gfx, gfy;
  collide_transpose<FORCING>(adjoint_consts(L), mu, mom[c], mom[P + c], mom[2 * P + c], F[c],
                             F[P + c], seed_u ? seed_u[c] : 0.0, seed_u ? seed_u[P + c] : 0.0,
                             gfx, gfy);
  grad_f[c] += gfx;
  grad_f[P + c] += gfy;
  if constexpr (!SCATTER) {
#pragma unroll
    for (int k = 0; k < 9; ++k) lam_dst[pop_index<B64>(L, i, j, k)] = mu[k];
    return;
  } else {
    lam_dst[pop_index<B64>(L, i, j, 0)] = mu[0];
    uint16_t rules[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    if (fl & D2Q9_CELL_BC) {
      const d2q9_bc_node node = L.bc_nodes[L.bc_slot[c]];
#pragma unroll
      for (int d = 0; d < 9; ++d) rules[d] = node.rule[d];
    }
#pragma unroll
    for (int d = 1; d < 9; ++d) {
      int xn = i - CX[d], yn = j - CY[d];
      bool bounce = (rules[d] & 15) == D2Q9_RULE_BB;
      if (!bounce && (fl & D2Q9_CELL_NEAR_SOLID))
        bounce = (L.flags[cell_index(L, xn, yn)] & D2Q9_CELL_SOLID) != 0;
      if (bounce) {
        lam_dst[pop_index<B64>(L, i, j, INV[d])] = mu[d];
        continue;
      }
      if (L.x_periodic) {
        if (xn == 0) xn = L.nx;
        else if (xn == L.nx + 1) xn = 1;
      }
      if (L.y_periodic) {
        if (yn == 0) yn = L.ny;
        else if (yn == L.ny + 1) yn = 1;
      }
      if (xn < 1 || xn > L.nx || yn < 1 || yn > L.ny) continue;  // from a ghost: no dependence
      lam_dst[pop_index<B64>(L, xn, yn, d)] = mu[d];
    }
  }
}

// K reverse steps of an output tile per launch, as the tiled forward sweep
// (d2q9_tiled.h: the same regions, special-cell records and LDS layout).  A
// reverse step is local up to its streaming: mu goes to LDS and the transpose
// of the pull gathers it back, lam_d(x) = mu_d(x + c_d), or the cell's own
// mu_{inv d} where the population p_d bounces back to it -- the directions
// whose record names the cell itself.  rho/u of a region cell are loaded a
// step ahead.  grad_f is read and written once per launch.
template <int FORCING, int W>
__global__ __launch_bounds__(tiled::MAX_CELLS) void k_adjoint_tiled(
    const d2q9_lattice L, const d2q9_tiled_desc D, int ntiles, int ntj, int K, int rows,
    int last_streamed, const double* __restrict__ lam_src, double* __restrict__ lam_dst,
    const double* __restrict__ mom, int64_t mom_stride, const double* __restrict__ seed_u,
    double* __restrict__ grad_f) {
  extern __shared__ __align__(16) char smem[];
  double* const s = reinterpret_cast<double*>(smem);
  const int tile = xcd_remap((int)blockIdx.x, ntiles);
  const int e = (int)threadIdx.x, r = e / W, c = e % W;
  const int i0 = 1 + (tile / ntj) * (rows - 2 * K) - K;
  const int j0 = 1 + (tile % ntj) * (W - 2 * K) - K;
  int i = i0 + r, j = j0 + c;
  bool own = i <= L.nx && j <= L.ny;
  if (L.x_periodic) {
    while (i < 1) i += L.nx;
    while (i > L.nx) i -= L.nx;
  }
  if (L.y_periodic) {
    while (j < 1) j += L.ny;
    while (j > L.ny) j -= L.ny;
  }
  const AdjointConsts Kc = adjoint_consts(L);
  int depth = -1;           // the last reverse step the cell collides in
  uint32_t pop = 0, bounce = 0;
  int32_t cell = 0;
  double g[9], fx = 0.0, fy = 0.0, gx = 0.0, gy = 0.0, sx = 0.0, sy = 0.0;
  double rho = 1.0, ux = 0.0, uy = 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) g[k] = 0.0;
  if (r < rows && i >= 1 && i <= L.nx && j >= 1 && j <= L.ny) {
    const unsigned jj = (unsigned)(j + B64 - 1);
    pop = ((unsigned)i * (unsigned)L.nbj + jj / B64) * (9u * B64) + jj % B64;
    cell = L.origin + i * L.pitch + j;
    const uint32_t info = D.cells[cell];
    if (info & D2Q9_CELL_FLUID) {
      depth = min(min(r, rows - 1 - r), min(c, W - 1 - c));
      const double* F = static_cast<const double*>(L.force_field);
#pragma unroll
      for (int k = 0; k < 9; ++k) g[k] = lam_src[pop + (unsigned)(k * B64)];
      fx = F[cell];
      fy = F[L.plane + cell];
      rho = mom[cell];
      ux = mom[L.plane + cell];
      uy = mom[2 * L.plane + cell];
      if (seed_u) {
        sx = seed_u[cell];
        sy = seed_u[L.plane + cell];
      }
      if (info & (D2Q9_CELL_NEAR_SOLID | D2Q9_CELL_BC)) {
        const uint4 v = reinterpret_cast<const uint4*>(D.codes)[info >> 8];
#pragma unroll
        for (int d = 1; d < 9; ++d) {
          const uint32_t w = ((d < 5 ? v.x : v.y) >> (8 * ((d - 1) & 3))) & 0xffu;
          if ((w & 0xfu) == 5u) bounce |= 1u << INV[d];  // from the cell itself
        }
      }
    }
  }
  own = own && depth >= K;
  if (own) {
    gx = grad_f[cell];
    gy = grad_f[L.plane + cell];
  }
#pragma unroll 1
  for (int st = 0; st < K; ++st) {
    // a step ahead: rho/u of the step before (in time)
    double rho1 = 1.0, ux1 = 0.0, uy1 = 0.0;
    if (st + 1 < K && depth > st) {
      const double* const m = mom - (int64_t)(st + 1) * mom_stride + cell;
      rho1 = m[0];
      ux1 = m[L.plane];
      uy1 = m[2 * L.plane];
    }
    if (depth >= st) {
      double gfx, gfy;
      collide_transpose<FORCING>(Kc, g, rho, ux, uy, fx, fy, sx, sy, gfx, gfy);
      gx += gfx;
      gy += gfy;
    }
    sx = sy = 0.0;
    if (st + 1 < K || last_streamed) {
      if (r < rows) {
#pragma unroll
        for (int k = 0; k < 9; ++k) s[e * 9 + k] = g[k];
      }
      __syncthreads();
      if (depth > st) {
        const double* const p = s + (e - W - 1) * 9;
#pragma unroll
        for (int d = 1; d < 9; ++d)
          g[d] = (bounce >> d) & 1u ? s[e * 9 + INV[d]]
                                    : p[((1 + CX[d]) * W + 1 + CY[d]) * 9 + d];
      }
      __syncthreads();
    }
    rho = rho1;
    ux = ux1;
    uy = uy1;
  }
  if (own) {
#pragma unroll
    for (int k = 0; k < 9; ++k) lam_dst[pop + (unsigned)(k * B64)] = g[k];
    grad_f[cell] = gx;
    grad_f[L.plane + cell] = gy;
  }
}

// dL/du0 (and dL/drho0) from mu_1 = dL/dg_0, g_0 = feq(rho0, u0).
__global__ __launch_bounds__(256) void k_adjoint_init(const d2q9_lattice L,
                                                      const double* __restrict__ mu,
                                                      const double* __restrict__ mom0,
                                                      double* __restrict__ grad_init) {
  const int64_t n = (int64_t)L.nx * L.ny;
  const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  const int i = 1 + (int)(e / L.ny), j = 1 + (int)(e % L.ny);
  const int64_t c = cell_index(L, i, j);
  const int64_t P = L.plane;
  if (!(L.flags[c] & D2Q9_CELL_FLUID)) {
    grad_init[c] = 0.0;
    grad_init[P + c] = 0.0;
    grad_init[2 * P + c] = 0.0;
    return;
  }
  const double a = L.inv_cs_2, b = 0.5 * L.inv_cs_4, c0 = 0.5 * L.inv_cs_2;
  const double rho = mom0[c], ux = mom0[P + c], uy = mom0[2 * P + c];
  const double u2 = ux * ux + uy * uy;
  double gr = 0.0, gx = 0.0, gy = 0.0;
#pragma unroll
  for (int k = 0; k < 9; ++k) {
    const double m = mu[pop_index<B64>(L, i, j, k)];
    const double cx = CX[k], cy = CY[k], w = L.w[k];
    const double cu = cx * ux + cy * uy;
    gr += m * w * (1.0 + a * cu + b * cu * cu - c0 * u2);
    gx += m * w * rho * (a * cx + 2.0 * b * cu * cx - 2.0 * c0 * ux);
    gy += m * w * rho * (a * cy + 2.0 * b * cu * cy - 2.0 * c0 * uy);
  }
  grad_init[c] = gr;
  grad_init[P + c] = gx;
  grad_init[2 * P + c] = gy;
}

int check(const d2q9_lattice* L) {
  if (!L) return afail(D2Q9_E_ARG, "null lattice descriptor");
  if (L->storage != D2Q9_STORE_F64 || L->cpl != 1)
    return afail(D2Q9_E_UNSUPPORTED, "the adjoint runs on FP64 storage");
  if (L->collision != D2Q9_BGK) return afail(D2Q9_E_UNSUPPORTED, "the adjoint needs BGK");
  if (L->force_source != D2Q9_FSRC_FIELD || !L->force_field)
    return afail(D2Q9_E_UNSUPPORTED, "the adjoint needs a per-cell force field");
  if (!L->flags) return afail(D2Q9_E_ARG, "null flags");
  return 0;
}

}  // namespace

extern "C" {

int d2q9_adjoint_step(const d2q9_lattice* L, int streamed, const void* lam_src,
                      void* lam_dst, const void* mom, const void* seed_u,
                      void* grad_force, void* stream) {
  if (int r = check(L)) return r;
  if (!lam_src || !lam_dst || !mom || !grad_force || lam_src == lam_dst)
    return afail(D2Q9_E_ARG, "adjoint buffers: null or aliased");
  const int64_t n = (int64_t)L->nx * L->ny;
  const unsigned blocks = (unsigned)((n + 255) / 256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto ls = static_cast<const double*>(lam_src);
  auto ld = static_cast<double*>(lam_dst);
  auto m = static_cast<const double*>(mom);
  auto su = static_cast<const double*>(seed_u);
  auto gf = static_cast<double*>(grad_force);
#define D2Q9_ADJ(FO)                                                                  \
  if (streamed)                                                                       \
    hipLaunchKernelGGL((k_adjoint<FO, true>), dim3(blocks), dim3(256), 0, s, *L, ls, ld, \
                       m, su, gf);                                                    \
  else                                                                                \
    hipLaunchKernelGGL((k_adjoint<FO, false>), dim3(blocks), dim3(256), 0, s, *L, ls,  \
                       ld, m, su, gf);
  switch (L->forcing) {
    case D2Q9_FORCING_NONE: D2Q9_ADJ(D2Q9_FORCING_NONE) break;
    case D2Q9_GUO_LINEAR: D2Q9_ADJ(D2Q9_GUO_LINEAR) break;
    case D2Q9_GUO_SECOND_ORDER: D2Q9_ADJ(D2Q9_GUO_SECOND_ORDER) break;
    default: return afail(D2Q9_E_ARG, "bad forcing");
  }
#undef D2Q9_ADJ
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(hipGetErrorString(e));
    return (int)e;
  }
  return 0;
}

int d2q9_adjoint_steps(const d2q9_lattice* L, const d2q9_tiled_desc* D, int32_t n,
                       int last_streamed, const void* lam_src, void* lam_dst, const void* mom,
                       int64_t mom_stride, const void* seed_u, void* grad_force, void* stream) {
  if (int r = check(L)) return r;
  if (int r = validate_lattice(L)) return r;
  if (!D || !lam_src || !lam_dst || !mom || !grad_force || lam_src == lam_dst)
    return afail(D2Q9_E_ARG, "adjoint steps: buffers null or aliased");
  if (int r = tiled::check_desc(L, D)) return r;
  if (n < 1 || n > D->steps) return afail(D2Q9_E_ARG, "adjoint steps: 1 .. steps per launch");
  const int rows = D->rows - 2 * (D->steps - n);
  const int tr = rows - 2 * n, tc = D->width - 2 * n;
  const int ntj = (L->ny + tc - 1) / tc, tiles = (L->nx + tr - 1) / tr * ntj;
  const dim3 grid((unsigned)tiles), block((unsigned)((rows * D->width + 63) / 64 * 64));
  const size_t lds = (size_t)rows * D->width * 9 * sizeof(double);
  hipStream_t s = static_cast<hipStream_t>(stream);
  auto ls = static_cast<const double*>(lam_src);
  auto ld = static_cast<double*>(lam_dst);
  auto m = static_cast<const double*>(mom);
  auto su = static_cast<const double*>(seed_u);
  auto gf = static_cast<double*>(grad_force);
  hipError_t e = hipErrorInvalidValue;
#define D2Q9_ADJ_ONE(FO, WV)                                                                   \
  case WV: {                                                                                   \
    auto kern = k_adjoint_tiled<FO, WV>;                                                       \
    static PerDevice limit;                                                                    \
    if ((e = tiled::allow_lds(limit, kern)) != hipSuccess) break;                              \
    hipLaunchKernelGGL(kern, grid, block, lds, s, *L, *D, tiles, ntj, n, rows, last_streamed,  \
                       ls, ld, m, mom_stride, su, gf);                                         \
    e = hipGetLastError();                                                                     \
    break;                                                                                     \
  }
#define D2Q9_ADJ_TILED(FO)                                                                     \
  switch (D->width) {                                                                          \
    D2Q9_ADJ_ONE(FO, 16)                                                                       \
    D2Q9_ADJ_ONE(FO, 32)                                                                       \
    D2Q9_ADJ_ONE(FO, 64)                                                                       \
  }
  switch (L->forcing) {
    case D2Q9_GUO_LINEAR: D2Q9_ADJ_TILED(D2Q9_GUO_LINEAR) break;
    case D2Q9_GUO_SECOND_ORDER: D2Q9_ADJ_TILED(D2Q9_GUO_SECOND_ORDER) break;
    default: return afail(D2Q9_E_UNSUPPORTED, "adjoint steps: a Guo forcing is needed");
  }
#undef D2Q9_ADJ_TILED
#undef D2Q9_ADJ_ONE
  if (e != hipSuccess) {
    set_error(hipGetErrorString(e));
    return (int)e;
  }
  return 0;
}

int d2q9_adjoint_init_grad(const d2q9_lattice* L, const void* mu, const void* mom0,
                           void* grad_init, void* stream) {
  if (int r = check(L)) return r;
  if (!mu || !mom0 || !grad_init) return afail(D2Q9_E_ARG, "null buffer");
  const int64_t n = (int64_t)L->nx * L->ny;
  hipLaunchKernelGGL(k_adjoint_init, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), *L, static_cast<const double*>(mu),
                     static_cast<const double*>(mom0), static_cast<double*>(grad_init));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error(hipGetErrorString(e));
    return (int)e;
  }
  return 0;
}

}  // extern "C"
