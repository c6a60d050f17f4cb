// C-ABI entries of the tiled sweep (kernels in d2q9_tiled.h and
// d2q9_tiled_batch.h, one translation unit per storage form).
#include <hip/hip_runtime.h>

#include "d2q9_tiled_batch.h"

using namespace d2q9;

namespace {

int tfail(int code, const char* what) {
  set_error(what);
  return code;
}

}  // namespace

int d2q9::tiled::check_desc(const d2q9_lattice* L, const d2q9_tiled_desc* D) {
  if (D->steps < 1 || (D->width != 16 && D->width != 32 && D->width != 64) ||
      2 * (int64_t)D->steps >= D->width || 2 * (int64_t)D->steps >= D->rows)
    return tfail(D2Q9_E_ARG, "tiled sweep: bad region or step count");
  if (D->pairs < 0 || D->pairs > 2 || (D->pairs && D->steps < 2))
    return tfail(D2Q9_E_ARG, "tiled sweep: bad pairs");
  if (D->n_elems < 0 || D->n_elems > tiled::MAX_ELEMS || (D->n_elems > 0 && !L->bc_elems) ||
      !D->cells || !D->codes)
    return tfail(D2Q9_E_ARG, "tiled sweep: bad special-cell tables");
  if ((int64_t)D->rows * D->width > tiled::MAX_CELLS)
    return tfail(D2Q9_E_TOO_LARGE, "tiled sweep: the region does not fit a workgroup");
  // cells are addressed by 32-bit byte offsets
  const uint64_t raw = L->storage == D2Q9_STORE_F64 ? 8 : (L->storage == D2Q9_STORE_F32 ? 4 : 2);
  if ((uint64_t)L->pop_len * raw > 0xffffffffull || L->plane > 0x7fffffffll)
    return tfail(D2Q9_E_TOO_LARGE, "tiled sweep: lattice over 4 GiB");
  return 0;
}

extern "C" int d2q9_tiled_steps(const d2q9_lattice* L, const d2q9_tiled_desc* D, void* f_a,
                                void* f_b, void* mom_a, void* mom_b, int32_t n,
                                int collide_first, int write_moments, void* mom_steps,
                                int64_t mom_stride, void* stream) {
  if (int r = validate_lattice(L)) return r;
  if (!D || !f_a || !f_b || !mom_a || !mom_b)
    return tfail(D2Q9_E_ARG, "tiled steps: null buffer");
  if (f_a == f_b || mom_a == mom_b)
    return tfail(D2Q9_E_ARG, "tiled steps: the two buffers must differ");
  if (n < 0) return tfail(D2Q9_E_ARG, "tiled steps: negative step count");
  if (int r = tiled::check_desc(L, D)) return r;
  const size_t elem = L->storage == D2Q9_STORE_F64 ? 8 : 4;
  if (n == 0) return 0;
  // launches of nearly equal length (the work on grown cells rises with their
  // steps; whole pairs of them where pairs are rounded, a single step left over
  // in the last launch, which has room for it)
  const int unit = D->pairs ? 2 : 1, most = D->steps / unit * unit;
  const int launches = n / most + (n % most != 0);
  const int base = n / unit / launches, longer = n / unit % launches;
  void* f[2] = {f_a, f_b};
  void* m[2] = {mom_a, mom_b};
  char* const per_step = static_cast<char*>(mom_steps);
  const int64_t step_bytes = mom_stride * (int64_t)elem;
  tiled::Launch A;
  A.stream = static_cast<hipStream_t>(stream);
  A.msrc = mom_a;
  A.mom_stride = mom_stride;
  int done = 0;
  for (int a = 0; a < launches; ++a) {
    A.K = unit * (base + (a < longer ? 1 : 0)) + (a == launches - 1 ? n % unit : 0);
    A.collide_first = a == 0 && collide_first;
    A.write_mom = a == launches - 1 && write_moments;
    A.fsrc = f[a & 1];
    A.fdst = f[1 - (a & 1)];
    A.mdst = m[1 - (a & 1)];
    A.mom_steps = per_step ? per_step + done * step_bytes : nullptr;
    hipError_t e = hipErrorInvalidValue;
    switch (L->storage) {
      case D2Q9_STORE_F64: e = tiled::launch<D2Q9_STORE_F64>(L, D, A); break;
      case D2Q9_STORE_F32: e = tiled::launch<D2Q9_STORE_F32>(L, D, A); break;
      case D2Q9_STORE_F16DEV: e = tiled::launch<D2Q9_STORE_F16DEV>(L, D, A); break;
      case D2Q9_STORE_BF16DEV: e = tiled::launch<D2Q9_STORE_BF16DEV>(L, D, A); break;
    }
    if (e != hipSuccess) {
      set_error(hipGetErrorString(e));
      return (int)e;
    }
    done += A.K;
    A.msrc = per_step ? per_step + (done - 1) * step_bytes : A.mdst;
  }
  return 0;
}

extern "C" int d2q9_tiled_batch(const d2q9_tiled_entry* entries, const d2q9_tiled_item* items,
                                int32_t n_items, int storage, int32_t rows, int32_t width,
                                int32_t steps, int32_t planes, int32_t n, int parity,
                                int collide_first, int write_moments, void* stream) {
  if (!entries || !items) return tfail(D2Q9_E_ARG, "tiled batch: null buffer");
  if (n < 0 || n_items < 0 || (parity != 0 && parity != 1) || planes < 9 || planes > 12 ||
      steps < 1 || (width != 16 && width != 32 && width != 64) || 2 * (int64_t)steps >= width ||
      2 * (int64_t)steps >= rows)
    return tfail(D2Q9_E_ARG, "tiled batch: bad region, steps, planes or parity");
  if ((int64_t)rows * width > tiled::MAX_CELLS)
    return tfail(D2Q9_E_TOO_LARGE, "tiled batch: the region does not fit a workgroup");
  if (storage != D2Q9_STORE_F64 && storage != D2Q9_STORE_F32)
    return tfail(D2Q9_E_UNSUPPORTED, "tiled batch: FP64 or FP32 storage only");
  if (n == 0 || n_items == 0) return 0;
  const int launches = (n + steps - 1) / steps;
  const int base = n / launches, longer = n % launches;
  tiled::BatchLaunch A;
  A.entries = entries;
  A.items = items;
  A.n_items = n_items;
  A.width = width;
  A.tile_c = width - 2 * steps;
  A.planes = planes;
  A.stream = static_cast<hipStream_t>(stream);
  for (int a = 0; a < launches; ++a) {
    A.K = base + (a < longer ? 1 : 0);
    A.rows = rows - 2 * (steps - A.K);
    A.collide_first = a == 0 && collide_first;
    A.write_mom = a == launches - 1 && write_moments;
    A.parity = (parity + a) & 1;
    const hipError_t e = storage == D2Q9_STORE_F64 ? tiled::launch_batch<D2Q9_STORE_F64>(A)
                                                   : tiled::launch_batch<D2Q9_STORE_F32>(A);
    if (e != hipSuccess) {
      set_error(hipGetErrorString(e));
      return (int)e;
    }
  }
  return 0;
}
