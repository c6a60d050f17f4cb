// C-ABI entry of the strip sweep (kernel in d2q9_strip.h, one translation
// unit per storage form).
#include <hip/hip_runtime.h>

#include "d2q9_strip.h"

using namespace d2q9;

namespace {

int sfail(int code, const char* what) {
  set_error(what);
  return code;
}

}  // namespace

extern "C" int d2q9_strip_shape(int32_t* steps, int32_t* cols, int32_t* tile) {
  if (!steps || !cols || !tile) return sfail(D2Q9_E_ARG, "strip shape: null pointer");
  *steps = strip::STEPS;
  *cols = strip::COLS;
  *tile = strip::TILE;
  return 0;
}

extern "C" int d2q9_strip_steps(const d2q9_lattice* L, const d2q9_tiled_desc* D,
                                const d2q9_strip_desc* P, void* f_a, void* f_b, void* mom_a,
                                void* mom_b, int32_t n, int write_moments,
                                void* stream) {
  if (int r = validate_lattice(L)) return r;
  if (!D || !P || !f_a || !f_b || !mom_a || !mom_b)
    return sfail(D2Q9_E_ARG, "strip steps: null buffer");
  if (f_a == f_b || mom_a == mom_b)
    return sfail(D2Q9_E_ARG, "strip steps: the two buffers must differ");
  if (int r = tiled::check_desc(L, D)) return r;
  if (n < 0 || P->n_tiles < 0 || P->n_chunks < 0 || (P->n_tiles > 0 && !P->tiles) ||
      (P->n_chunks > 0 && !P->chunks) || (int64_t)P->n_tiles + P->n_chunks > 0x7fffffff)
    return sfail(D2Q9_E_ARG, "strip steps: bad step count or lists");
  if (n == 0 || P->n_tiles + P->n_chunks == 0) return 0;
  // as d2q9_tiled_steps: whole pairs where pairs are rounded
  const int unit = D->pairs ? 2 : 1;
  const int launches = (n + strip::STEPS - 1) / strip::STEPS;
  const int base = n / unit / launches, longer = n / unit % launches;
  void* f[2] = {f_a, f_b};
  void* m[2] = {mom_a, mom_b};
  strip::Launch A;
  A.stream = static_cast<hipStream_t>(stream);
  for (int a = 0; a < launches; ++a) {
    A.K = unit * (base + (a < longer ? 1 : 0)) + (a == launches - 1 ? n % unit : 0);
    A.write_mom = a == launches - 1 && write_moments;
    A.fsrc = f[a & 1];
    A.fdst = f[1 - (a & 1)];
    A.msrc = m[a & 1];
    A.mdst = m[1 - (a & 1)];
    hipError_t e = hipErrorInvalidValue;
    switch (L->storage) {
      case D2Q9_STORE_F64: e = strip::launch<D2Q9_STORE_F64>(L, D, P, A); break;
      case D2Q9_STORE_F32: e = strip::launch<D2Q9_STORE_F32>(L, D, P, A); break;
      case D2Q9_STORE_F16DEV: e = strip::launch<D2Q9_STORE_F16DEV>(L, D, P, A); break;
      case D2Q9_STORE_BF16DEV: e = strip::launch<D2Q9_STORE_BF16DEV>(L, D, P, A); break;
    }
    if (e != hipSuccess) {
      set_error(hipGetErrorString(e));
      return (int)e;
    }
  }
  return 0;
}
