// Strip sweep, f32 population storage.
#include "d2q9_strip.h"

namespace d2q9 {
namespace strip {
template <>
hipError_t launch<D2Q9_STORE_F32>(const d2q9_lattice* L, const d2q9_tiled_desc* D,
                                  const d2q9_strip_desc* P, const Launch& A) {
  return launch_model<D2Q9_STORE_F32>(L, D, P, A);
}
}  // namespace strip
}  // namespace d2q9
