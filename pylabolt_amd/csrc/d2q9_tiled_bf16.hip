// Tiled sweep, bf16 population storage.
#include "d2q9_tiled.h"

namespace d2q9 {
namespace tiled {
template <>
hipError_t launch<D2Q9_STORE_BF16DEV>(const d2q9_lattice* L, const d2q9_tiled_desc* D,
                                  const Launch& A) {
  return launch_model<D2Q9_STORE_BF16DEV>(L, D, A);
}
}  // namespace tiled
}  // namespace d2q9
