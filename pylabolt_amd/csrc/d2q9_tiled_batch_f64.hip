// Batched tiled sweep, f64 population storage.
#include "d2q9_tiled_batch.h"

namespace d2q9 {
namespace tiled {
D2Q9_TILED_BATCH_DEFINE(D2Q9_STORE_F64)
}  // namespace tiled
}  // namespace d2q9
