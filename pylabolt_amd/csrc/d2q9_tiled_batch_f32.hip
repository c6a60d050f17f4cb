// Batched tiled sweep, f32 population storage.
#include "d2q9_tiled_batch.h"

namespace d2q9 {
namespace tiled {
D2Q9_TILED_BATCH_DEFINE(D2Q9_STORE_F32)
}  // namespace tiled
}  // namespace d2q9
