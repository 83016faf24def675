// j3d_persistent_bf16_shared.hip -- the persistent 3D kernels for BF16 storage, shared neighbour products.
#include "j3d_persistent_kernel.h"

namespace perks {
namespace j3dp {
template void* pick_bc<PERKS_BF16, false, kUpdShared>(int, bool, int);
}  // namespace j3dp
}  // namespace perks
