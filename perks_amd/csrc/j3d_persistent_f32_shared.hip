// j3d_persistent_f32_shared.hip -- the persistent 3D kernels for FP32 storage, shared neighbour products.
#include "j3d_persistent_kernel.h"

namespace perks {
namespace j3dp {
template void* pick_bc<PERKS_F32, false, kUpdShared>(int, bool, int);
}  // namespace j3dp
}  // namespace perks
