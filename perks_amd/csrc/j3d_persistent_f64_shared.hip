// j3d_persistent_f64_shared.hip -- the persistent 3D kernels for FP64 storage, shared neighbour products.
#include "j3d_persistent_kernel.h"

namespace perks {
namespace j3dp {
template void* pick_bc<PERKS_F64, false, kUpdShared>(int, bool, int);
}  // namespace j3dp
}  // namespace perks
