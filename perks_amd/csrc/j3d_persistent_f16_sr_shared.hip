// j3d_persistent_f16_sr_shared.hip -- the persistent 3D kernels for FP16 storage, stochastic rounding, shared neighbour products.
#include "j3d_persistent_kernel.h"

namespace perks {
namespace j3dp {
template void* pick_bc<PERKS_F16, true, kUpdShared>(int, bool, int);
}  // namespace j3dp
}  // namespace perks
