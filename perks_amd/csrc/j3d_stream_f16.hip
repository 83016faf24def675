// j3d_stream_f16.hip -- instantiates the register-streaming 3D kernels for f16 storage.
#include "j3d_stream_kernel.h"
#include "j3d_sweep_kernel.h"

namespace perks {
void* j3s_kernel_f16(int shape, int bc, int rows) { return j3s::sptr<j3g::f16s>(shape, bc, rows); }
void* j3z_kernel_f16(int shape, int bc, bool has_div) { return j3z::zptr<j3g::f16s>(shape, bc, has_div); }
}  // namespace perks
