// j3d_stream_f32.hip -- instantiates the register-streaming 3D kernels for f32 storage.
#include "j3d_stream_kernel.h"
#include "j3d_sweep_kernel.h"

namespace perks {
void* j3s_kernel_f32(int shape, int bc, int rows) { return j3s::sptr<float>(shape, bc, rows); }
void* j3z_kernel_f32(int shape, int bc, bool has_div) { return j3z::zptr<float>(shape, bc, has_div); }
}  // namespace perks
