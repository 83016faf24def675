// j3d_stream_bf16.hip -- instantiates the register-streaming 3D kernels for bf16 storage.
#include "j3d_stream_kernel.h"
#include "j3d_sweep_kernel.h"

namespace perks {
void* j3s_kernel_bf16(int shape, int bc, int rows) { return j3s::sptr<j3g::bf16s>(shape, bc, rows); }
void* j3z_kernel_bf16(int shape, int bc, bool has_div) { return j3z::zptr<j3g::bf16s>(shape, bc, has_div); }
}  // namespace perks
