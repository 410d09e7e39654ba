// ocfd_inviscid_xyz_mixed.hip -- the three sweeps of a small block in one
// launch (k_inviscid_xyz, ocfd_sweep.h), FP32 for the mixed-precision form.
#include "ocfd_sweep.h"

namespace ocfd {

hipError_t launch_inviscid_xyz_mixed(const Block &B, hipStream_t st) { return launch_sweep_xyz<float>(B, st); }

}  // namespace ocfd
