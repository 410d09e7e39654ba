// ocfd_inviscid_xyz.hip -- the three sweeps of a small block in one launch
// (k_inviscid_xyz, ocfd_sweep.h), FP64.
#include "ocfd_sweep.h"

namespace ocfd {

hipError_t launch_inviscid_xyz_mixed(const Block &B, hipStream_t st);

hipError_t launch_inviscid_xyz(const Block &B, hipStream_t st) {
  if (!B.du2 || !B.du3 || !prims_match(B)) return hipErrorInvalidValue;
  if (B.prec == OCFD_PREC_MIXED_CODE) return launch_inviscid_xyz_mixed(B, st);
  return launch_sweep_xyz<double>(B, st);
}

}  // namespace ocfd
