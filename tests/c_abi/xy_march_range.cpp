// Which hybrid blocks take the x and y sweeps in one march: reads "nx ny nz"
// lines, prints 1 or 0 each (host code of the library only, no device needed).
#include <cstdio>

#include "ocfd_kernels.h"

int main() {
  int nx, ny, nz;
  while (std::scanf("%d %d %d", &nx, &ny, &nz) == 3) {
    ocfd::Block B = {};
    B.g.nx = nx;
    B.g.ny = ny;
    B.g.nz = nz;
    B.g.ni = (int64_t)nx * ny * nz;
    B.S.scheme_invis = ocfd::SCH_HYBRID;
    B.S.is_char = 1;
    B.S.flux_split = 2;
    for (int a = 0; a < 3; a++) B.S.iperiodic[a] = 1;
    B.M.uniform = 1;
    for (int prec : {ocfd::OCFD_PREC_FP64_CODE, ocfd::OCFD_PREC_MIXED_CODE}) {
      B.prec = prec;
      std::printf("%d ", ocfd::inviscid_xy_wins(B) ? 1 : 0);
    }
    std::printf("\n");
  }
  return 0;
}
