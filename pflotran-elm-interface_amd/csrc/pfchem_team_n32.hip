// pfchem_team_n32.hip -- instantiations of the batched kernel for teams of
// 32 rows (lanes per cell x rows per lane).
// One wave per SIMD: with the registers of two, both kernels spilled to
// scratch; with all of them the 32x1 kernels hold their rows without scratch,
// which is worth more than the second wave.  100,000 cells of 24 primaries and
// 80 complexes: FP64 17.5 -> 8.6 ms, mixed 18.9 -> 10.9 ms.  (8x4: the LDS of
// its eight cells allows no second wave.)
#define PFCHEM_TEAM_WAVES_PER_EU 1
#include "pfchem_team_impl.hpp"

namespace pfchem {

hipError_t launch_team_8_4(const DevNet& n, const DevNet* dn, const DevState* ds, int64_t ncell,
                          double dt, int mixed, const LaunchCfg& cfg,
                          unsigned long long* cursors, int num_cus, int nxcd,
                          hipStream_t stream, bool has_status) {
  return launch_pair<8, 4>(n, dn, ds, ncell, dt, mixed, cfg, cursors, num_cus, nxcd, stream,
                           has_status);
}

hipError_t launch_team_32_1(const DevNet& n, const DevNet* dn, const DevState* ds, int64_t ncell,
                          double dt, int mixed, const LaunchCfg& cfg,
                          unsigned long long* cursors, int num_cus, int nxcd,
                          hipStream_t stream, bool has_status) {
  return launch_pair<32, 1>(n, dn, ds, ncell, dt, mixed, cfg, cursors, num_cus, nxcd, stream,
                           has_status);
}

}  // namespace pfchem
