// pfchem_team_n64.hip -- instantiation of the batched kernel for teams of
// 64 rows: one cell per wavefront (networks of 33..64 unknowns).
// One wave per SIMD: the LDS of its cells allows no second one, and with the
// registers of two waves the FP32 kernel spilled enough to wait on scratch
// memory for 81 % of its time.  32,768 cells of 64 primaries: 78.4 ms with
// the registers of two, 57 ms with all.
#define PFCHEM_TEAM_WAVES_PER_EU 1
#include "pfchem_team_impl.hpp"

namespace pfchem {

hipError_t launch_team_64_1(const DevNet& n, const DevNet* dn, const DevState* ds, int64_t ncell,
                            double dt, int mixed, const LaunchCfg& cfg,
                            unsigned long long* cursors, int num_cus, int nxcd,
                            hipStream_t stream, bool has_status) {
  return launch_pair<64, 1>(n, dn, ds, ncell, dt, mixed, cfg, cursors, num_cus, nxcd, stream,
                            has_status);
}

}  // namespace pfchem
