// pfchem_lane.h -- library-internal interface of the network-specialized
// lane kernel (device source pfchem_lane.hpp, host side pfchem_lane.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "pfchem.h"

namespace pfchem {

// networks the lane kernel takes (the team kernel takes the others)
constexpr int kLaneMaxAq = 16;
constexpr int kLaneMaxCplx = 256;
constexpr int kLaneMaxMnrl = 16;
// per-lane LDS doubles of one cell's state (x 256 lanes x 8 B <= 160 KB)
constexpr int kLaneMaxLdsFields = 80;

// kernel arguments; the same layout as pflane::Args in pfchem_lane.hpp
struct LaneArgs {
  long long ld, ncell;
  double* pri_molal;
  double* total;
  double* immobile;
  double* sec_molal;
  double* pri_act_coef;
  double* sec_act_coef;
  double* ln_act_h2o;
  double* mnrl_volfrac;
  const double* mnrl_area;
  double* mnrl_rate;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  int* num_iterations;
  int* num_sub_steps;
  int* status;
  unsigned long long* cursors;
  double dt;
  int nxcd;
  int rescue;
  int escalate;
  int list_min;
  const int* list;
  const int* list_count;
  int* esc_list;
  unsigned long long* esc_count;
  const double* sd_ft;
  const double* sd_fw;
};
static_assert(sizeof(LaneArgs) == 240, "LaneArgs layout");

// adjoint kernel arguments; the same layout as pflane::SensArgs
struct LaneSensArgs {
  long long ld, ncell;
  const double* pri_molal;
  const double* total;
  const double* pri_act_coef;
  const double* sec_act_coef;
  const double* ln_act_h2o;
  const double* mnrl_volfrac;
  const double* mnrl_area;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  const double* wv;
  const double* ws;
  double* grad;
  long long ldo;
  double* fcell;
  int* status;
  double* log;
  long long ldl;
  double dt;
  int jacobian;
  int pad;
};
static_assert(sizeof(LaneSensArgs) == 192, "LaneSensArgs layout");
constexpr int kLaneSensSub = 8;  // sub-steps the adjoint kernel records per cell
// first line of an adjoint module's source (followed by lane_source)
constexpr char kLaneAdjointDefine[] = "#define PFLANE_ADJOINT 1\n";

// GIRT block kernel arguments; the same layout as pflane::GirtArgs
struct LaneGirtArgs {
  long long ld, ncell;
  const double* pri_molal;
  double* total;
  const double* immobile;
  double* sec_molal;
  const double* pri_act_coef;
  const double* sec_act_coef;
  const double* ln_act_h2o;
  const double* mnrl_volfrac;
  const double* mnrl_area;
  double* mnrl_rate;
  const double* porosity;
  const double* saturation;
  const double* den_kg;
  const double* volume;
  const double* temperature;
  const double* fixed_total;
  const double* fixed_imm;
  double* res;
  double* jac;
  double dt;
};
static_assert(sizeof(LaneGirtArgs) == 176, "LaneGirtArgs layout");
// Complexes up to which the GIRT block runs one cell per lane.  The kernel is
// faster at every size (131,072 cells, 5 minerals, block against the team
// kernel: 15 x 60 123 / 588 us, 16 x 100 155 / 809, 16 x 150 217 / 1,085,
// 16 x 200 354 / 1,343), but its module is compiled in the first call, and it
// holds a coefficient per complex: 1.8 s at 60, 5.7 s and 172 B of scratch at
// 150, 9.5 s and 884 B at 200, 12.8 s at 250.  The line keeps the first call
// under that of the largest SomDec step (7 s).
constexpr int kLaneGirtMaxCplx = 160;
// prefix of lane_source that makes a GIRT module
constexpr char kLaneGirtDefine[] = "#define PFLANE_GIRT 1\n";

// networks of at least this many primaries evaluate mass action as products
// of powers (pfchem_lane.hpp)
constexpr int kProdMinAq = 9;

// 1 if the lane kernel handles this network and these options (else `why`)
int lane_supported(const pfchem_network* net, const pfchem_options* opt, std::string& why);
// Entries of the SomDec Jacobian pattern up to which the step kernel takes a
// network.  Its unrolled elimination grows with the pattern, and with it the
// first step's compile and the FP64 kernel's scratch.  200,000 cells, one step
// of the default against the team kernel alone, FP64 and mixed:
//   entries  unknowns  compile  scratch    FP64 ms        mixed ms
//   115      15        2.2 s    144 B      26.3 / 34.2    26.5 / 38.8
//   181      24        5.2 s    976 B      63.4 / 216     64.0 / 396
//   271      22        6.9 s    1,856 B    38.4 / 49.1    38.7 / 74.6
//   389      26        17.8 s   3,920 B    29.6 / 45.4    21.5 / 59.7
// (most of the default's time is the handed-over cells').  Beyond 288 the
// compile grows faster than the pattern (528 entries: 2-3 times the 389 ones)
// for what a step gains, so larger networks keep the team kernel, which
// compiles nothing.
constexpr int kSdMaxEntries = 288;
// 1 if the step kernel takes this network with its SomDec sandbox (no
// complexes, minerals, Monod oxygen response, O2 tracking or activity update
// per Newton iteration, at most kSdMaxEntries pattern entries)
int lane_sd_supported(const pfchem_network* net, const pfchem_options* opt);
// full device source: the network as constants followed by the template
std::string lane_source(const pfchem_network* net, const pfchem_options* opt);
// compile `src` for gfx950 and load it on `device` (cached per process)
int lane_compile(const std::string& src, int device, std::string& err);
// compile only (no device needed); code object in *code when non-null
int lane_compile_only(const std::string& src, std::vector<char>* code, std::string& err);
// launch the FP32 (f32 = 1) or FP64 kernel of a compiled source over
// args.ncell cells; persistent grid of num_cus x min(blocks_per_cu,
// occupancy) workgroups of 256 lanes (blocks_per_cu <= 0: occupancy).  With
// nclear > 0 one fill kernel first clears that many cursors (the passes of a
// step use consecutive sets of nxcd) and *args.esc_count.
hipError_t lane_launch(const std::string& src, int device, int f32, const LaneArgs& args,
                       int num_cus, int blocks_per_cu, unsigned long long* cursors, int nclear,
                       hipStream_t stream);
// launch the GIRT kernel of a compiled source, one cell per lane
hipError_t lane_girt_launch(const std::string& src, int device, const LaneGirtArgs& args,
                            hipStream_t stream);
// launch the adjoint kernel of a compiled source, one cell per lane
hipError_t lane_adjoint_launch(const std::string& src, int device, const LaneSensArgs& args,
                               hipStream_t stream);

}  // namespace pfchem
