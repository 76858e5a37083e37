// lane_host_girt.cpp -- runs the host build of a generated residual and
// Jacobian block (PFLANE_GIRT) over SoA state files, one cell at a time (test
// infrastructure, see lane_host_shim.h).
// usage: lane_host_girt <dir> <ncell> <ld> <dt> <ncomp>
// <dir>/<field>.bin holds each FP64 input; writes res.out ([ncomp][ld]),
// jac.out ([ncomp * ncomp][ld]), total.out, sec_molal.out, mnrl_rate.out.
#include <cstdio>
#include <cstdlib>
#include <string>
#include <vector>

static std::vector<char> slurp(const std::string& p) {
  std::vector<char> b;
  FILE* f = std::fopen(p.c_str(), "rb");
  if (!f) return b;
  std::fseek(f, 0, SEEK_END);
  b.resize(std::ftell(f));
  std::fseek(f, 0, SEEK_SET);
  if (!b.empty() && std::fread(b.data(), 1, b.size(), f) != b.size()) b.clear();
  std::fclose(f);
  return b;
}
static void spill(const std::string& p, const void* d, size_t n) {
  FILE* f = std::fopen(p.c_str(), "wb");
  std::fwrite(d, 1, n, f);
  std::fclose(f);
}

int main(int argc, char** argv) {
  if (argc < 6) return 2;
  const std::string dir = argv[1];
  pflane::GirtArgs a{};
  a.ncell = std::atoll(argv[2]);
  a.ld = std::atoll(argv[3]);
  a.dt = std::atof(argv[4]);
  const size_t n = (size_t)std::atoi(argv[5]);
  const char* names[] = {"pri_molal", "total", "immobile", "sec_molal", "pri_act_coef",
                         "sec_act_coef", "ln_act_h2o", "mnrl_volfrac", "mnrl_area", "mnrl_rate",
                         "porosity", "saturation", "den_kg", "volume", "temperature",
                         "fixed_total", "fixed_imm"};
  void** slots[] = {(void**)&a.pri_molal, (void**)&a.total, (void**)&a.immobile,
                    (void**)&a.sec_molal, (void**)&a.pri_act_coef, (void**)&a.sec_act_coef,
                    (void**)&a.ln_act_h2o, (void**)&a.mnrl_volfrac, (void**)&a.mnrl_area,
                    (void**)&a.mnrl_rate, (void**)&a.porosity, (void**)&a.saturation,
                    (void**)&a.den_kg, (void**)&a.volume, (void**)&a.temperature,
                    (void**)&a.fixed_total, (void**)&a.fixed_imm};
  std::vector<std::vector<char>> buf(17);
  for (int k = 0; k < 17; ++k) {
    buf[k] = slurp(dir + "/" + names[k] + ".bin");
    *slots[k] = buf[k].empty() ? nullptr : (void*)buf[k].data();
  }
  std::vector<double> res(n * a.ld), jac(n * n * a.ld);
  a.res = res.data();
  a.jac = jac.data();
  for (long long c = 0; c < a.ncell; ++c) {
    blockIdx.x = (unsigned)c;
    pfchem_lane_girt(a);
  }
  spill(dir + "/res.out", res.data(), res.size() * sizeof(double));
  spill(dir + "/jac.out", jac.data(), jac.size() * sizeof(double));
  for (int k : {1, 3, 9})
    if (!buf[k].empty()) spill(dir + "/" + names[k] + ".out", buf[k].data(), buf[k].size());
  return 0;
}
