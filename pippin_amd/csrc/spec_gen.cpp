// Build-time generator of model-specialised kernel parameters.
//
// For each MJCF file given, compiles the model exactly as the library does at
// create time (build_host_model + init_dmodel_scalars) and prints a struct
// deriving from phk::DModel whose sizes and LDS layout are static constexpr
// members. The kernels are templates over the model type, so an instance for
// such a struct sees these values as compile-time constants (LDS offsets fold
// into immediate offsets, loop bounds are known), while the model's arrays
// and per-env parameter variants are read from the same device buffers as
// with the generic DModel. The runtime picks a specialised instance only when
// a model's values equal the struct's (spec_matches).
#include <cstdio>
#include <string>

#include "../../include/pippin_hip.h"
#include "host_model.hpp"

extern "C" int pippin_hip_model_load_file(const char* path, ph_model** out);
extern "C" const ph_model_desc* pippin_hip_model_desc(const ph_model* m);
void ph_set_error(const std::string&) {}

static void emit(const char* name, const phk::DModel& M) {
  const phk::Layout& L = M.L;
  // the layout as an aggregate, fields in declaration order
  printf("constexpr Layout %s_layout = {\n", name);
#define LF(f) printf("    %d,  // " #f "\n", L.f);
  LF(qpos) LF(qvel) LF(ctrl) LF(qacc) LF(applied) LF(xpos) LF(xquat) LF(xmat) LF(xipos) LF(jq) LF(cdof) LF(cinert)
  LF(crb) LF(cvel) LF(cacc) LF(cfrc) LF(qm) LF(chol) LF(H) LF(bias) LF(passive) LF(qfrc_act) LF(actf) LF(actclamp)
  LF(smooth) LF(qfrc_c) LF(acc) LF(vel) LF(gxpos) LF(gxmat) LF(aabb) LF(paircnt) LF(pairoff) LF(cact) LF(a) LF(a0)
  LF(grad) LF(p) LF(tmp) LF(tmp2) LF(mp) LF(J) LF(aref) LF(dd) LF(jar) LF(jp) LF(rpos) LF(rdiag) LF(ract) LF(rprev)
  LF(rf) LF(scal) LF(ndouble) LF(i_iscal) LF(i_isl) LF(nint) LF(bytes)
#undef LF
  printf("};\n");
  printf("struct %s : DModel {\n", name);
#define SZ(f) printf("  static constexpr int " #f " = %d;\n", M.f);
  SZ(nq) SZ(nv) SZ(nu) SZ(nbody) SZ(njnt) SZ(ngeom) SZ(ncam) SZ(neq) SZ(npair) SZ(nlevel) SZ(nblock) SZ(nacc)
  SZ(integrator) SZ(solver_kind) SZ(iterations) SZ(ncmax) SZ(nrmax) SZ(nrl) SZ(ngeneral) SZ(bmax)
#undef SZ
  printf("  static constexpr Layout L = %s_layout;\n", name);
  printf("  static bool matches(const DModel& m) {\n    return ");
  const char* f[] = {"nq", "nv", "nu", "nbody", "njnt", "ngeom", "ncam", "neq", "npair", "nlevel", "nblock", "nacc",
                     "integrator", "solver_kind", "iterations", "ncmax", "nrmax", "nrl", "ngeneral", "bmax"};
  for (const char* x : f) printf("m.%s == %s && ", x, x);
  printf("layout_equal(m.L, %s_layout);\n  }\n};\n\n", name);
}

int main(int argc, char** argv) {
  printf("// Generated by spec_gen from the models named below; do not edit.\n");
  printf("// Included after dmodel.hpp.\n#pragma once\n\nnamespace phk {\n\n");
  for (int i = 1; i + 1 < argc; i += 2) {
    ph_model* m;
    if (pippin_hip_model_load_file(argv[i + 1], &m)) {
      fprintf(stderr, "spec_gen: cannot load %s\n", argv[i + 1]);
      return 1;
    }
    phh::HostModel hm;
    std::string err;
    if (!phh::build_host_model(*pippin_hip_model_desc(m), hm, &err)) {
      fprintf(stderr, "spec_gen: %s: %s\n", argv[i + 1], err.c_str());
      return 1;
    }
    phk::DModel M{};
    phh::init_dmodel_scalars(hm, hm.d.solver_kind, 0, M);
    std::string path = argv[i + 1];
    printf("// %s\n", path.substr(path.find_last_of('/') + 1).c_str());
    emit(argv[i], M);
  }
  printf("}  // namespace phk\n");
  return 0;
}
