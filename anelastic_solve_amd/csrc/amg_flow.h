// Time-stepper boundary handling (ghost) and the implicit vertical viscous
// step (var_advance_CN_PL): host planning and device launchers.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "amg.h"

namespace amg {

// Ghost-inclusive 1-D metrics of the finest grid (length n+2 per direction,
// direction 0/1/2 = x/y/z) and rho(z), as the instance's hierarchy holds them.
struct FlowGrid {
  int nx = 0, ny = 0, nz = 0;
  const double *dxc[3], *dxe[3];
  const double* rho;
};

// One face's bound_update rule with its products value*metric precomputed.
struct FaceRule {
  int btype;
  int rt;
  double value;
  double prod;      // value * metric at the ghost-side index
  double prod_rt;   // value * metric one further in (rtype == 1 rules)
};

// ghost(var, vtype): the periodic wrap of every ghost, then per direction
// nrules face rules (0 when the direction has nothing to apply).
struct GhostPlan {
  int bound;              // bound_update knows the type (else wraps only)
  int fused;              // the whole sequence is one pass (ghost_fused)
  FaceRule r[3][2];
  int nrules[3];
};

// One row k of the vertical CN system (every column alike): the eliminated
// sub-diagonal ap and pivot bp, the super-diagonal c, a constant right-hand
// side (kind 1) or the physics row's viscous factors c1, m1, c2, m2, m3.
struct CnRow {
  double ap, bp, c;
  double cval;
  double c1, m1, c2, m2, m3;
  double pz;        // 1/dze(k): the predicted-pressure metric of w
  int kind;
};

int plan_ghost(const FlowGrid& G, const char* vtype, const amg_flowbc& bc, GhostPlan* out,
               std::string* err);
// ghost() of nf (1 to 3) fields with a plan each.
void launch_flow_ghost(double* const* a, const GhostPlan* P, int nf, int nx, int ny, int nz,
                       hipStream_t s);

int plan_cn(const FlowGrid& G, int var, double rkdt, double rRe, double rPr, double rSc,
            const amg_flowbc& bc, std::vector<CnRow>* rows, std::string* err);
// The table a launch reads, as doubles: the rows themselves for the serial
// kernel, or the segmented kernel's (cn_segmented).
bool cn_segmented(int nx, int ny, int nz);
std::vector<double> cn_table(const std::vector<CnRow>& rows, int nx, int ny);
size_t cn_table_doubles(int nz);   // at most
// n doubles of it from pinned host memory to the device.
void launch_cn_table(const double* host, double* table, int n, hipStream_t s);
void launch_cn_column(const double* v1, double* v2, const double* p, const double* T,
                      const double* rdxe, const double* rdye, int nx, int ny, int nz, double f1,
                      double f2, double f3, double rkdt, int var, hipStream_t s);

}  // namespace amg
