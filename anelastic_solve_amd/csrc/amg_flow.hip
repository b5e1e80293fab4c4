// Time-stepper boundary handling and the implicit vertical viscous step:
//   ghost(var, vtype)            dns/BC.F90:1-187 (+ bound_update :334-584), serial
//   var_advance_CN_PL(...)       dns/NSsolver.F90:3054-3465, DNS branch: the Thomas
//                                solve of mgMK/mg_relax.F90:541-595 on every interior
//                                column, in segments (nz <= 256) or serially
// Fields are the reference's ghosted FP64 arrays, x fastest:
//   e(i,j,k) = (k*(ny+2) + j)*(nx+2) + i,   0 <= i <= nx+1 (ghosts 0 and nx+1).
// Floating-point contraction is off in this file: every product and sum is
// rounded as written, in the order of the Fortran source, so the results
// equal a plain IEEE evaluation of the reference's expressions (the
// segmented line solve, with explicit multiply-adds: to rounding).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <string>
#include <type_traits>
#include <vector>

#include "amg_flow.h"

#pragma clang fp contract(off)

namespace amg {
namespace {

constexpr int kFlowBlock = 256;

__device__ __forceinline__ size_t fidx(int i, int j, int k, int nx, int ny) {
  return ((size_t)k * (ny + 2) + j) * (size_t)(nx + 2) + i;
}

// Every ghost first takes its periodic image (dns/BC.F90:51-61: x, then y,
// then z over the full extents).  Composed, the three wraps map a ghost cell
// to the interior cell (w(i), w(j), w(k)) with w(0) = n, w(n+1) = 1, so each
// ghost is one copy from an interior cell and the copies are independent.
// Ghost cells are enumerated as the two z planes (full), the two y planes
// (interior k) and the two x planes (interior j, k).
__global__ __launch_bounds__(kFlowBlock) void k_flow_wrap(double* __restrict__ a, int nx, int ny,
                                                          int nz) {
  const long long t = (long long)blockIdx.x * kFlowBlock + threadIdx.x;
  const long long Z = 2LL * (nx + 2) * (ny + 2), Y = 2LL * (nx + 2) * nz, X = 2LL * ny * nz;
  int i, j, k;
  if (t < Z) {
    const long long pl = (nx + 2) * (long long)(ny + 2);
    k = t < pl ? 0 : nz + 1;
    const long long r = t % pl;
    j = (int)(r / (nx + 2));
    i = (int)(r % (nx + 2));
  } else if (t < Z + Y) {
    const long long u = t - Z, pl = (nx + 2) * (long long)nz;
    j = u < pl ? 0 : ny + 1;
    const long long r = u % pl;
    k = 1 + (int)(r / (nx + 2));
    i = (int)(r % (nx + 2));
  } else if (t < Z + Y + X) {
    const long long u = t - Z - Y, pl = (long long)ny * nz;
    i = u < pl ? 0 : nx + 1;
    const long long r = u % pl;
    k = 1 + (int)(r / ny);
    j = 1 + (int)(r % ny);
  } else {
    return;
  }
  const int si = i == 0 ? nx : (i == nx + 1 ? 1 : i);
  const int sj = j == 0 ? ny : (j == ny + 1 ? 1 : j);
  const int sk = k == 0 ? nz : (k == nz + 1 ? 1 : k);
  a[fidx(i, j, k, nx, ny)] = a[fidx(si, sj, sk, nx, ny)];
}

// One direction's face rules (bound_update) on every line of that direction,
// over the full extents of the other two (ghosts included); face 1 then face 2
// on the same line, as the reference calls them.  Products value*metric are
// precomputed on the host (FaceRule::prod, prod_rt).
__device__ __forceinline__ void face_rule(double* __restrict__ a, size_t base, long long st, int n,
                                          const FaceRule& R, int face, int d) {
  const int s = 1, e = n;
  auto at = [&](int q) -> double& { return a[base + (size_t)((long long)q * st)]; };
  switch (R.btype) {
    case 1:
      if (face == 1) at(s - 1) = R.value;
      else at(e + 1) = R.value;
      break;
    case 2:
      if (face == 1) {
        if (R.rt) at(s) = at(s + 1) - R.prod_rt;
        at(s - 1) = at(s) - R.prod;
      } else {
        if (R.rt) at(e) = at(e - 1) + R.prod_rt;
        at(e + 1) = at(e) + R.prod;
      }
      break;
    case 3:
      at(s - 1) = at(e);
      at(e + 1) = at(s);
      break;
    case 4:
      if (face == 1) at(s - 1) = at(s) - R.prod;
      else at(e + 1) = at(e) + R.prod;
      break;
    case 6:
      if (d == 2) {
        if (face == 1) at(s - 1) = 2.0 * R.value - 1.0 * at(s);
        else at(e + 1) = 2.0 * R.value - 1.0 * at(e);
      }
      break;
    case 7:
      if (d == 2) {
        if (face == 1) {
          at(s) = 0.0;
          at(s - 1) = -1.0 * at(s + 1);
        } else {
          at(e) = 0.0;
          at(e + 1) = -1.0 * at(e - 1);
        }
      }
      break;
    case 8:
      if (d == 0) {
        if (face == 1) at(s - 1) = 2.0 * at(s) - at(s + 1);
        else at(e + 1) = 2.0 * at(e) - at(e - 1);
      }
      break;
    default:
      break;
  }
}

__global__ __launch_bounds__(kFlowBlock) void k_flow_face(double* __restrict__ a, int nx, int ny,
                                                          int nz, int d, FaceRule r1, FaceRule r2,
                                                          int nrules) {
  const long long t = (long long)blockIdx.x * kFlowBlock + threadIdx.x;
  const int ex = nx + 2, ey = ny + 2;
  size_t base;
  long long st;
  int n;
  if (d == 0) {          // lines along x, one per (j, k)
    if (t >= (long long)ey * (nz + 2)) return;
    base = (size_t)t * ex;
    st = 1;
    n = nx;
  } else if (d == 1) {   // lines along y, one per (i, k)
    if (t >= (long long)ex * (nz + 2)) return;
    const long long k = t / ex, i = t % ex;
    base = (size_t)(k * ey) * ex + (size_t)i;
    st = ex;
    n = ny;
  } else {               // lines along z, one per (i, j)
    if (t >= (long long)ex * ey) return;
    base = (size_t)t;
    st = (long long)ex * ey;
    n = nz;
  }
  face_rule(a, base, st, n, r1, 1, d);
  if (nrules > 1) face_rule(a, base, st, n, r2, 2, d);
}

// The whole of ghost() for up to three fields in one launch, where every
// written cell's value follows from cells that nothing writes (ghost_fused):
// a thread takes one written cell, steps inward through the rules that hold
// it -- z, then y, then x, the last applied first -- and applies them outward
// again to the interior value it ends at, with the serial sequence's
// operations.  The sequence of one wrap and three face launches per field was
// all launch latency (64^3: 12 us of kernels per field, now 4.2).
struct GhostPlans {
  double* a[3];
  GhostPlan p[3];
};

// Whether rule R writes its face's ghost in direction d, and whether it also
// rewrites the interior layer next to it.
__host__ __device__ inline bool rule_writes(const FaceRule& R, int d) {
  return R.btype == 1 || R.btype == 2 || R.btype == 4 || ((R.btype == 6 || R.btype == 7) && d == 2) ||
         (R.btype == 8 && d == 0);
}
__host__ __device__ inline bool rule_layer(const FaceRule& R, int d) {
  return (R.btype == 2 && R.rt) || (R.btype == 7 && d == 2);
}

// One direction's step: the cell at c (0..n+1) of a line takes its value from
// the cell at src by the rule of face (0: the cell itself, wrapped where the
// direction has no rules).  A rule of type 8 also reads the cell beyond src.
struct GhostStep {
  int face, layer, src;
};
__device__ __forceinline__ GhostStep ghost_step(const GhostPlan& P, int d, int c, int n) {
  if (P.nrules[d] < 2) return {0, 0, c == 0 ? n : (c == n + 1 ? 1 : c)};
  const int f = (c == 0 || (c == 1 && rule_layer(P.r[d][0], d))) ? 1
              : (c == n + 1 || (c == n && rule_layer(P.r[d][1], d))) ? 2 : 0;
  if (f == 0) return {0, 0, c};
  const int in = rule_layer(P.r[d][f - 1], d) ? 2 : 1;   // layers in from the ghost
  return {f, c == 1 || c == n, f == 1 ? in : n + 1 - in};
}
// The value of a written cell from its source's value v (v2: the cell beyond).
__device__ __forceinline__ double ghost_apply(const FaceRule& R, const GhostStep& g, double v, double v2) {
  switch (R.btype) {
    case 1: return R.value;
    case 2: {
      if (R.rt) v = g.face == 1 ? v - R.prod_rt : v + R.prod_rt;
      if (R.rt && g.layer) return v;
      return g.face == 1 ? v - R.prod : v + R.prod;
    }
    case 4: return g.face == 1 ? v - R.prod : v + R.prod;
    case 6: return 2.0 * R.value - 1.0 * v;
    case 7: return g.layer ? 0.0 : -1.0 * v;
    default: return 2.0 * v - v2;
  }
}

__global__ __launch_bounds__(kFlowBlock) void k_flow_ghost(GhostPlans G, int nx, int ny, int nz) {
  const GhostPlan& P = G.p[blockIdx.y];
  double* __restrict__ a = G.a[blockIdx.y];
  // written layers per direction: the two ghosts, and the interior ones that
  // the direction's rules rewrite (at most four: l-th layer of direction d)
  auto layers = [&](int d) {
    int m = 2;
    if (P.nrules[d] == 2) m += rule_layer(P.r[d][0], d) + rule_layer(P.r[d][1], d);
    return m;
  };
  auto layer = [&](int d, int l, int n) {
    if (l < 2) return l == 0 ? 0 : n + 1;
    return l == 2 && rule_layer(P.r[d][0], d) ? 1 : n;
  };
  const int lx = layers(0), ly = layers(1), lz = layers(2);
  const int sx = nx + 2, sy = ny + 2;
  const int Z = lz * sx * sy, Y = ly * sx * nz, X = lx * ny * nz;
  int t = blockIdx.x * kFlowBlock + threadIdx.x;
  int i, j, k;
  if (t < Z) {
    const int l = t / (sx * sy);
    t -= l * sx * sy;
    k = layer(2, l, nz);
    j = t / sx;
    i = t - j * sx;
  } else if (t < Z + Y) {
    t -= Z;
    const int l = t / (sx * nz);
    t -= l * sx * nz;
    j = layer(1, l, ny);
    k = t / sx;
    i = t - k * sx;
    ++k;
  } else if (t < Z + Y + X) {
    // a line's layers on neighbouring lanes: they share cache lines with the
    // next line's
    t -= Z + Y;
    const int line = t / lx;
    i = layer(0, t - line * lx, nx);
    k = line / ny;
    j = line - k * ny;
    ++k;
    ++j;
  } else {
    return;
  }
  const GhostStep gz = ghost_step(P, 2, k, nz), gy = ghost_step(P, 1, j, ny), gx = ghost_step(P, 0, i, nx);
  const size_t e = fidx(gx.src, gy.src, gz.src, nx, ny);
  double v = a[e];
  if (gx.face) {
    const FaceRule& R = P.r[0][gx.face - 1];
    const double v2 = R.btype == 8 ? a[gx.face == 1 ? e + 1 : e - 1] : 0.0;
    v = ghost_apply(R, gx, v, v2);
  }
  if (gy.face) v = ghost_apply(P.r[1][gy.face - 1], gy, v, 0.0);
  if (gz.face) v = ghost_apply(P.r[2][gz.face - 1], gz, v, 0.0);
  a[fidx(i, j, k, nx, ny)] = v;
}

// Whether k_flow_ghost may take the plan: per direction either no rule (or
// the periodic one, which repeats the wrap), or both faces' rules write their
// ghosts, so that no written cell is read -- with interior layers rewritten
// only on lines of three cells or more, whose layers then read cells that
// stay.  Anything else runs the launches one by one.
bool ghost_fused(const GhostPlan& P, const int n[3]) {
  for (int d = 0; d < 3; ++d) {
    if (P.nrules[d] == 0 || (P.nrules[d] == 1 && P.r[d][0].btype == 3)) continue;
    if (P.nrules[d] != 2) return false;
    bool layers = false;
    for (const FaceRule& R : P.r[d]) {
      if (!rule_writes(R, d)) return false;
      layers = layers || rule_layer(R, d);
    }
    if (n[d] < (layers ? 3 : 1)) return false;
    if (n[d] < 2 && (P.r[d][0].btype == 8 || P.r[d][1].btype == 8)) return false;
  }
  return true;
}

// var_advance_CN_PL on one interior column (i, j) per lane (nz > 256;
// k_cn_seg below takes nz <= 256): the right-hand side of every physics row
// from the old values (f1*v2 + f2*v1*f3, the predicted
// pressure term when p is given, the explicit half of the vertical viscous
// term), the constant rows (walls, and rows a ghost rule zeroed), then the
// mgMK Thomas with the column-independent eliminated rows ap/bp: forward
// G_k = r_k + ap_k G_{k-1}, written into v2 as it goes (the old v2 values
// the next rows need are held in registers), and backward
// x_k = (G_k - c_k x_{k+1}) / bp_k.  Table row k (CnRow) is wave-uniform.
// Both passes run in chunks of rows (16 or 32 forward, 32 backward) whose
// loads (which do not depend on the recurrence) are issued before the
// chunk's dependent steps, so a thread keeps a chunk of loads in flight
// instead of one row.

// PV selects the predicted-pressure term at compile time: 0 none, 1 the x
// neighbour (u), 2 the y neighbour (v), 3 the z neighbour (w), so the march
// has no run-time branch on the variable.
template <int PV>
__global__ __launch_bounds__(kFlowBlock) void k_cn_column(const double* __restrict__ v1,
                                                          double* __restrict__ v2,
                                                          const double* __restrict__ p,
                                                          const CnRow* __restrict__ T,
                                                          const double* __restrict__ rdxe,
                                                          const double* __restrict__ rdye,
                                                          int nx, int ny, int nz, double f1,
                                                          double f2, double f3, double rkdt,
                                                          double h) {
  const int t = blockIdx.x * kFlowBlock + threadIdx.x;
  if (t >= nx * ny) return;
  const int i = 1 + t % nx, j = 1 + t / nx;
  const size_t st = (size_t)(nx + 2) * (ny + 2);
  const size_t base = (size_t)j * (nx + 2) + i;
  const int n = nz + 2;
  // the pressure neighbour is in the plane for u and v, one plane up for w
  // (clamped at the top row, which is a constant row); its metric is
  // per thread for u and v, per row (the table) for w
  constexpr bool pcv = PV != 0;
  const size_t poff = PV == 1 ? 1 : (size_t)(nx + 2);
  auto pnb = [&](int k) -> size_t {
    return PV == 3 ? base + (size_t)min(k + 1, n - 1) * st : base + (size_t)k * st + poff;
  };
  const double dmc = PV == 1 ? rdxe[i] : (PV == 2 ? rdye[j] : 0.0);
  // old values of rows k-1 and k; row 0 is a constant row, so vm is first
  // read at k = 1 (row 0)
  double vm = 0.0, vc = v2[base];
  double G = 0.0;
  // Every row evaluates the physics expression and a constant row then
  // selects its value, so no load is used only under a branch (the compiler
  // would move such loads down to their use and undo the prefetch).
  auto step = [&](int k, double vp, double a1, double pa, double pb) {
    const CnRow R = T[k];
    double r = f1 * vc + f2 * a1 * f3;
    if constexpr (pcv) r = r - rkdt * (pb - pa) * (PV == 3 ? R.pz : dmc);
    const double tv = R.c1 * (vp - vc) * R.m1 - R.c2 * (vc - vm) * R.m2;
    r = r + h * tv * R.m3;
    r = R.kind ? R.cval : r;
    G = k == 0 ? r : r + R.ap * G;
    v2[base + (size_t)k * st] = G;
    vm = vc;
    vc = vp;
  };
  // Forward, then backward, in self-contained chunks: all loads of a chunk
  // are issued together, then its dependent steps run.  With one column
  // per thread a 256^2 grid gives one wave per SIMD, so the chunks are made
  // long (deep prefetch) rather than double-buffered: a buffer live across
  // the loop's back edge would make the compiler wait for every load there.
  constexpr int KF = PV ? 16 : 32;
  constexpr int KB = 32;
  const int ncf = n / KF;
  for (int c = 0; c < ncf; ++c) {
    double vp[KF], a1[KF], pa[KF], pb[KF];
#pragma unroll
    for (int q = 0; q < KF; ++q) {
      const int kk = c * KF + q;
      vp[q] = v2[base + (size_t)min(kk + 1, n - 1) * st];   // the top row's is unused
      a1[q] = v1[base + (size_t)kk * st];
      if constexpr (pcv) {
        pa[q] = p[base + (size_t)kk * st];
        pb[q] = p[pnb(kk)];
      } else {
        pa[q] = pb[q] = 0.0;
      }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < KF; ++q) step(c * KF + q, vp[q], a1[q], pa[q], pb[q]);
  }
  for (int k = ncf * KF; k < n; ++k) {
    const double vp = v2[base + (size_t)min(k + 1, n - 1) * st];
    const double a1 = v1[base + (size_t)k * st];
    const double pa = pcv ? p[base + (size_t)k * st] : 0.0;
    const double pb = pcv ? p[pnb(k)] : 0.0;
    step(k, vp, a1, pa, pb);
  }
  // backward: the top row, the rows above the full chunks, then the chunks
  // downward (chunk b holds rows rb - q with rb = n - 2 - r0 - b*KB)
  double x = G / T[n - 1].bp;
  v2[base + (size_t)(n - 1) * st] = x;
  const int r0 = (n - 1) % KB;            // rows n-2 .. n-1-r0 go first, one by one
  for (int k = n - 2; k > n - 2 - r0; --k) {
    const size_t e = base + (size_t)k * st;
    x = (v2[e] - T[k].c * x) / T[k].bp;
    v2[e] = x;
  }
  const int ncb = (n - 1) / KB;
  for (int b = 0; b < ncb; ++b) {
    const int rb = n - 2 - r0 - b * KB;
    double g[KB];
#pragma unroll
    for (int q = 0; q < KB; ++q) g[q] = v2[base + (size_t)(rb - q) * st];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < KB; ++q) {
      const int kk = rb - q;
      x = (g[q] - T[kk].c * x) / T[kk].bp;
      v2[base + (size_t)kk * st] = x;
    }
  }
}

// The same step with every column split into P segments of S interior rows
// (at most kCnSeg rows and kCnSeg segments: nz <= 256), one wave per segment
// and 64 columns per workgroup.  The recurrences' coefficients are the same
// in every column, so their values are linear in the value carried into a
// segment, with factors that the host's table holds:
//   forward   G_k = G'_k + PF_k G_{r0-1},  PF_k = prod_{i=r0..k} ap_i,          G' from G_{r0-1} = 0,
//   backward  x_k = x'_k + QB_k x_{r1},    QB_k = prod_{i=k..r1-1} (-c_i/bp_i), x' from x_{r1} = 0.
// Each wave solves its segment, the segments' end values are chained through
// LDS (a scan over at most 16 segments), and each row adds its carry term.  The
// right-hand side is the serial kernel's, operation for operation (with products
// of constants made once and fused multiply-adds it was nearer to the exact
// value, 1.5e-16 against 1.6e-16, but further from the reference's evaluation:
// 1.9e-16); the solve is the serial kernel's to rounding.  The wall rows 0 and
// nz+1 are constant rows: their right-hand sides are numbers.  Every load comes
// before the first barrier and every store after the last, so the column is
// rewritten in place.
//
// It reads and writes each value once (24 B/cell, 32 with the pressure) and
// is bound by memory as long as two 1024-lane workgroups share a CU, one's
// loads under the other's chains: hence at most 64 registers, which is why the
// table's backward part goes through LDS and rows are addressed as a scalar
// row offset plus one lane offset (raw buffers).  256^3 u with the pressure
// (549 MB): 135 us; 161 with 86 registers and one workgroup per CU.
constexpr int kCnSeg = 16;     // rows per wave and waves per column group, at most
constexpr int kCnFwd = 9;      // table words of a row: c1 m1 c2 m2 m3 pz ap cval kind
constexpr int kCnBack = 4;     // and of its backward part: PF 1/bp c QB
struct CnEnds {
  double g0, c0, rb0;          // row 0: right-hand side, -c/bp of its super-diagonal, 1/bp
  double gt, at, rbt;          // row nz+1: right-hand side, eliminated sub-diagonal, 1/bp
};
typedef int int2v __attribute__((ext_vector_type(2)));
template <int PV>
__global__ __launch_bounds__(1024, 8) void k_cn_seg(const double* __restrict__ v1, double* v2,
                                                    const double* __restrict__ p,
                                                    const double* __restrict__ T,
                                                    const double* __restrict__ rdxe,
                                                    const double* __restrict__ rdye, int nx, int ny,
                                                    int nz, int S, double f1, double f2, double f3,
                                                    double rkdt, double h) {
  constexpr int N = kCnSeg;
  __shared__ double gend[N][64], xfirst[N][64], xtop[64], back[N][N * kCnBack];
  const int lane = threadIdx.x;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.y), P = blockDim.y;
  const int t = blockIdx.x * 64 + lane;
  const bool live = t < nx * ny;
  const int tc = live ? t : nx * ny - 1;              // a spare lane repeats the last column
  const int jr = tc / nx, i = 1 + tc - jr * nx, j = 1 + jr;
  const int r0 = 1 + w * S, len = min(S, nz + 1 - r0);
  // the segment's backward table, one word per lane
  const double* Bt = T + kCnFwd * (nz + 2) + sizeof(CnEnds) / 8;
  const double bw = Bt[w * (N * kCnBack) + lane];
  const CnEnds E = *reinterpret_cast<const CnEnds*>(T + kCnFwd * (nz + 2));
  const size_t st = (size_t)(nx + 2) * (ny + 2);
  const unsigned plane = (unsigned)st * 8u;
  // raw buffers from the row below the segment to the field's end
  const size_t off = (size_t)(r0 - 1) * st;
  const unsigned left = (unsigned)min((size_t)0x7fffffff, ((size_t)(nz + 2) * st - off) * 8);
  auto buf = [&](const double* a) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(a + off), 0, (int)left, 0x00027000);
  };
  const __amdgpu_buffer_rsrc_t b1 = buf(v1), b2 = buf(v2), bp = buf(PV ? p : v1);
  auto ld = [](__amdgpu_buffer_rsrc_t b, unsigned l, unsigned row) {
    return __builtin_bit_cast(double, (int2v)__builtin_amdgcn_raw_buffer_load_b64(b, (int)l, (int)row, 0));
  };
  const unsigned bl = (unsigned)(j * (nx + 2) + i) * 8u;
  const unsigned bn = bl + (PV == 1 ? 8u : (unsigned)(nx + 2) * 8u);   // the pressure's x or y neighbour
  const double dm = PV == 1 ? rdxe[i] : (PV == 2 ? rdye[j] : 0.0);
  // row q of the segment is q+1 rows past the buffers' start; rows past the
  // segment repeat its last row's upper neighbour
  auto row = [&](int q) { return (unsigned)min(q + 1, nz + 2 - r0) * plane; };
  double G[N];
  // right-hand sides of rows c0 .. c0+M-1
  auto rhs = [&](int c0, auto M) {
    constexpr int m = decltype(M)::value;
    double v[m + 2], a1[m], pa[m + 1], pb[m];
#pragma unroll
    for (int q = 0; q < m + 2; ++q) v[q] = ld(b2, bl, q == 0 && c0 == 0 ? 0u : row(c0 + q - 1));
#pragma unroll
    for (int q = 0; q < m; ++q) {
      a1[q] = ld(b1, bl, row(c0 + q));
      if constexpr (PV != 0) pa[q] = ld(bp, bl, row(c0 + q));
      if constexpr (PV == 1 || PV == 2) pb[q] = ld(bp, bn, row(c0 + q));
    }
    if constexpr (PV == 3) pa[m] = ld(bp, bl, row(c0 + m));
#pragma unroll
    for (int q = 0; q < m; ++q) {
      const double* R = T + kCnFwd * min(r0 + c0 + q, nz + 1);
      // the serial kernel's operations in their order
      double r = f1 * v[q + 1] + f2 * a1[q] * f3;
      if constexpr (PV == 1 || PV == 2) r = r - rkdt * (pb[q] - pa[q]) * dm;
      if constexpr (PV == 3) r = r - rkdt * (pa[q + 1] - pa[q]) * R[5];
      const double tv = R[0] * (v[q + 2] - v[q + 1]) * R[1] - R[2] * (v[q + 1] - v[q]) * R[3];
      r = r + h * tv * R[4];
      G[c0 + q] = R[8] != 0.0 ? R[7] : r;
    }
  };
  if (len == N) {
    rhs(0, std::integral_constant<int, N>());
  } else {
#pragma unroll
    for (int c0 = 0; c0 < N; c0 += 4)
      if (c0 < S) rhs(c0, std::integral_constant<int, 4>());
  }
  double g = 0.0;
#pragma unroll
  for (int q = 0; q < N; ++q)
    if (q < len) {
      g = __builtin_fma(T[kCnFwd * (r0 + q) + 6], g, G[q]);
      G[q] = g;
    }
  gend[w][lane] = g;
  back[w][lane] = bw;
  __syncthreads();
  // G_{r0-1}, the value carried into this segment (a segment's PF is its last
  // row's)
  double C = E.g0;
  for (int q = 0; q < w; ++q) C = __builtin_fma(back[q][(S - 1) * kCnBack], C, gend[q][lane]);
  const double* B = back[w];
  // the segment with its carry; then backward, locally
  double gl = g;
  double x = 0.0;
#pragma unroll
  for (int q = N - 1; q >= 0; --q)
    if (q < len) {
      const double Gq = __builtin_fma(B[q * kCnBack], C, G[q]);
      if (q == len - 1) gl = Gq;
      x = __builtin_fma(-B[q * kCnBack + 2], x, Gq) * B[q * kCnBack + 1];
      G[q] = x;
    }
  // the top wall row: G_{nz+1} from G_nz, x_{nz+1}
  if (w == P - 1) xtop[lane] = __builtin_fma(E.at, gl, E.gt) * E.rbt;
  xfirst[w][lane] = x;
  __syncthreads();
  // x_{r1}, the value carried into this segment from above, and the stores
  double X = xtop[lane];
  for (int q = P - 1; q > w; --q) X = __builtin_fma(back[q][3], X, xfirst[q][lane]);
  const unsigned bs = live ? bl : 0x80000000u;          // a spare lane's stores are dropped
  auto store = [&](double v, unsigned r) {
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(int2v, v), b2, (int)bs, (int)r, 0);
  };
  double x1 = 0.0;
#pragma unroll
  for (int q = N - 1; q >= 0; --q)
    if (q < len) {
      x1 = __builtin_fma(B[q * kCnBack + 3], X, G[q]);
      store(x1, (unsigned)(q + 1) * plane);
    }
  if (w == 0) store(__builtin_fma(E.c0, x1, E.g0 * E.rb0), 0u);
  if (w == P - 1) store(xtop[lane], (unsigned)(len + 1) * plane);
}

unsigned cdiv(long long a, int b) { return (unsigned)((a + b - 1) / b); }

// ghost()'s variable classes (dns/BC.F90:66-95) and bound_update's metrics
// (:384-447): l, rt, and per direction 0 = centre distance dxe, 1 = width dxc.
struct VClass {
  const char* name;
  int l, rt, bound;       // bound: bound_update knows the type
  int mx, my, mz, of1, of2;
};
const VClass kClasses[] = {
    {"u", 1, 0, 1, 1, 0, 0, 0, 1},       {"uc", 1, 0, 1, 0, 0, 0, -1, 0},
    {"v", 2, 0, 1, 0, 1, 0, 0, 1},       {"vc", 2, 0, 1, 0, 0, 0, -1, 0},
    {"w", 3, 0, 1, 0, 0, 1, 0, 1},       {"wc", 3, 0, 1, 0, 0, 0, -1, 0},
    {"p", 4, 0, 1, 0, 0, 0, -1, 0},      {"r", 5, 1, 0, 0, 0, 0, 0, 0},
    {"rho", 5, 1, 1, 0, 0, 0, -1, 0},    {"rf", 5, 1, 1, 0, 0, 0, -1, 0},
    {"cfluc", 6, 0, 1, 0, 0, 0, -1, 0},  {"fluc", 6, 0, 1, 0, 0, 0, -1, 0},
    {"rp", 6, 1, 1, 0, 0, 0, -1, 0},     {"psource", 7, 0, 1, 0, 0, 0, -1, 0},
    {"utemp", 7, 0, 1, 1, 0, 0, 0, 1},   {"vtemp", 7, 0, 1, 0, 1, 0, 0, 1},
    {"wtemp", 7, 0, 1, 0, 0, 1, 0, 1},   {"rtemp", 7, 0, 1, 0, 0, 0, -1, 0},
    {"s1temp", 7, 0, 1, 0, 0, 0, -1, 0}, {"scal1", 8, 1, 1, 0, 0, 0, -1, 0},
    {"scal1temp", 8, 0, 1, 0, 0, 0, -1, 0},
};

// The step's table from pinned host memory: as a kernel it costs a launch; the
// runtime's copy of the same few KB took the host and the stream 5 us more.
__global__ __launch_bounds__(kFlowBlock) void k_cn_table(const double* __restrict__ host,
                                                         double* __restrict__ table, int n) {
  const int e = blockIdx.x * kFlowBlock + threadIdx.x;
  if (e < n) table[e] = host[e];
}

}  // namespace

int plan_ghost(const FlowGrid& G, const char* vtype, const amg_flowbc& bc, GhostPlan* out,
               std::string* err) {
  const VClass* c = nullptr;
  for (const VClass& v : kClasses)
    if (vtype && std::strcmp(v.name, vtype) == 0) c = &v;
  if (!c) {
    *err = std::string("BC TYPE NOT AVAILABLE: ") + (vtype ? vtype : "(null)");
    return -1;
  }
  GhostPlan P{};
  P.bound = c->bound;
  const int n[3] = {G.nx, G.ny, G.nz};
  const int mk[3] = {c->mx, c->my, c->mz};
  for (int d = 0; d < 3; ++d) {
    const double* dt = mk[d] ? G.dxc[d] : G.dxe[d];
    const int l = c->l;
    auto TB = [&](int f) { return bc.tb[d + 3 * (f - 1) + 6 * (l - 1)]; };
    auto VB = [&](int f) { return bc.vb[d + 3 * (f - 1) + 6 * (l - 1)]; };
    const int s = 1, e = n[d];
    int nr = 0;
    for (int m = 1; m <= 2; ++m) {
      // face 1's type decides for both faces (dns/BC.F90:100-176)
      if (!(TB(1) != 3 || m == 1)) continue;
      FaceRule R{};
      R.btype = TB(m);
      R.rt = c->rt;
      R.value = VB(m);
      const int i1 = m == 1 ? s + c->of1 : e + c->of2;
      const int i2 = m == 1 ? s + 1 + c->of1 : e - 1 + c->of2;
      if (R.btype == 2 || R.btype == 4) {
        if (i1 < 0 || i1 > n[d] + 1 || i2 < 0 || i2 > n[d] + 1) {
          *err = "ghost: metric index out of range";
          return -1;
        }
        R.prod = R.value * dt[i1];
        R.prod_rt = R.value * dt[i2];
      }
      (m == 1 ? P.r[d][0] : P.r[d][1]) = R;
      nr = m;
    }
    P.nrules[d] = P.bound ? nr : 0;
  }
  P.fused = ghost_fused(P, n);
  *out = P;
  return 0;
}

static void launch_flow_ghost_steps(double* a, int nx, int ny, int nz, const GhostPlan& P, hipStream_t s) {
  const long long ng = 2LL * (nx + 2) * (ny + 2) + 2LL * (nx + 2) * nz + 2LL * ny * nz;
  hipLaunchKernelGGL(k_flow_wrap, dim3(cdiv(ng, kFlowBlock)), dim3(kFlowBlock), 0, s, a, nx, ny, nz);
  const long long lines[3] = {(long long)(ny + 2) * (nz + 2), (long long)(nx + 2) * (nz + 2),
                              (long long)(nx + 2) * (ny + 2)};
  for (int d = 0; d < 3; ++d) {
    if (P.nrules[d] == 0) continue;
    hipLaunchKernelGGL(k_flow_face, dim3(cdiv(lines[d], kFlowBlock)), dim3(kFlowBlock), 0, s, a, nx,
                       ny, nz, d, P.r[d][0], P.r[d][1], P.nrules[d]);
  }
}

void launch_flow_ghost(double* const* a, const GhostPlan* P, int nf, int nx, int ny, int nz,
                       hipStream_t s) {
  // (32-bit cell numbers: at most four layers per direction)
  const long long most = 4LL * (nx + 2) * (ny + 2) + 4LL * (nx + 2) * nz + 4LL * ny * nz;
  bool fused = most < (1LL << 31);
  for (int f = 0; f < nf; ++f) fused = fused && P[f].fused;
  if (!fused) {
    for (int f = 0; f < nf; ++f) launch_flow_ghost_steps(a[f], nx, ny, nz, P[f], s);
    return;
  }
  GhostPlans G{};
  long long cells = 0;
  for (int f = 0; f < nf; ++f) {
    G.a[f] = a[f];
    G.p[f] = P[f];
    int l[3];
    for (int d = 0; d < 3; ++d)
      l[d] = 2 + (P[f].nrules[d] == 2 ? rule_layer(P[f].r[d][0], d) + rule_layer(P[f].r[d][1], d) : 0);
    cells = std::max(cells, (long long)l[2] * (nx + 2) * (ny + 2) + (long long)l[1] * (nx + 2) * nz +
                                (long long)l[0] * ny * nz);
  }
  hipLaunchKernelGGL(k_flow_ghost, dim3(cdiv(cells, kFlowBlock), nf), dim3(kFlowBlock), 0, s, G, nx, ny,
                     nz);
}

int plan_cn(const FlowGrid& G, int var, double rkdt, double rRe, double rPr, double rSc,
            const amg_flowbc& bc, std::vector<CnRow>* rows, std::string* err) {
  const int nz = G.nz;
  const double* r = G.rho;
  const double* dzc = G.dxc[2];
  const double* dze = G.dxe[2];
  if (var != 1 && var != 2 && var != 3 && var != 5 && var != 8) {
    *err = "ABORTING ADVANCE CN, VARID IS NOT VALID";
    return -1;
  }
  std::vector<double> rdzc(nz + 2), rdze(nz + 2);
  for (int k = 0; k < nz + 2; ++k) {
    rdzc[k] = 1.0 / dzc[k];
    rdze[k] = 1.0 / dze[k];
  }
  // rows of the system, every column alike (dns/NSsolver.F90:3136-3216)
  std::vector<double> sub(nz + 2, 0.0), diag(nz + 2, 0.0), sup(nz + 2, 0.0);
  std::vector<CnRow> R(nz + 2);
  for (int k = 1; k <= nz; ++k) {
    double tmp1, tmp2;
    if (var == 1 || var == 2 || var == 5) {
      const double raver1 = 0.5 * (r[k + 1] + r[k]);
      const double raver2 = 0.5 * (r[k] + r[k - 1]);
      const double c = var == 5 ? rRe * rPr : rRe;
      tmp1 = c * raver1 / r[k];
      tmp2 = c * raver2 / r[k];
    } else if (var == 8) {
      tmp1 = tmp2 = rRe * rSc;
    } else {
      tmp1 = rRe * r[k] / (0.5 * (r[k + 1] + r[k]));
      tmp2 = rRe * r[k + 1] / (0.5 * (r[k + 1] + r[k]));
    }
    CnRow& w = R[k];
    w.c1 = tmp2;
    w.c2 = tmp1;
    w.pz = rdze[k];
    if (var == 3) {
      sub[k] = -0.5 * rkdt * tmp1 * rdze[k] * rdzc[k];
      sup[k] = -0.5 * rkdt * tmp2 * rdze[k] * rdzc[k + 1];
      diag[k] = 1.0 + 0.5 * rkdt * (tmp1 * rdzc[k] + tmp2 * rdzc[k + 1]) * rdze[k];
      w.m1 = rdzc[k + 1];
      w.m2 = rdzc[k];
      w.m3 = rdze[k];
    } else {
      sub[k] = -0.5 * rkdt * tmp1 * rdze[k - 1] * rdzc[k];
      sup[k] = -0.5 * rkdt * tmp2 * rdze[k] * rdzc[k];
      diag[k] = 1.0 + 0.5 * rkdt * (tmp1 * rdze[k - 1] + tmp2 * rdze[k]) * rdzc[k];
      w.m1 = rdze[k];
      w.m2 = rdze[k - 1];
      w.m3 = rdzc[k];
    }
  }
  // ghost(sub/diag/sup/rhs, 'cfluc') (:3331-3335): on interior columns only
  // the z rules reach rows that survive the wall rows below: type 7 zeroes
  // row sz (ez) of all four arrays.  Rows 0 and nz+1 are always rewritten
  // by the wall rows (every accepted type sets them).
  auto TB = [&](int f, int v) { return bc.tb[2 + 3 * (f - 1) + 6 * (v - 1)]; };
  auto VB = [&](int f, int v) { return bc.vb[2 + 3 * (f - 1) + 6 * (v - 1)]; };
  R[0].kind = R[nz + 1].kind = 1;
  for (int m = 1; m <= 2; ++m) {
    if (!(TB(1, 6) != 3 || m == 1)) continue;
    if (TB(m, 6) == 7) {
      const int k = m == 1 ? 1 : nz;
      sub[k] = diag[k] = sup[k] = 0.0;
      R[k].kind = 1;
      R[k].cval = 0.0;
    }
  }
  // the wall rows (:3337-3428)
  auto row = [&](int k, double a, double b, double c, double v) {
    sub[k] = a;
    diag[k] = b;
    sup[k] = c;
    R[k].kind = 1;
    R[k].cval = v;
  };
  const int s = 1, e = nz;
  int tb = TB(1, var);
  double vb = VB(1, var);
  if (tb == 1) {
    row(s - 1, 0.0, 1.0, 0.0, vb);
  } else if (tb == 2) {
    if (var == 3) {
      row(s - 1, 0.0, -1.0, 1.0, dzc[s - 1] * vb);
    } else if (var == 5 || var == 8) {
      row(s - 1, 0.0, -1.0, 1.0, dze[s - 1] * vb);
      row(s, 0.0, -1.0, 1.0, dze[s] * vb);
    } else {
      row(s - 1, 0.0, -1.0, 1.0, dze[s - 1] * vb);
    }
  } else if (tb == 6) {
    row(s - 1, 0.0, 1.0, 1.0, 2.0 * vb);
  } else {
    *err = "Incorrect BC for bottom for variable " + std::to_string(var) + " in var_advance_CN";
    return -1;
  }
  tb = TB(2, var);
  vb = VB(2, var);
  if (tb == 1) {
    row(e + 1, 0.0, 1.0, 0.0, vb);
  } else if (tb == 2) {
    if (var == 3) {
      row(e + 1, -1.0, 1.0, 0.0, dzc[e + 1] * vb);
    } else if (var == 5 || var == 8) {
      row(e + 1, -1.0, 1.0, 0.0, dze[e + 1] * vb);
      row(e, -1.0, 1.0, 0.0, dze[e] * vb);
    } else {
      row(e + 1, -1.0, 1.0, 0.0, dze[e + 1] * vb);
    }
  } else if (tb == 6) {
    row(e + 1, 1.0, 1.0, 0.0, 2.0 * vb);
  } else if (tb == 7) {
    row(e + 1, 0.0, 1.0, 0.0, 0.0);
    row(e, 0.0, 1.0, 0.0, 0.0);
  } else {
    *err = "Incorrect BC for top for variable " + std::to_string(var) + " in var_advance_CN";
    return -1;
  }
  // the matrix half of Thomas (mgMK/mg_relax.F90:577-581), the same for
  // every column
  std::vector<double> a = sub, b = diag;
  for (int j = 0; j < nz + 1; ++j) {
    if (b[j] == 0.0) {
      *err = "var_advance_CN: zero pivot in the vertical system";
      return -1;
    }
    a[j + 1] = -a[j + 1] / b[j];
    b[j + 1] = b[j + 1] + a[j + 1] * sup[j];
  }
  if (b[nz + 1] == 0.0) {
    *err = "var_advance_CN: zero pivot in the vertical system";
    return -1;
  }
  for (int k = 0; k < nz + 2; ++k) {
    R[k].ap = a[k];
    R[k].bp = b[k];
    R[k].c = sup[k];
  }
  *rows = std::move(R);
  return 0;
}

// The segmented kernel takes columns of at most 256 cells whose 18 rows of a
// segment lie within 2 GiB.
bool cn_segmented(int nx, int ny, int nz) {
  return nz <= kCnSeg * kCnSeg && (long long)(nx + 2) * (ny + 2) * 8 * (kCnSeg + 2) < (1LL << 31);
}

size_t cn_table_doubles(int nz) {
  return std::max(sizeof(CnRow) / 8 * (size_t)(nz + 2),
                  kCnFwd * (size_t)(nz + 2) + sizeof(CnEnds) / 8 + kCnSeg * kCnSeg * kCnBack);
}

std::vector<double> cn_table(const std::vector<CnRow>& rows, int nx, int ny) {
  const int nz = (int)rows.size() - 2;
  std::vector<double> t;
  if (!cn_segmented(nx, ny, nz)) {
    t.resize(sizeof(CnRow) / 8 * rows.size());
    std::memcpy(t.data(), rows.data(), sizeof(CnRow) * rows.size());
    return t;
  }
  for (const CnRow& R : rows) {
    const double fwd[kCnFwd] = {R.c1, R.m1, R.c2, R.m2, R.m3, R.pz, R.ap, R.cval, R.kind ? 1.0 : 0.0};
    t.insert(t.end(), fwd, fwd + kCnFwd);
  }
  const CnRow &B = rows.front(), &E = rows.back();
  for (double v : {B.cval, -(B.c / B.bp), 1.0 / B.bp, E.cval, E.ap, 1.0 / E.bp}) t.push_back(v);
  // segments of S <= 16 rows: PF downward from the segment's start, QB from
  // its end
  const int S = (nz + kCnSeg - 1) / kCnSeg;
  std::vector<double> back((size_t)kCnSeg * kCnSeg * kCnBack, 0.0);
  for (int r0 = 1, w = 0; r0 <= nz; r0 += S, ++w) {
    const int len = std::min(S, nz + 1 - r0);
    double* b = back.data() + (size_t)w * kCnSeg * kCnBack;
    long double pf = 1.0, qb = 1.0;   // (products in extended precision, rounded once)
    for (int q = 0; q < len; ++q) {
      const CnRow& R = rows[r0 + q];
      pf = R.ap * pf;
      b[q * kCnBack] = (double)pf;
      b[q * kCnBack + 1] = 1.0 / R.bp;
      b[q * kCnBack + 2] = R.c;
    }
    for (int q = len - 1; q >= 0; --q) {
      qb = -((long double)rows[r0 + q].c / rows[r0 + q].bp) * qb;
      b[q * kCnBack + 3] = (double)qb;
    }
  }
  t.insert(t.end(), back.begin(), back.end());
  return t;
}

void launch_cn_table(const double* host, double* table, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_cn_table, dim3(cdiv(n, kFlowBlock)), dim3(kFlowBlock), 0, s, host, table, n);
}

void launch_cn_column(const double* v1, double* v2, const double* p, const double* T,
                      const double* rdxe, const double* rdye, int nx, int ny, int nz, double f1,
                      double f2, double f3, double rkdt, int var, hipStream_t s) {
  const int pv = (p != nullptr && var <= 3) ? var : 0;
  const double h = rkdt * 0.5;
  if (cn_segmented(nx, ny, nz)) {
    const int S = (nz + kCnSeg - 1) / kCnSeg, P = (nz + S - 1) / S;
    const dim3 g(cdiv((long long)nx * ny, 64)), b(64, P);
#define CS(V) hipLaunchKernelGGL(k_cn_seg<V>, g, b, 0, s, v1, v2, p, T, rdxe, rdye, nx, ny, nz, S, f1, f2, f3, rkdt, h)
    if (pv == 1) CS(1);
    else if (pv == 2) CS(2);
    else if (pv == 3) CS(3);
    else CS(0);
#undef CS
    return;
  }
  const CnRow* R = reinterpret_cast<const CnRow*>(T);
  const dim3 g(cdiv((long long)nx * ny, kFlowBlock)), b(kFlowBlock);
#define CC(V) hipLaunchKernelGGL(k_cn_column<V>, g, b, 0, s, v1, v2, p, R, rdxe, rdye, nx, ny, nz, f1, f2, f3, rkdt, h)
  if (pv == 1) CC(1);
  else if (pv == 2) CC(2);
  else if (pv == 3) CC(3);
  else CC(0);
#undef CC
}

}  // namespace amg
