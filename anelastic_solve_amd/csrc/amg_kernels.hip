// amg_kernels.hip -- gfx950 kernels of the multigrid pressure solve.
//
// Every V-cycle kernel runs over a work list: one launch covers the same
// step of several instances/levels (LaunchList in amg_internal.h), so a
// single solve and a batch of uneven solves share the same code.  All
// kernels are HBM-streaming stencils (about 0.5 flop/byte): no MFMA.
//
// Field pointers carry their address space: global (1) in the standalone
// kernels, LDS (3) inside the coarse tail.  Generic (flat) accesses would
// make every load wait for both the vector-memory and the LDS counters and
// serialise the loads of a line solve; the element routines are therefore
// templates over the pointer types and the kernels cast the level
// descriptors' pointers before use.  Chequer indices are 32-bit.
#include "amg.h"
#include "amg_internal.h"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <type_traits>

namespace amg {
namespace {

template <int AS, class T> using sp = __attribute__((address_space(AS))) T*;
constexpr int kG = 1;   // global memory
constexpr int kS = 3;   // LDS

template <class T> __device__ __forceinline__ sp<kG, T> gp(T* p) { return (sp<kG, T>)p; }
template <class T> __device__ __forceinline__ sp<kG, T> gfield(void* p) {
  return (sp<kG, T>)static_cast<T*>(p);
}
template <class T> __device__ __forceinline__ sp<kG, const T> gfield(const void* p) {
  return (sp<kG, const T>)static_cast<const T*>(p);
}

__device__ __forceinline__ int find_item(const int* prefix, int n, int b) {
  int lo = 0, hi = n - 1;
  while (lo < hi) {
    int mid = (lo + hi + 1) >> 1;
    if (prefix[mid] <= b) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Keeps values in scalar registers from here on.  The compiler loads a
// descriptor field where it is first used and waits for each: a kernel's
// start was a chain of up to ten dependent scalar loads.  Pinning the fields
// after reading them together leaves one round trip.
template <class A, class... V> __device__ __forceinline__ void pin_s(A& a, V&... v);
template <class A, class B, class C, class D, class E, class F, class G, class H, class... V>
__device__ __forceinline__ void pin_s8(A& a, B& b, C& c, D& d, E& e, F& f, G& g, H& h, V&... v) {
  asm("" : "+s"(a), "+s"(b), "+s"(c), "+s"(d), "+s"(e), "+s"(f), "+s"(g), "+s"(h));
  if constexpr (sizeof...(V) > 0) pin_s(v...);
}
template <class A, class... V> __device__ __forceinline__ void pin_s(A& a, V&... v) {
  if constexpr (sizeof...(V) >= 7) {
    pin_s8(a, v...);
  } else {
    asm("" : "+s"(a));
    if constexpr (sizeof...(V) > 0) pin_s(v...);
  }
}

// A kernel's list: the counts and the first item as scalar arguments, then the
// list itself.  Scalar arguments are preloaded into registers by the dispatch
// (kernarg preload), so a launch of one item (a single solve) starts with its
// level's address at hand: it used to read the list, the item, the stop word
// and then field after field, each from memory in turn, which small launches
// mostly consist of.  Back to back: 64^3 FP64 point half-sweep 3.24 -> 2.69
// us, 128^3 FP32 z-line 5.1 -> 4.8, 64^3 direct solve (three launches) 22.1
// -> 18.8; also the 256^3 sweep 19.5 -> 18.5.
#define LIST_PARAMS int ln, int lnb, int li0
#define LIST_ARGS(ll) (ll).nitems, (ll).nblocks, (ll).items[0]

__device__ __forceinline__ int xcd_swizzle(int b, int n);
// The item of this block and the block's number within it (blocks swizzled
// over the XCDs); b is the block's number in the launch.
struct Work {
  int t, idx, lb, b;
};
__device__ __forceinline__ Work work_item(LIST_PARAMS, const LaunchList& ll) {
  const int b = xcd_swizzle(blockIdx.x, lnb);
  if (ln == 1) return {0, li0, b, b};
  const int t = find_item(ll.prefix, ln, b);
  return {t, ll.items[t], b - ll.prefix[t], b};
}

// The head of a level's descriptor, read in one go.
__device__ __forceinline__ LevelHead level_head(const DevLevel& L) {
  LevelHead h = L;
  pin_s(h.nx, h.ny, h.nz, h.hx, h.stop, h.warm, h.skipc, h.pcur, h.gmhx, h.gmny, h.gshx, h.gsny, h.px,
        h.py, h.pz, h.ncell, h.u, h.f, h.u2, h.co64, h.co32, h.zt, h.vol, h.rho);
  return h;
}

// A gated cycle has stopped (DevLevel::stop): the kernel returns at once.
__device__ __forceinline__ bool level_off(const LevelHead& L) { return L.stop != 0; }

// Zero-guess flags of a smoothing launch (bit 0: the other colour is zero;
// bit 1: the own colour's old values are zero).  With kZgDyn, the finest
// level's first sweep of a mixed cycle, they hold only when the cycle does
// not continue the previous one's iterate (DevLevel::warm); kZgWarm marks
// the launch that does that sweep when the cycle continues it.
__device__ __forceinline__ int zero_flags(const LevelHead& L, int zero_guess) {
  if (zero_guess & kZgWarm) return 0;
  if (!(zero_guess & kZgDyn)) return zero_guess;
  return L.warm ? 0 : (zero_guess & 3);
}

// Blocks are dispatched round-robin over the 8 XCDs (each with its own L2);
// remap so that every XCD walks a contiguous range of tiles and neighbouring
// rows share an L2.  A bijection on [0, n).
__device__ __forceinline__ int xcd_swizzle(int b, int n) {
  const int q = n >> 3, rem = n & 7, x = b & 7, idx = b >> 3;
  return x * q + min(x, rem) + idx;
}

// Reciprocal for the line solves: the hardware rcp (1 ulp) in FP32, 1.0 / x in
// FP64: the hardware's 24-bit estimate, two Newton steps, which leave it within
// 1 ulp, and a third, which then rounds it correctly (Markstein's theorem); the
// fixup gives the special arguments what the division does.  It equals the
// division in all of 1e11 arguments tried, random ones and the 2^34 significands
// next to 1 and to 2 (two steps differ in 6 of the last), and in zeros,
// infinities, NaN, subnormal arguments and subnormal results.
//
// A z-line sweep has a chain of kZSeg of them per segment.  Half-sweeps with
// the division, with three steps, with two: 64^3 7.03, 6.87, 6.83 us, 128^3
// 10.0, 9.64, 9.50, 256^3 44.4, 43.3, 43.0.
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp(double x) {
  double r = __builtin_amdgcn_rcp(x);
#pragma unroll
  for (int q = 0; q < 3; ++q) r = __builtin_fma(r, __builtin_fma(-x, r, 1.0), r);
  return __builtin_amdgcn_div_fixup(r, x, 1.0);
}

// Fused multiply-add a*b + c, written out where several kernels have to
// round alike.
__device__ __forceinline__ float fm(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double fm(double a, double b, double c) { return __builtin_fma(a, b, c); }

// a / d in the point smoother: times the hardware reciprocal in FP32 (an
// IEEE division is about a dozen instructions), a division in FP64.
__device__ __forceinline__ float over(float a, float d) { return a * __builtin_amdgcn_rcpf(d); }
__device__ __forceinline__ double over(double a, double d) { return a / d; }

template <class T> __device__ __forceinline__ sp<kG, const T> coefs(const LevelHead& L);
template <> __device__ __forceinline__ sp<kG, const double> coefs<double>(const LevelHead& L) {
  return gp(L.co64);
}
template <> __device__ __forceinline__ sp<kG, const float> coefs<float>(const LevelHead& L) {
  return gp(L.co32);
}

// NaN-propagating maximum (fmax ignores NaN).
__device__ __forceinline__ double nmax(double a, double b) {
  return (a != a) ? a : ((b != b) ? b : fmax(a, b));
}

// max(acc, |x|) for accumulators of magnitudes (acc >= 0 or a NaN with the
// sign bit clear): the bit patterns of non-negative doubles order as their
// values, and a NaN orders above +inf, so one 64-bit integer maximum
// propagates NaN without a branch.
__device__ __forceinline__ double amax(double acc, double x) {
  const unsigned long long a = (unsigned long long)__double_as_longlong(acc);
  const unsigned long long b = (unsigned long long)__double_as_longlong(fabs(x));
  return __longlong_as_double((long long)(a > b ? a : b));
}

__device__ __forceinline__ double wave_max(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = nmax(v, __shfl_xor(v, off, 64));
  return v;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// Block-wide reduction of NV values; thread 0..NV-1 writes out[q].
template <int NV, bool SUM>
__device__ __forceinline__ void block_reduce_store(double (&v)[NV], double* __restrict__ out) {
  __shared__ double sm[NV][kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double x = SUM ? wave_sum(v[q]) : wave_max(v[q]);
    if (lane == 0) sm[q][w] = x;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double a = sm[threadIdx.x][0];
    for (int i = 1; i < (int)(blockDim.x >> 6); ++i)
      a = SUM ? a + sm[threadIdx.x][i] : nmax(a, sm[threadIdx.x][i]);
    out[threadIdx.x] = a;
  }
}

// Chequer-layout index of (m, j, k) in the half-row of colour c.
__device__ __forceinline__ int cidx(int m, int j, int k, int c, int hx, int ny) {
  return ((k * ny + j) * 2 + c) * hx + m;
}

// Seven chequer indices of cell (i,j,k): centre, x-, x+, y-, y+, z-, z+.
struct Nb {
  int c, xm, xp, ym, yp, zm, zp;
};

// The planes a cell of plane k is coupled to.  Past a wall the coupling is
// zero, but what it multiplies has to be finite: a plane in which the column's
// cell has the other colour, so that a half-sweep from zero reads what the
// half-sweep before it wrote.  nz - 1 and 0 are that for an even nz; for an
// odd one (walls on both sides) it is the plane next to the wall.
__device__ __forceinline__ int z_below(int k, int nz) {
  return k > 0 ? k - 1 : (nz & 1) ? min(1, nz - 1) : nz - 1;
}
__device__ __forceinline__ int z_above(int k, int nz) {
  return k < nz - 1 ? k + 1 : (nz & 1) ? max(nz - 2, 0) : 0;
}
__device__ __forceinline__ Nb neighbours(const LevelHead& L, int i, int j, int k) {
  const int hx = L.hx, ny = L.ny, nz = L.nz;
  const int col = (i + j) & 1, oth = col ^ 1, m = i >> 1, r = i & 1;
  int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
  int mr = m + r;     if (mr >= hx) mr = 0;
  const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
  const int km = z_below(k, nz), kp = z_above(k, nz);
  Nb n;
  n.c = cidx(m, j, k, col, hx, ny);
  const int ro = cidx(0, j, k, oth, hx, ny);
  n.xm = ro + ml;
  n.xp = ro + mr;
  n.ym = cidx(m, jm, k, oth, hx, ny);
  n.yp = cidx(m, jp, k, oth, hx, ny);
  n.zm = cidx(m, j, km, col, hx, ny);
  n.zp = cidx(m, j, kp, col, hx, ny);
  return n;
}

// Decode a chequer element index into (i, j, k).
// floor(n / d) by the invariant divisor of a level (DevLevel::gmhx/gshx,
// gmny/gsny: Granlund-Montgomery multiplier and shifts, exact for every
// 32-bit n).
__device__ __forceinline__ int gm_div(int n, unsigned m, int sh) {
  const unsigned un = (unsigned)n, t = __umulhi(m, un);
  return (int)((t + ((un - t) >> (sh & 0xff))) >> (sh >> 8));
}

__device__ __forceinline__ void decode(const LevelHead& L, int e, int& i, int& j, int& k) {
  const int t = gm_div(e, L.gmhx, L.gshx);
  const int m = e - t * L.hx;
  const int c = t & 1;
  const int row = t >> 1;
  k = gm_div(row, L.gmny, L.gsny);
  j = row - k * L.ny;
  i = 2 * m + ((c + j) & 1);
}

// Off-diagonal stencil sum, in a fixed order: x-, x+, y-, y+, z-, z+.
template <class T, class CP>
__device__ __forceinline__ T offsum(CP co, const LevelHead& L, int i, int j, int k, T uxm, T uxp,
                                    T uym, T uyp, T uzm, T uzp) {
  const int nx = L.nx, ny = L.ny;
  const auto cy = co + 3 * nx;
  const auto cz = cy + 3 * ny;
  T s = co[i] * uxm + co[nx + i] * uxp;
  s += cy[j] * uym;
  s += cy[ny + j] * uyp;
  s += cz[k] * uzm;
  s += cz[L.nz + k] * uzp;
  return s;
}

template <class T, class CP>
__device__ __forceinline__ T diag_at(CP co, const LevelHead& L, int i, int j, int k) {
  const int nx = L.nx, ny = L.ny;
  const auto cy = co + 3 * nx;
  const auto cz = cy + 3 * ny;
  return (cz[2 * L.nz + k] + cy[2 * ny + j]) + co[2 * nx + i];
}

// ---------------------------------------------------------------------------
// Point red-black Gauss-Seidel half-sweep (mgMK/mg_relax.F90:146-168):
// u = (f - sum w_n u_n)/diag on the cells with (i+j+k)&1 == parity.  Element
// e enumerates the cells of the colour; in plane k the colour is column
// colour (parity+k)&1, so consecutive e are one contiguous half-row.
template <class T, class UP, class FP, class CP>
__device__ __forceinline__ void rb_point_mjk(const LevelHead& L, UP u, FP f, CP co, int m, int j,
                                             int k, int parity, int zero_guess) {
  const int c = (k + parity) & 1;
  const int i = 2 * m + ((c + j) & 1);
  const Nb n = neighbours(L, i, j, k);
  const T d = diag_at<T>(co, L, i, j, k);
  T val;
  if (zero_guess & 1) {
    val = over(f[n.c], d);
  } else {
    const T s = offsum<T>(co, L, i, j, k, u[n.xm], u[n.xp], u[n.ym], u[n.yp], u[n.zm], u[n.zp]);
    val = over(f[n.c] - s, d);
  }
  u[n.c] = val;
}

template <class T, class UP, class FP, class CP>
__device__ __forceinline__ void rb_point_elem(const LevelHead& L, UP u, FP f, CP co, int e,
                                              int parity, int zero_guess) {
  const int row = gm_div(e, L.gmhx, L.gshx), m = e - row * L.hx;
  const int k = gm_div(row, L.gmny, L.gsny), j = row - k * L.ny;
  rb_point_mjk<T>(L, u, f, co, m, j, k, parity, zero_guess);
}

// The same with the element index decoded by multiply-high reciprocals
// (DevLevel::mhx, mny), exact for the small levels of the coarse tail.
__device__ __forceinline__ int fast_div(int e, unsigned mag) {
  return mag ? (int)__umulhi((unsigned)e, mag) : e;
}
template <class T, class UP, class FP, class CP>
__device__ __forceinline__ void rb_point_small(const DevLevel& L, UP u, FP f, CP co, int e,
                                               int parity, int zero_guess) {
  const int row = fast_div(e, L.mhx), m = e - row * L.hx;
  const int k = fast_div(row, L.mny), j = row - k * L.ny;
  rb_point_mjk<T>(L, u, f, co, m, j, k, parity, zero_guess);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_rb_point(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                     int parity, int zero_guess, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const LevelHead L = level_head(Lt[wk.idx]);
  if (level_off(L)) return;
  const int e = wk.lb * kBlock + threadIdx.x;
  if (e < L.hx * L.ny * L.nz)
    rb_point_elem<T>(L, gfield<T>(L.u), gfield<const T>((const void*)L.f), coefs<T>(L), e, parity,
                     zero_flags(L, zero_guess));
}

// The same half-sweep marching in z (large levels): a thread owns position
// (m, j) of a plane, both halves, and K consecutive planes.  In plane k the
// colour's cells are in half h = (parity + k) & 1, so the thread updates one
// cell per plane, i = 2m + ((h + j) & 1).  Its z-neighbours are the same
// half of the planes k-1 and k+1 (the other colour), so the one above plane
// k is the one below plane k+2 and is loaded once.  Every load of the slab
// (the other colour only, which the sweep does not write) is issued before
// the first store, the coefficients of the thread's two columns and row once
// per thread, those of z (wave-uniform) from the scalar cache.  The update is
// rb_point_mjk's, in its order.
template <class T, int K>
__global__ __launch_bounds__(kBlock) void k_rb_march(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                     int parity, int zero_guess, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const LevelHead L = level_head(Lt[wk.idx]);
  if (level_off(L)) return;
  const int zg = zero_flags(L, zero_guess);
  const int hx = L.hx, ny = L.ny, nz = L.nz, nx = L.nx;
  const int npos = hx * ny, ncb = (npos + kBlock - 1) / kBlock;
  const int lb = wk.lb;
  const int bk = lb / ncb, pos = (lb - bk * ncb) * kBlock + threadIdx.x;
  if (pos >= npos) return;
  const int j = gm_div(pos, L.gmhx, L.gshx), m = pos - j * hx;
  const int k0 = bk * K;
  const sp<kG, const T> co = coefs<T>(L);
  const sp<kG, const T> cy = co + 3 * nx;
  const sp<kG, const T> cz = cy + 3 * ny;
  const auto u = gfield<T>(L.u);
  const auto f = gfield<const T>((const void*)L.f);
  // the thread's two columns (half h: i = 2m + ((h + j) & 1))
  int ml[2], mr[2];
  T wxl[2], wxr[2], dxx[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int i = 2 * m + ((h + j) & 1), r = i & 1;
    ml[h] = m - 1 + r; if (ml[h] < 0) ml[h] = hx - 1;
    mr[h] = m + r;     if (mr[h] >= hx) mr[h] = 0;
    wxl[h] = co[i];
    wxr[h] = co[nx + i];
    dxx[h] = co[2 * nx + i];
  }
  const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
  const T wys = cy[j], wyn = cy[ny + j], dyy = cy[2 * ny + j];
  const bool nbr = !(zg & 1);
  // plane k of half h, row jj: index of position mm
  auto at = [&](int k, int h, int jj, int mm) { return ((k * ny + jj) * 2 + h) * hx + mm; };
  T fv[K], xl[K], xr[K], ys[K], yn[K], zp[K], zm01[2];
#pragma unroll
  for (int s = 0; s < K; ++s) {
    const int k = min(k0 + s, nz - 1);              // a short last slab re-reads its last plane
    const int h = (parity + k0 + s) & 1, o = h ^ 1;
    fv[s] = f[at(k, h, j, m)];
    if (nbr) {
      xl[s] = u[at(k, o, j, ml[h])];
      xr[s] = u[at(k, o, j, mr[h])];
      ys[s] = u[at(k, o, jm, m)];
      yn[s] = u[at(k, o, jp, m)];
      zp[s] = u[at(z_above(k, nz), h, j, m)];
    }
  }
  if (nbr) {
    // below the slab's first two planes
    const int h0 = (parity + k0) & 1;
    zm01[0] = u[at(z_below(k0, nz), h0, j, m)];
    zm01[1] = u[at(k0, h0 ^ 1, j, m)];
  }
#pragma unroll
  for (int s = 0; s < K; ++s) {
    const int k = k0 + s;
    if (k >= nz) break;
    const int h = (parity + k) & 1;
    const T d = (cz[2 * nz + k] + dyy) + dxx[h];
    T val;
    if (!nbr) {
      val = over(fv[s], d);
    } else {
      const T zmv = s < 2 ? zm01[s] : zp[s - 2];
      T a = wxl[h] * xl[s] + wxr[h] * xr[s];
      a += wys * ys[s];
      a += wyn * yn[s];
      a += cz[k] * zmv;
      a += cz[nz + k] * zp[s];
      val = over(fv[s] - a, d);
    }
    u[at(k, h, j, m)] = val;
  }
}

// Both half-sweeps of a point sweep in one launch.  A workgroup takes kPairY
// rows by TZ planes of whole x rows: it updates their red cells and those of
// the rows and planes around them (whose owners do the same sums) into LDS,
// then its black cells from there.  Other workgroups still read the old black
// values, so the new ones go to another buffer: `back` 0 reads them from u and
// writes w, 1 the other way; a level's sweeps run in such pairs.  Red cells
// are written to u, and no workgroup reads them from memory.
//
// Small levels are bound by launches: a half-sweep of 64^3 in FP64 takes 2.4
// us and the gap to the next 1, a whole sweep here 4.1 (solve 4500 -> 4100
// us).  Larger ones are bound by the cache's traffic: b once and u read and
// written once, for half of u four times and b once: at 256x64x256 in FP32
// 17.2 -> 13.0 us.
//
// Thread (m, row) owns a position of row j0 - 1 + row, both halves, and
// marches in z as k_rb_march does, so a red cell costs six loads and no z
// coefficient (a thread per cell with all of its own loads took 4.4 us at
// 64^3, 24 at 256x64x256).  kPairY 2, 6, 8 and TZ 8 were slower on both (64^3:
// 4370, 4235, 4450 us and, spilling, 6490).
template <class T, int TZ>
__global__ __launch_bounds__(1024) void k_rb_pair(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                  int zero_guess, int back, LaunchList ll) {
  constexpr int TY = kPairY;
  extern __shared__ unsigned char lds_raw[];
  const sp<kS, T> red = (sp<kS, T>)(sp<kS, unsigned char>)lds_raw;
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevLevel& D = Lt[wk.idx];
  void *w0 = D.w[0], *w1 = D.w[1];
  pin_s(w0, w1);
  const LevelHead L = level_head(D);
  if (level_off(L)) return;
  void* const wp = L.pcur ? w1 : w0;
  const bool nbr = !(zero_flags(L, zero_guess) & 1);
  const int hx = L.hx, ny = L.ny, nz = L.nz, nx = L.nx;
  const int nty = (ny + TY - 1) / TY;
  const int bz = wk.lb / nty, j0 = (wk.lb - bz * nty) * TY, k0 = bz * TZ;
  const int row = gm_div(threadIdx.x, L.gmhx, L.gshx), m = threadIdx.x - row * hx, dy = row - 1;
  const bool act = row < TY + 2;
  auto wrap = [](int a, int n) { return a < 0 ? a + n : a >= n ? a - n : a; };
  const int j = act ? wrap(j0 + dy, ny) : 0, jm = wrap(j - 1, ny), jp = wrap(j + 1, ny);
  const bool own = act && dy >= 0 && dy < TY && j0 + dy < ny;
  const sp<kG, const T> co = coefs<T>(L);
  const sp<kG, const T> cy = co + 3 * nx;
  const sp<kG, const T> cz = cy + 3 * ny;
  const auto u = gfield<T>(L.u);
  const auto f = gfield<const T>((const void*)L.f);
  const sp<kG, const T> ub = gfield<const T>((const void*)(back ? wp : L.u));
  const sp<kG, T> wb = gfield<T>(back ? L.u : wp);
  // the thread's two columns, of half h: i = 2m + b with b = (h + j) & 1
  const int b0 = j & 1, b1 = b0 ^ 1;
  const int mm = m == 0 ? hx - 1 : m - 1, mp = m == hx - 1 ? 0 : m + 1;
  const int ml[2] = {b0 ? m : mm, b0 ? mm : m}, mr[2] = {b0 ? mp : m, b0 ? m : mp};
  const T wxl[2] = {co[2 * m + b0], co[2 * m + b1]}, wxr[2] = {co[nx + 2 * m + b0], co[nx + 2 * m + b1]};
  const T dxx[2] = {co[2 * nx + 2 * m + b0], co[2 * nx + 2 * m + b1]};
  const T wys = cy[j], wyn = cy[ny + j], dyy = cy[2 * ny + j];
  auto at = [&](int k, int h, int jj, int q) { return ((k * ny + jj) * 2 + h) * hx + q; };
  // red plane s of the march is plane k0 - 1 + s = pk[s + 1], black plane s
  // k0 + s; the half of a plane is its number's (k0 is even).  Planes outside
  // are wrapped, or with an odd nz (walls) mirrored: of the same half either
  // way, as z_below.
  constexpr int NR = TZ + 2;
  int pk[NR + 2];
#pragma unroll
  for (int t = 0; t < NR + 2; ++t) pk[t] = k0 - 2 + t;
  if (k0 == 0 || k0 + TZ + 1 >= nz) {
    const bool odd = nz & 1;
#pragma unroll
    for (int t = 0; t < NR + 2; ++t) {
      const int k = pk[t], lo = odd ? -k : k + nz, hi = odd ? max(2 * (nz - 1) - k, 0) : k - nz;
      pk[t] = k < 0 ? lo : k < nz ? k : hi;
    }
  }
  auto value = [&](int h, T fv, T zm_, T zp_, T zd, T xl, T xr, T ys, T yn, T zm, T zp) {
    const T d = (zd + dyy) + dxx[h];
    T a = wxl[h] * xl + wxr[h] * xr;
    a += wys * ys;
    a += wyn * yn;
    a += zm_ * zm;
    a += zp_ * zp;
    return over(fv - a, d);
  };
  T wzm[NR], wzp[NR], dzz[NR];
  T fv[NR], xl[NR], xr[NR], ys[NR], yn[NR], zc[NR + 2], fb[TZ];
  auto hr = [](int s) { return (s + 1) & 1; };   // half of red plane s
#pragma unroll
  for (int s = 0; s < NR; ++s) {
    const int k = pk[s + 1];
    wzm[s] = cz[k];
    wzp[s] = cz[nz + k];
    dzz[s] = cz[2 * nz + k];
  }
  if (act) {
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const int k = pk[s + 1], h = hr(s);
      fv[s] = f[at(k, h, j, m)];
      if (nbr) {
        xl[s] = ub[at(k, h ^ 1, j, ml[h])];
        xr[s] = ub[at(k, h ^ 1, j, mr[h])];
        ys[s] = ub[at(k, h ^ 1, jm, m)];
        yn[s] = ub[at(k, h ^ 1, jp, m)];
        zc[s + 2] = ub[at(pk[s + 2], h, j, m)];
      }
    }
    if (nbr) {
      zc[0] = ub[at(pk[0], hr(0), j, m)];
      zc[1] = ub[at(pk[1], hr(1), j, m)];
    }
    if (own) {
#pragma unroll
      for (int s = 0; s < TZ; ++s) fb[s] = f[at(min(k0 + s, nz - 1), (s + 1) & 1, j, m)];
    }
#pragma unroll
    for (int s = 0; s < NR; ++s) {
      const int h = hr(s);
      const T v = nbr ? value(h, fv[s], wzm[s], wzp[s], dzz[s], xl[s], xr[s], ys[s], yn[s], zc[s], zc[s + 2])
                      : over(fv[s], (dzz[s] + dyy) + dxx[h]);
      red[(s * (TY + 2) + row) * hx + m] = v;
      fv[s] = v;
    }
  }
  __syncthreads();
  if (!own) return;
  // the red cells are stored here: a barrier waits for stores
#pragma unroll
  for (int s = 0; s < TZ; ++s)
    if (k0 + s < nz) u[at(k0 + s, s & 1, j, m)] = fv[s + 1];
  auto rd = [&](int s, int r, int q) { return red[(s * (TY + 2) + r) * hx + q]; };
#pragma unroll
  for (int s = 0; s < TZ; ++s) {
    if (k0 + s >= nz) break;
    const int h = (s + 1) & 1;
    wb[at(k0 + s, h, j, m)] =
        value(h, fb[s], wzm[s + 1], wzp[s + 1], dzz[s + 1], rd(s + 1, row, ml[h]), rd(s + 1, row, mr[h]),
              rd(s + 1, row - 1, m), rd(s + 1, row + 1, m), rd(s, row, m), rd(s + 2, row, m));
  }
}

// ---------------------------------------------------------------------------
// z-line red-black Gauss-Seidel half-sweep (mgMK/mg_relax.F90:423-600, LJ):
// the columns (i,j) of one colour ((i+j)&1 == parity) solve their
// tridiagonal z-system with the other colour's current values on the
// right-hand side.  A workgroup takes 64 columns (one per lane) and splits
// each column into P segments of S cells (wave p owns segment p).  Every
// segment eliminates its rows once, forward, for three right-hand sides:
// its data, and unit couplings to the last value of the segment below and
// to the first value of the segment above.  Its end values are then linear
// in those two unknowns; the 2P interface unknowns are solved by parallel
// cyclic reduction in LDS, and one back substitution per segment gives its
// values.  The result equals a Thomas solve of the whole column up to
// rounding.  Periodic z: the wrap couplings are lagged (the other end's old
// value on the right-hand side), in the order of the oracle's restatement.
// A row's coupling past either end of the column (a wrap or a wall ghost)
// only ever multiplies an interface value that does not exist, which the
// reduction takes as zero, so the rows are used as the tables hold them.

// Row access at a uniform row base plus a per-lane 32-bit byte offset: the
// global load/store form with a 64-bit scalar base and a 32-bit vector
// offset, so a row's address costs no vector arithmetic.
template <class T> __device__ __forceinline__ T ld_row(sp<kG, const T> row, unsigned boff) {
  return *(sp<kG, const T>)((sp<kG, const char>)row + boff);
}
template <class T> __device__ __forceinline__ void st_row(sp<kG, T> row, unsigned boff, T v) {
  *(sp<kG, T>)((sp<kG, char>)row + boff) = v;
}
// The same, non-temporal: for data that is not read again before it would
// have left the L2 (the streaming stages of the mixed outer step).
template <class T> __device__ __forceinline__ void st_row_nt(sp<kG, T> row, unsigned boff, T v) {
  __builtin_nontemporal_store(v, (T*)(sp<kG, T>)((sp<kG, char>)row + boff));
}
template <class T> __device__ __forceinline__ T ld_row_nt(sp<kG, const T> row, unsigned boff) {
  return __builtin_nontemporal_load((const T*)(sp<kG, const T>)((sp<kG, const char>)row + boff));
}

// The four in-plane neighbours' part of a row's stencil sum.
template <class T>
__device__ __forceinline__ T zline_nbr(T wxl, T wxr, T wys, T wyn, T xl, T xr, T ys, T yn) {
  return fm(wyn, yn, fm(wys, ys, fm(wxr, xr, wxl * xl)));
}

// NBR false: the other colour is zero (zero_guess bit 0, the first
// half-sweep from u = 0) and is not read.  LEAN: the register-lean form of
// the segment elimination (below).  H: a wave holds two segments of 32
// columns (lanes 0-31 segment 2w, lanes 32-63 segment 2w+1), so a workgroup
// has half the waves; p and lane (the column within the workgroup's 32) are
// then per lane, and the z rows are staged in LDS.  Every lane does the same
// operations in either shape.
template <class T, int S, int C, bool NBR, bool LEAN, bool H>
__device__ __forceinline__ void zline_group(const LevelHead& L, int parity, int zero_guess, int col0,
                                            int p, int lane, int P, T* __restrict__ lds, bool act) {
  const int hx = L.hx, ny = L.ny, nz = L.nz, nx = L.nx;
  const int ncol = hx * ny;
  const bool live = act && col0 < ncol;
  const int col = live ? col0 : ncol - 1;
  const int j = gm_div(col, L.gmhx, L.gshx), m = col - j * hx;
  const int c = parity, oth = parity ^ 1;
  const int i = 2 * m + ((c + j) & 1), r = i & 1;
  int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
  int mr = m + r;     if (mr >= hx) mr = 0;
  const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
  const sp<kG, const T> co = coefs<T>(L);
  const sp<kG, const T> cy = co + 3 * nx;
  const sp<kG, const T> cz = cy + 3 * ny;
  const T wxl = co[i], wxr = co[nx + i], wys = cy[j], wyn = cy[ny + j];
  const T dxy = co[2 * nx + i] + cy[2 * ny + j];
  const sp<kG, T> u = gfield<T>(L.u);
  const sp<kG, const T> f = gfield<const T>((const void*)L.f);
  const int plane = ny * 2 * hx;
  // byte offsets within a plane (the same in every row)
  constexpr unsigned W = sizeof(T);
  const unsigned bown = (unsigned)cidx(m, j, 0, c, hx, ny) * W;
  const unsigned xo = (unsigned)cidx(0, j, 0, oth, hx, ny);
  const unsigned bxl = (xo + ml) * W, bxr = (xo + mr) * W;
  const unsigned bso = (unsigned)cidx(m, jm, 0, oth, hx, ny) * W;
  const unsigned bno = (unsigned)cidx(m, jp, 0, oth, hx, ny) * W;
  const bool pz = L.pz != 0;
  const int Pi = (nz + S - 1) / S;            // segments of this item (<= blockDim.y)
  const int ks = p * S;
  const int len = max(0, min(S, nz - ks));    // 0 for spare waves of a shorter item
  // A (sub-diagonal), E (super-diagonal) and the z part of the diagonal
  // depend on k only and p is wave-uniform, so they are scalar values
  // (uniform loads issued with the rest, read without memory latency in the
  // serial elimination chain); the lane's x/y diagonal share dxy is added
  // at use.  All loads -- these rows, the lagged wrap values and the
  // right-hand-side data -- are unconditional (every address is in bounds,
  // uses are selected) and issued before the first wait: a sweep pays one
  // memory round trip.
  // FP64 rows do not fit in scalar registers, and with H a wave's two
  // segments have different rows: they are staged in LDS by lanes 0..S-1
  // (of each half) and read back as broadcasts (LDS_COEF).
  constexpr bool LDS_COEF = sizeof(T) == 8 || H;
  constexpr int CW = H ? 32 : 64;             // columns of a workgroup
  constexpr int SR = LDS_COEF ? 1 : S;
  T A[SR], E[SR], Dz[SR];
  T* const cA = lds + (sizeof(T) == 8 ? 6 : 12) * P * CW + p * 3 * S;
  T* const cE = cA + S;
  T* const cD = cE + S;
  T za = T(0), ze = T(0), zd = T(0);
  if constexpr (LDS_COEF) {
    const int kq = min(ks + (lane & (S - 1)), nz - 1);
    za = cz[kq];
    ze = cz[nz + kq];
    zd = cz[2 * nz + kq];
  } else {
    // rows kc..kc+S-1 from one base (three 16-word scalar loads); the tables
    // end with kZSeg spare words, so a ragged or spare segment stays in bounds
    const sp<kG, const T> cr = cz + min(ks, nz - 1);
#pragma unroll
    for (int q = 0; q < S; ++q) {
      A[q] = cr[q];
      E[q] = cr[nz + q];
      Dz[q] = cr[2 * nz + q];
    }
  }
  // zero_guess bit 1: this colour's old values are zero (no lagged wrap)
  const bool lag = pz && !(zero_guess & 2);
  const T cz_first = cz[0], cz_last = cz[2 * nz - 1];
  const T ubot = ld_row<T>(u + (nz - 1) * plane, bown), utop = ld_row<T>(u, bown);
  const T lagb = (lag && p == 0) ? cz_first * ubot : T(0);
  const T lagt = (lag && ks + len == nz) ? cz_last * utop : T(0);
  T g[S];
#pragma unroll
  for (int q0 = 0; q0 < S; q0 += C) {
    // keep this chunk's loads behind the previous chunk's arithmetic
    if (q0 > 0) __builtin_amdgcn_sched_barrier(0);
    T fv[C], xl[C], xr[C], ys[C], yn[C];
#pragma unroll
    for (int qq = 0; qq < C; ++qq) {
      const int kb = min(ks + q0 + qq, nz - 1) * plane;   // rows clamped: in bounds
      fv[qq] = ld_row<T>(f + kb, bown);
      if constexpr (NBR) {
        const sp<kG, const T> ur = u + kb;
        xl[qq] = ld_row<T>(ur, bxl);
        xr[qq] = ld_row<T>(ur, bxr);
        ys[qq] = ld_row<T>(ur, bso);
        yn[qq] = ld_row<T>(ur, bno);
      }
    }
    if (LDS_COEF && q0 == 0) {
      if (lane < S) {
        cA[lane] = za;
        cE[lane] = ze;
        cD[lane] = zd;
      }
      __syncthreads();
    }
#pragma unroll
    for (int qq = 0; qq < C; ++qq) {
      if constexpr (NBR) {
        g[q0 + qq] = fv[qq] - zline_nbr(wxl, wxr, wys, wyn, xl[qq], xr[qq], ys[qq], yn[qq]);
      } else {
        g[q0 + qq] = fv[qq];
      }
    }
  }
  g[0] -= lagb;                                            // row 0 of the column (p == 0)
#define A(q) (LDS_COEF ? cA[q] : A[LDS_COEF ? 0 : (q)])
#define E(q) (LDS_COEF ? cE[q] : E[LDS_COEF ? 0 : (q)])
#define D(q) ((LDS_COEF ? cD[q] : Dz[LDS_COEF ? 0 : (q)]) + dxy)
  const T a_first = A(0);                                  // coupling to u_{ks-1}
  // phase 1: forward elimination of the segment's rows for the data (g, in
  // place), the coupling a_first to u_{ks-1} entering row 0 (v) and the
  // coupling E(len-1) to u_{ks+len} entering the last row (w).  The first
  // values of the three solutions accumulate during the pass,
  // x_0 = sum_q pi_q x'_q with pi_q = prod_{i<q} (-E(i) rd_i); the last
  // values are the last row's.
  // Short form: the eliminated v (vv) and super-diagonal (cp) are stored.
  // LEAN form (two values per row instead of three, so a 1024-lane block
  // fits in 64 registers and two blocks share a CU): only the pivot
  // reciprocals rd are stored, and v and cp are recomputed from them with
  // the same operations.  Both forms round alike, so every launch gives the
  // same values whichever form it takes.
  // A full segment (n == S, every segment but the last of a ragged column)
  // instantiates the passes with a constant n, so the unrolled chains carry
  // no branches.
  constexpr int SS = LEAN ? 1 : S, SL = LEAN ? S : 1;
  T vv[SS], cp[SS], rdv[SL];
  T y0 = T(0), yl = T(0), v0 = T(0), vl = T(0), w0 = T(0), wl = T(0);
  auto factor = [&](const int len) {
    T cq = T(0), y = T(0), v = T(0), pi = T(1);
#pragma unroll
    for (int q = 0; q < S; ++q) {
      if (q < len) {
        if (q == len - 1) g[q] -= lagt;                    // row nz-1 (last segment)
        const T a = (q == 0) ? T(0) : A(q);
        const T rd = rcp(fm(-a, cq, D(q)));
        y = fm(-a, y, g[q]) * rd;
        v = (q == 0) ? a_first * rd : -(a * rd) * v;
        cq = E(q) * rd;
        g[q] = y;
        if (q == 0) { y0 = y; v0 = v; }
        else { y0 = fm(pi, y, y0); v0 = fm(pi, v, v0); }
        if (q == len - 1) { yl = y; vl = v; wl = cq; w0 = pi * cq; }
        else pi = (q == 0) ? -cq : pi * -cq;
        if constexpr (LEAN) {
          rdv[q] = rd;
        } else {
          vv[q] = v;
          cp[q] = cq;
        }
      }
    }
  };
  if (sizeof(T) == 4 && len == S) factor(S);
  else if (len > 0) factor(len);
  // phase 2: reduced system X_p = (t_p, b_p) (first/last values of segment p)
  //   t_p + v0_p b_{p-1} + w0_p t_{p+1} = y0_p
  //   b_p + vl_p b_{p-1} + wl_p t_{p+1} = yl_p
  // with (y, v, w) the segment's solutions for the three right-hand sides,
  // taken at its first and last rows.  Parallel cyclic reduction over the
  // segments: at distance d every segment substitutes b_{p-d} (row b of
  // p-d) and t_{p+d} (row t of p+d); the couplings keep their shape (to
  // b_{p-2d} and t_{p+2d} only), so after ceil(log2 P) steps every segment
  // holds its own values.  Segments past either end of the column
  // contribute zeros.  Every wave takes part.
  // FP32 double-buffers the state in LDS (one barrier per step); FP64 uses
  // one buffer and two barriers, keeping the block within 64 KiB of LDS.
  const int sl = p * CW + lane;
  T bprev = T(0), tnext = T(0);
  constexpr int kZBuf = sizeof(T) == 8 ? 1 : 2;
  if (Pi > 1) {
    const int PS = P * CW;
    T at = v0, ab = vl, ct = w0, cb = wl, rt = y0, rb = yl;
    int buf = 0;
    for (int d = 1; d < Pi; d <<= 1, buf ^= (kZBuf - 1)) {
      T* W = lds + buf * 6 * PS;
      W[sl] = at; W[PS + sl] = ab; W[2 * PS + sl] = ct;
      W[3 * PS + sl] = cb; W[4 * PS + sl] = rt; W[5 * PS + sl] = rb;
      __syncthreads();
      const bool hm = p - d >= 0, hp = p + d < Pi;
      const int sm = hm ? (p - d) * CW + lane : sl, spp = hp ? (p + d) * CW + lane : sl;
      // row b of segment p-d, row t of segment p+d
      const T abm = W[PS + sm], cbm = W[3 * PS + sm], rbm = W[5 * PS + sm];
      const T atp = W[spp], ctp = W[2 * PS + spp], rtp = W[4 * PS + spp];
      const T ab_m = hm ? abm : T(0), cb_m = hm ? cbm : T(0), rb_m = hm ? rbm : T(0);
      const T at_p = hp ? atp : T(0), ct_p = hp ? ctp : T(0), rt_p = hp ? rtp : T(0);
      if (kZBuf == 1) __syncthreads();   // every read done before the next writes
      const T m11 = fm(-at, cb_m, T(1)), m12 = -ct * at_p;
      const T m21 = -ab * cb_m, m22 = fm(-cb, at_p, T(1));
      const T id = rcp(fm(m11, m22, -(m12 * m21)));
      const T qt = fm(-ct, rt_p, fm(-at, rb_m, rt)), qb = fm(-cb, rt_p, fm(-ab, rb_m, rb));
      const T lt = -at * ab_m, lb = -ab * ab_m;     // couplings to b_{p-2d}
      const T ut = -ct * ct_p, ub = -cb * ct_p;     // couplings to t_{p+2d}
      at = id * fm(m22, lt, -(m12 * lb));
      ab = id * fm(m11, lb, -(m21 * lt));
      ct = id * fm(m22, ut, -(m12 * ub));
      cb = id * fm(m11, ub, -(m21 * ut));
      rt = id * fm(m22, qt, -(m12 * qb));
      rb = id * fm(m11, qb, -(m21 * qt));
    }
    T* W = lds + buf * 6 * PS;
    W[sl] = rt;
    W[PS + sl] = rb;
    __syncthreads();
    bprev = (p > 0) ? W[PS + (p - 1) * CW + lane] : T(0);
    tnext = (p < Pi - 1) ? W[(p + 1) * CW + lane] : T(0);
    __syncthreads();   // the group's LDS may be rewritten by its next call
  }
  // phase 3: back substitution of g - v bprev - w tnext (LEAN: v is
  // recomputed from rd by the forward pass's own operations first)
  auto backsub = [&](const int len) {
    if constexpr (LEAN) {
      if (p > 0) {
        T v = T(0);
#pragma unroll
        for (int q = 0; q < S; ++q) {
          if (q < len) {
            v = (q == 0) ? a_first * rdv[q] : -(A(q) * rdv[q]) * v;
            g[q] = fm(-v, bprev, g[q]);
          }
        }
      }
    }
    T x = T(0);
#pragma unroll
    for (int q = S - 1; q >= 0; --q) {
      if (q < len) {
        if constexpr (LEAN) {
          const T cq = E(q) * rdv[q];
          x = fm(-cq, (q == len - 1) ? tnext : x, g[q]);
        } else {
          const T gq = fm(-vv[q], bprev, g[q]);
          x = fm(-cp[q], (q == len - 1) ? tnext : x, gq);
        }
        if (live) st_row<T>(u + (ks + q) * plane, bown, x);
      }
    }
  };
  if (sizeof(T) == 4 && len == S) backsub(S);
  else if (len > 0) backsub(len);
#undef A
#undef E
#undef D
}

// The LEAN FP32 form is built for 8 waves per SIMD (64 registers), so two
// 1024-lane blocks share a CU and one's loads overlap the other's solve; the
// LEAN FP64 form needs 128 registers and gets the same overlap from H, whose
// workgroups have 8 waves.  H without LEAN is for launches of few column
// groups: a CU holds one workgroup, which may use up to 256 registers.
template <class T, int S, int C, bool NBR, bool LEAN, bool H>
__global__ __launch_bounds__(H ? 512 : 1024, LEAN ? 32 / (int)sizeof(T) : (H ? 2 : 4)) void k_zline(
    const DevLevel* __restrict__ Lt, LIST_PARAMS, int parity, int zero_guess, LaunchList ll) {
  extern __shared__ unsigned char lds_raw[];
  const Work wk = work_item(ln, lnb, li0, ll);
  const LevelHead L = level_head(Lt[wk.idx]);
  if (level_off(L)) return;
  // the first sweep of a mixed cycle's finest level runs as two launches,
  // from zero (NBR false) and continuing the iterate (kZgWarm): one returns
  if (!NBR && (zero_guess & kZgDyn) && L.warm) return;
  if ((zero_guess & kZgWarm) && !L.warm) return;
  // threadIdx.y is constant across a wave (blockDim.x == 64): say so to the compiler
  const int seg = __builtin_amdgcn_readfirstlane(threadIdx.y);
  if constexpr (H) {
    const int cl = threadIdx.x & 31;
    zline_group<T, S, C, NBR, LEAN, true>(L, parity, zero_flags(L, zero_guess),
                                          wk.lb * 32 + cl, 2 * seg + (threadIdx.x >> 5),
                                          cl, 2 * blockDim.y, reinterpret_cast<T*>(lds_raw), true);
  } else {
    zline_group<T, S, C, NBR, LEAN, false>(L, parity, zero_flags(L, zero_guess),
                                           wk.lb * 64 + threadIdx.x, seg, threadIdx.x,
                                           blockDim.y, reinterpret_cast<T*>(lds_raw), true);
  }
}

// ---------------------------------------------------------------------------
// The FP32 half-sweep of a level whose columns all have the same x/y diagonal
// share (both horizontal axes uniform, periodic or with Dirichlet walls): every
// column then has the same matrix, so the pivots, the segments' coupling solutions and
// the whole cyclic reduction of the interface matrix are the same numbers in
// every column.  They are computed once, when the level is built
// (k_zline_table), with the operations of zline_group, and the sweep keeps
// only the right-hand side's own arithmetic: the results are those of
// zline_group bit for bit.
//
// Table (DevLevel::zt): one record of kZRec words per segment,
//   [0, 32)    A | RD, kZSeg words each: the sub-diagonal within the segment
//              (0 in its first row) and the pivot's reciprocal
//   [64, 112)  V | CQ | PI: the coupling solution v, the eliminated
//              super-diagonal and the weight of the row's y in the segment's
//              first value
//   [128, 164) kZStep words per reduction step: at ab ct cb m11 m12 m21 m22 id.
// Rows past nz are zero: they leave the carried values zero; so is the record
// past an odd count of segments (the half-wave form's spare segment).
constexpr int kZRec = 192, kZRecBack = 64, kZRecStep = 128, kZStep = 9;

// One thread per segment.
__global__ __launch_bounds__(64) void k_zline_table(const float* __restrict__ co, int nx, int ny, int nz,
                                                    float* __restrict__ zt) {
  __shared__ float st[4][64];
  constexpr int S = kZSeg;
  const int P = (nz + S - 1) / S, p = threadIdx.x;
  const bool on = p < P;
  for (int e = p; e < kZRec * ((P + 1) & ~1); e += 64) zt[e] = 0.0f;
  __syncthreads();
  const float* cz = co + 3 * nx + 3 * ny;
  const float dxy = co[2 * nx] + co[3 * nx + 2 * ny];
  const int ks = p * S, len = on ? min(S, nz - ks) : 0;
  float* z = zt + p * kZRec;
  float v0 = 0.0f, vl = 0.0f, w0 = 0.0f, wl = 0.0f;
  float cq = 0.0f, v = 0.0f, pi = 1.0f;
  if (on) {
    const float a_first = cz[ks];
    for (int q = 0; q < S; ++q) {
      float a = 0.0f, rd = 0.0f, pw = 0.0f, vq = 0.0f, cw = 0.0f;
      if (q < len) {
        const int k = ks + q;
        a = (q == 0) ? 0.0f : cz[k];
        rd = rcp(fm(-a, cq, cz[2 * nz + k] + dxy));
        v = (q == 0) ? a_first * rd : -(a * rd) * v;
        cq = cz[nz + k] * rd;
        if (q == 0) v0 = v;
        else v0 = fm(pi, v, v0);
        pw = pi;
        vq = v;
        cw = cq;
        if (q == len - 1) { vl = v; wl = cq; w0 = pi * cq; }
        else pi = (q == 0) ? -cq : pi * -cq;
      }
      z[q] = a;
      z[S + q] = rd;
      z[kZRecBack + q] = vq;
      z[kZRecBack + S + q] = cw;
      z[kZRecBack + 2 * S + q] = pw;
    }
  }
  float at = v0, ab = vl, ct = w0, cb = wl;
  z += kZRecStep;
  for (int d = 1; d < P; d <<= 1, z += kZStep) {
    st[0][p] = at; st[1][p] = ab; st[2][p] = ct; st[3][p] = cb;
    __syncthreads();
    const bool hm = on && p - d >= 0, hp = p + d < P;
    const float ab_m = hm ? st[1][p - d] : 0.0f, cb_m = hm ? st[3][p - d] : 0.0f;
    const float at_p = hp ? st[0][p + d] : 0.0f, ct_p = hp ? st[2][p + d] : 0.0f;
    __syncthreads();
    const float m11 = fm(-at, cb_m, 1.0f), m12 = -ct * at_p;
    const float m21 = -ab * cb_m, m22 = fm(-cb, at_p, 1.0f);
    const float id = rcp(fm(m11, m22, -(m12 * m21)));
    if (on) {
      z[0] = at; z[1] = ab; z[2] = ct; z[3] = cb;
      z[4] = m11; z[5] = m12; z[6] = m21; z[7] = m22;
      z[8] = id;
    }
    const float lt = -at * ab_m, lb = -ab * ab_m;
    const float ut = -ct * ct_p, ub = -cb * ct_p;
    at = id * fm(m22, lt, -(m12 * lb));
    ab = id * fm(m11, lb, -(m21 * lt));
    ct = id * fm(m22, ut, -(m12 * ub));
    cb = id * fm(m11, ub, -(m21 * ut));
  }
}

// A field as a raw buffer: a row's 32-bit byte offset is a scalar, a lane's
// the vector offset, and an access past the field's end reads zero or is
// dropped (a spare lane's offset is kNoLane).
typedef __amdgpu_buffer_rsrc_t Buf;
constexpr unsigned kNoLane = 0x80000000u;
__device__ __forceinline__ Buf field_buf(const void* p, unsigned bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00027000);
}
__device__ __forceinline__ float buf_ld(Buf b, unsigned lane, unsigned row) {
  return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, (int)lane, (int)row, 0));
}
__device__ __forceinline__ void buf_st(Buf b, unsigned lane, unsigned row, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_int(v), b, (int)lane, (int)row, 0);
}

// H false: 64 columns per workgroup, one segment per wave, whose table the
// wave holds without a vector load per row: A and RD in scalar registers
// (32 words; 48 spilled), the others one word per lane of two vector registers,
// read back with readlane.  H true (launches of few column groups, to spread
// over twice the CUs): 32 columns and two segments per wave; each wave stages
// its two records in LDS and reads them back per half while the data is on
// its way.  Either way the whole table is loaded with the data, before the
// first barrier: read where it is used, each part would be a cold dependent
// load (the sweep then took 3-10 % longer than zline_group).
//
// What it gives (FP32 half-sweep, zline_group -> this): 64x48x32 4.1 -> 3.1,
// 160x112x80 6.2 -> 5.7, 128^3 5.8 -> 5.1, from zero at 256^3 15.7 -> 13.3 us.
// The finest 256^3 sweep keeps its 20 us (100.7 MB): it is bound by the
// memory phase and by the start of its 8192 waves, not by arithmetic.
template <bool H>
__global__ __launch_bounds__(H ? 512 : 1024, H ? 2 : 8) void k_zline_shared(
    const DevLevel* __restrict__ Lt, LIST_PARAMS, int parity, int zero_guess, LaunchList ll) {
  extern __shared__ float zlds[];
  constexpr int S = kZSeg, CW = H ? 32 : 64;
  const Work wk = work_item(ln, lnb, li0, ll);
  const LevelHead L = level_head(Lt[wk.idx]);
  if (level_off(L)) return;
  const int nx = L.nx, ny = L.ny, nz = L.nz, hx = L.hx;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.y), tx = threadIdx.x;
  const int half = H ? tx >> 5 : 0, lane = tx & (CW - 1);
  const int P = (nz + S - 1) / S, PA = H ? (P + 1) & ~1 : P;
  const int p = H ? 2 * wave + half : wave;
  const sp<kG, const float> zr = gp(L.zt) + (H ? 2 * wave : wave) * kZRec;
  float* const zl = zlds + 4 * PA * CW + 2 * wave * kZRec;   // H: the wave's two records
  float ra[S], rd[S], tback = 0.0f, tstep = 0.0f, tr[6];
  if constexpr (H) {
#pragma unroll
    for (int q = 0; q < 6; ++q) tr[q] = zr[q * 64 + tx];
  } else {
#pragma unroll
    for (int q = 0; q < S; ++q) {
      ra[q] = zr[q];
      rd[q] = zr[S + q];
    }
    tback = zr[kZRecBack + tx];
    tstep = zr[kZRecStep + tx];
  }
  auto word = [](float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
  // word q of the segment's record, backward and step parts
  auto rec = [&](int q) { return zl[half * kZRec + q]; };
  auto back = [&](int q) { return H ? rec(kZRecBack + q) : word(tback, q); };
  auto stepw = [&](int q) { return H ? rec(kZRecStep + q) : word(tstep, q); };
  const int col0 = wk.lb * CW + lane, ncol = hx * ny;
  const int col = min(col0, ncol - 1);
  const int j = gm_div(col, L.gmhx, L.gshx), m = col - j * hx;
  const int c = parity, oth = parity ^ 1;
  const int r = (c + j) & 1, i = 2 * m + r;
  int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
  int mr = m + r;     if (mr >= hx) mr = 0;
  const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
  const sp<kG, const float> co = gp(L.co32);
  const sp<kG, const float> cy = co + 3 * nx;
  const sp<kG, const float> cz = cy + 3 * ny;
  const float wxl = co[i], wxr = co[nx + i], wys = cy[j], wyn = cy[ny + j];
  constexpr unsigned W = sizeof(float);
  const Buf u = field_buf(L.u, (unsigned)L.ncell * W), f = field_buf(L.f, (unsigned)L.ncell * W);
  const unsigned plane = (unsigned)(ny * 2 * hx) * W;
  const int ks = p * S, len = max(0, min(S, nz - ks));
  const unsigned bown = (unsigned)cidx(m, j, 0, c, hx, ny) * W;
  const unsigned xo = (unsigned)cidx(0, j, 0, oth, hx, ny);
  const unsigned bxl = (xo + ml) * W, bxr = (xo + mr) * W;
  const unsigned bso = (unsigned)cidx(m, jm, 0, oth, hx, ny) * W;
  const unsigned bno = (unsigned)cidx(m, jp, 0, oth, hx, ny) * W;
  // the sweep from zero reads b alone; a mixed cycle's first sweep is one
  // unless the cycle continues the previous one's iterate (kZgDyn)
  const int zg = (zero_guess & kZgDyn) && L.warm ? 0 : zero_guess & 3;
  // periodic z: the lagged wrap values, as in zline_group
  const bool lag = L.pz != 0 && !(zg & 2);
  float lagb = 0.0f, lagt = 0.0f;
  if (lag) {
    const float ubot = buf_ld(u, bown, (unsigned)(nz - 1) * plane), utop = buf_ld(u, bown, 0);
    lagb = p == 0 ? cz[0] * ubot : 0.0f;
    lagt = p == P - 1 ? cz[2 * nz - 1] * utop : 0.0f;
  }
  float g[S];
  // rows at vector offset vrow(q) and scalar offset srow(q)
  auto load = [&](auto vrow, auto srow) {
#pragma unroll
    for (int q = 0; q < S; ++q) g[q] = buf_ld(f, bown + vrow(q), srow(q));
    if (!(zg & 1)) {
      float xl[S], xr[S], ys[S], yn[S];
#pragma unroll
      for (int q = 0; q < S; ++q) {
        const unsigned v = vrow(q), o = srow(q);
        xl[q] = buf_ld(u, bxl + v, o);
        xr[q] = buf_ld(u, bxr + v, o);
        ys[q] = buf_ld(u, bso + v, o);
        yn[q] = buf_ld(u, bno + v, o);
      }
#pragma unroll
      for (int q = 0; q < S; ++q) g[q] -= zline_nbr(wxl, wxr, wys, wyn, xl[q], xr[q], ys[q], yn[q]);
    }
  };
  if constexpr (H) {
#pragma unroll
    for (int q = 0; q < 6; ++q) zl[q * 64 + tx] = tr[q];
  }
  // rows past nz are clamped to the last one: in bounds
  if constexpr (!H) {
    load([](int) { return 0u; }, [&](int q) { return (unsigned)min(ks + q, nz - 1) * plane; });
  } else if (nz == PA * S) {
    const unsigned v0 = (unsigned)ks * plane;
    load([=](int) { return v0; }, [=](int q) { return (unsigned)q * plane; });
  } else {
    load([=](int q) { return (unsigned)min(ks + q, nz - 1) * plane; }, [](int) { return 0u; });
  }
  if constexpr (H) {
    // the wave's own records: written and read by its lanes alone
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < S; ++q) {
      ra[q] = rec(q);
      rd[q] = rec(S + q);
    }
  } else {
#pragma unroll
    for (int q = 0; q < S; ++q) pin_s(ra[q], rd[q]);
  }
  if (lag) {
    g[0] -= lagb;
#pragma unroll
    for (int q = 0; q < S; ++q)
      if (q == len - 1) g[q] -= lagt;
  }
  float y = 0.0f, y0 = 0.0f;
#pragma unroll
  for (int q = 0; q < S; ++q) {
    y = fm(-ra[q], y, g[q]) * rd[q];
    g[q] = y;
    y0 = (q == 0) ? y : fm(back(2 * S + q), y, y0);
  }
  // the interface values, reduced as in zline_group: only the right-hand
  // sides are exchanged, the couplings are the table's
  float bprev = 0.0f, tnext = 0.0f;
  if (P > 1) {
    const int PS = PA * CW, sl = p * CW + lane;
    float rt = y0, rb = y;
    int buf = 0;
    for (int d = 1, w = 0; d < P; d <<= 1, buf ^= 1, w += kZStep) {
      const float at = stepw(w), ab = stepw(w + 1), ct = stepw(w + 2), cb = stepw(w + 3);
      const float m11 = stepw(w + 4), m12 = stepw(w + 5), m21 = stepw(w + 6), m22 = stepw(w + 7);
      const float id = stepw(w + 8);
      float* B = zlds + buf * 2 * PS;
      B[sl] = rt;
      B[PS + sl] = rb;
      __syncthreads();
      const bool hm = p - d >= 0, hp = p + d < P;
      const float rbm = B[PS + (hm ? sl - d * CW : sl)], rtp = B[hp ? sl + d * CW : sl];
      const float rb_m = hm ? rbm : 0.0f, rt_p = hp ? rtp : 0.0f;
      const float qt = fm(-ct, rt_p, fm(-at, rb_m, rt)), qb = fm(-cb, rt_p, fm(-ab, rb_m, rb));
      rt = id * fm(m22, qt, -(m12 * qb));
      rb = id * fm(m11, qb, -(m21 * qt));
    }
    float* B = zlds + buf * 2 * PS;
    B[sl] = rt;
    B[PS + sl] = rb;
    __syncthreads();
    const bool hm = p > 0, hp = p < P - 1;
    const float rbm = B[PS + (hm ? sl - CW : sl)], rtp = B[hp ? sl + CW : sl];
    bprev = hm ? rbm : 0.0f;
    tnext = hp ? rtp : 0.0f;
  }
  float x = tnext;
#pragma unroll
  for (int q = S - 1; q >= 0; --q) {
    x = fm(-back(S + q), x, fm(-back(q), bprev, g[q]));
    g[q] = x;
  }
  const unsigned bst = col0 < ncol ? bown + (H ? (unsigned)ks * plane : 0u) : kNoLane;
  const unsigned srow0 = H ? 0u : (unsigned)ks * plane;
  if (nz == PA * S) {
#pragma unroll
    for (int q = S - 1; q >= 0; --q) buf_st(u, bst, srow0 + (unsigned)q * plane, g[q]);
  } else {
#pragma unroll
    for (int q = S - 1; q >= 0; --q)
      if (q < len) buf_st(u, bst, srow0 + (unsigned)q * plane, g[q]);
  }
}

template <class T> struct TailNz;
template <> struct TailNz<float> { static constexpr int value = kTailNz; };
template <> struct TailNz<double> { static constexpr int value = kTailNz64; };

// Short columns (nz <= NZ) inside the coarse tail: one thread per column,
// the whole column in registers, plain Thomas (the reference's line solve,
// mgMK/mg_relax.F90:541-595); column index col = j*hx + m.  Every load (the
// right-hand-side data and the z coefficients) is issued before the
// elimination; with EXACT (nz == NZ) the chains carry no predicates.
template <class T, int NZ, bool EXACT, class UP, class FP, class CP>
__device__ __forceinline__ void zline_column(const LevelHead& L, UP u, FP f, CP co, int parity,
                                             int zero_guess, int col) {
  const int hx = L.hx, ny = L.ny, nx = L.nx;
  const int nz = EXACT ? NZ : L.nz;
  // A compiler barrier: it keeps the solve in a scheduling region of its own,
  // apart from the caller's step dispatch.  Without it the coarse tail's
  // line-solve steps run about 1.3x slower on gfx950 (measured: 60 -> 46 us
  // per FP32 tail at 16^3..4^3).
  asm volatile("" ::: "memory");
  const int m = col % hx, j = col / hx;
  const int c = parity, oth = parity ^ 1;
  const int i = 2 * m + ((c + j) & 1), r = i & 1;
  int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
  int mr = m + r;     if (mr >= hx) mr = 0;
  const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
  const auto cy = co + 3 * nx;
  const auto cz = cy + 3 * ny;
  const T wxl = co[i], wxr = co[nx + i], wys = cy[j], wyn = cy[ny + j];
  const T dxy = co[2 * nx + i] + cy[2 * ny + j];
  const int plane = ny * 2 * hx;
  const int own = cidx(m, j, 0, c, hx, ny);
  const int xo = cidx(0, j, 0, oth, hx, ny);
  const int so = cidx(m, jm, 0, oth, hx, ny);
  const int no = cidx(m, jp, 0, oth, hx, ny);
  const bool pz = L.pz != 0;
  const bool lag = pz && !(zero_guess & 2);
  const bool nbr = !(zero_guess & 1);
  const T ubot = u[(nz - 1) * plane + own], utop = u[own];
  const T lagb = lag ? cz[0] * ubot : T(0);
  const T lagt = lag ? cz[2 * nz - 1] * utop : T(0);
  // z coefficients held in registers for columns of up to 16 cells
  constexpr bool HOIST = NZ <= 16;
  constexpr int NH = HOIST ? NZ : 1;
  T g[NZ], za[NH], ze[NH], zd[NH];
#pragma unroll
  for (int q = 0; q < NZ; ++q) {
    const int k = EXACT ? q : min(q, nz - 1);     // rows clamped: every load in bounds
    const int kb = k * plane;
    const T fv = f[kb + own];
    const T xl = u[kb + xo + ml], xr = u[kb + xo + mr], ys = u[kb + so], yn = u[kb + no];
    if constexpr (HOIST) {
      za[q] = cz[k];
      ze[q] = cz[nz + k];
      zd[q] = cz[2 * nz + k];
    }
    T sn = wxl * xl + wxr * xr;
    sn += wys * ys;
    sn += wyn * yn;
    T v = nbr ? fv - sn : fv;
    v -= (q == 0) ? lagb : T(0);
    v -= (q == nz - 1) ? lagt : T(0);
    g[q] = v;
  }
  T cpa[NZ];
  T cp = T(0), yf = T(0);
#pragma unroll
  for (int q = 0; q < NZ; ++q) {
    if (EXACT || q < nz) {
      const T a = (q == 0) ? T(0) : (HOIST ? za[HOIST ? q : 0] : cz[q]);
      const T e = (q == nz - 1) ? T(0) : (HOIST ? ze[HOIST ? q : 0] : cz[nz + q]);
      const T rd = rcp(((HOIST ? zd[HOIST ? q : 0] : cz[2 * nz + q]) + dxy) - a * cp);
      yf = (g[q] - a * yf) * rd;
      cp = e * rd;
      g[q] = yf;
      cpa[q] = cp;
    }
  }
  T x = T(0);
#pragma unroll
  for (int q = NZ - 1; q >= 0; --q) {
    if (EXACT || q < nz) {
      x = g[q] - cpa[q] * x;
      u[q * plane + own] = x;
    }
  }
}

// Dispatch on the column length: an exact instantiation for full columns
// of NZ, NZ/2 and NZ/4 cells, the predicated one otherwise.
template <class T, int NZ, class UP, class FP, class CP>
__device__ __forceinline__ void zline_column_n(const LevelHead& L, UP u, FP f, CP co, int parity,
                                               int zero_guess, int col) {
  const int nz = L.nz;
  if (nz == NZ) zline_column<T, NZ, true>(L, u, f, co, parity, zero_guess, col);
  else if (NZ >= 8 && nz == NZ / 2) zline_column<T, (NZ >= 8 ? NZ / 2 : NZ), true>(L, u, f, co, parity, zero_guess, col);
  else if (NZ >= 16 && nz == NZ / 4) zline_column<T, (NZ >= 16 ? NZ / 4 : NZ), true>(L, u, f, co, parity, zero_guess, col);
  else zline_column<T, NZ, false>(L, u, f, co, parity, zero_guess, col);
}

// The standalone short-column sweep (tests of the tail's line solve).
template <class T, class UP, class FP, class CP>
__device__ __forceinline__ void zline_column_any(const LevelHead& L, UP u, FP f, CP co, int parity,
                                                 int zero_guess, int col) {
  if (L.nz <= 16 || TailNz<T>::value <= 16) zline_column_n<T, 16>(L, u, f, co, parity, zero_guess, col);
  else zline_column_n<T, TailNz<T>::value>(L, u, f, co, parity, zero_guess, col);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_zline_col(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                      int parity, int zero_guess, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const LevelHead L = level_head(Lt[wk.idx]);
  if (level_off(L)) return;
  const int e = wk.lb * kBlock + threadIdx.x;
  if (e < L.hx * L.ny)
    zline_column_any<T>(L, gfield<T>(L.u), gfield<const T>((const void*)L.f), coefs<T>(L), parity,
                        zero_flags(L, zero_guess), e);
}

// ---------------------------------------------------------------------------
// Fused residual + volume-weighted restriction (mgMK/mg_restr.F90:124-164):
// element e is a coarse cell in natural (I fastest) order, so the fine reads
// of a wave are contiguous half-rows; the fine residual is never stored.
// FX, FY, FZ: the coarsening factors (1 or 2), compile-time so that the
// children loop unrolls and its loads are issued together.
template <class T, int FX, int FY, int FZ, class UP, class FP, class CP, class VP, class CFP>
__device__ __forceinline__ void restrict_elem(const LevelHead& F, UP u, FP f, CP co, VP vol,
                                              const LevelHead& C, CFP fc, int e) {
  // nx = 2 hx: e / nx = (e >> 1) / hx
  const int JK = gm_div(e >> 1, C.gmhx, C.gshx), I = e - JK * C.nx;
  const int K = gm_div(JK, C.gmny, C.gsny), J = JK - K * C.ny;
  const auto vx = vol;
  const auto vy = vx + F.nx;
  const auto vz = vy + F.ny;
  T acc = T(0), vs = T(0);
#pragma unroll
  for (int cz = 0; cz < FZ; ++cz) {
    const int k = K * FZ + cz;
#pragma unroll
    for (int cy = 0; cy < FY; ++cy) {
      const int j = J * FY + cy;
#pragma unroll
      for (int cx = 0; cx < FX; ++cx) {
        const int i = I * FX + cx;
        const Nb n = neighbours(F, i, j, k);
        const T s = offsum<T>(co, F, i, j, k, u[n.xm], u[n.xp], u[n.ym], u[n.yp], u[n.zm], u[n.zp]);
        const T rr = f[n.c] - (s + diag_at<T>(co, F, i, j, k) * u[n.c]);
        const T v = T(vz[k] * vy[j] * vx[i]);
        acc += v * rr;
        vs += v;
      }
    }
  }
  fc[cidx(I >> 1, J, K, (I + J) & 1, C.hx, C.ny)] = acc / vs;
}

template <class T, class UP, class FP, class CP, class VP, class CFP>
__device__ __forceinline__ void restrict_any(const LevelHead& F, UP u, FP f, CP co, VP vol,
                                             const LevelHead& C, CFP fc, const DevXfer& x, int e) {
  const int code = (x.fx - 1) * 4 + (x.fy - 1) * 2 + (x.fz - 1);
  switch (code) {
    case 7: restrict_elem<T, 2, 2, 2>(F, u, f, co, vol, C, fc, e); break;
    case 6: restrict_elem<T, 2, 2, 1>(F, u, f, co, vol, C, fc, e); break;
    case 5: restrict_elem<T, 2, 1, 2>(F, u, f, co, vol, C, fc, e); break;
    case 4: restrict_elem<T, 2, 1, 1>(F, u, f, co, vol, C, fc, e); break;
    case 3: restrict_elem<T, 1, 2, 2>(F, u, f, co, vol, C, fc, e); break;
    case 2: restrict_elem<T, 1, 2, 1>(F, u, f, co, vol, C, fc, e); break;
    case 1: restrict_elem<T, 1, 1, 2>(F, u, f, co, vol, C, fc, e); break;
    default: restrict_elem<T, 1, 1, 1>(F, u, f, co, vol, C, fc, e); break;
  }
}

// A transfer's descriptor and its two levels' heads: two reads, not one per
// field used.
__device__ __forceinline__ DevXfer xfer_of(const DevXfer& X) {
  DevXfer x = X;
  pin_s(x.fine, x.coarse, x.fx, x.fy, x.fz, x.skip, x.rskip, x.pmx, x.pmy, x.psx, x.psy);
  return x;
}
__device__ __forceinline__ void level_heads(const DevLevel& A, const DevLevel& B, LevelHead& a,
                                            LevelHead& b) {
  a = A;
  b = B;
  pin_s(a.nx, a.ny, a.nz, a.hx, a.stop, a.gmhx, a.gmny, a.gshx, a.gsny, a.px, a.py, a.pz, a.u, a.f);
  pin_s(a.co64, a.co32, a.vol, b.nx, b.ny, b.nz, b.hx, b.gmhx, b.gmny, b.gshx, b.gsny, b.ncell, b.u, b.f);
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_restrict(const DevLevel* __restrict__ Lt,
                                                     const DevXfer* __restrict__ X, LIST_PARAMS,
                                                     LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevXfer x = xfer_of(X[wk.idx]);
  LevelHead F, C;
  level_heads(Lt[x.fine], Lt[x.coarse], F, C);
  if (level_off(F)) return;
  const int e = wk.lb * kBlock + threadIdx.x;
  if (e < C.ncell)
    restrict_any<T>(F, gfield<const T>((const void*)F.u), gfield<const T>((const void*)F.f),
                    coefs<T>(F), gp(F.vol), C, gfield<T>(C.f), x, e);
}

// The same with factor 2 in every direction, four lanes per coarse cell: each
// takes the two fine cells of one row of its block, the quad adds up.  For
// levels of few cells (restrict_quad_ok), where one thread per coarse cell is
// a chain of eight residuals on a few workgroups: 32x24x16 coarse cells in
// FP32 5.3 -> 3.0 us.  sk: as restrict222_cols (a row has one cell of colour
// 1, so half the loads go).
template <class T>
__device__ __forceinline__ T quad_sum(T v) {
  // lanes xor 1, then xor 2 (DPP quad permutes)
  auto move = [](T x, auto ctrl) {
    constexpr int W = sizeof(T) / 4, C = decltype(ctrl)::value;
    int w[W];
    __builtin_memcpy(w, &x, sizeof(T));
#pragma unroll
    for (int q = 0; q < W; ++q) w[q] = __builtin_amdgcn_update_dpp(0, w[q], C, 0xf, 0xf, true);
    T r;
    __builtin_memcpy(&r, w, sizeof(T));
    return r;
  };
  v += move(v, std::integral_constant<int, 0xb1>());
  return v + move(v, std::integral_constant<int, 0x4e>());
}
template <class T>
__global__ __launch_bounds__(kBlock) void k_restrict_quad(const DevLevel* __restrict__ Lt,
                                                          const DevXfer* __restrict__ X, LIST_PARAMS,
                                                          int use_skip, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevXfer x = xfer_of(X[wk.idx]);
  LevelHead F, C;
  level_heads(Lt[x.fine], Lt[x.coarse], F, C);
  if (level_off(F)) return;
  const int t = wk.lb * kBlock + threadIdx.x, q = t & 3;
  const int e = min(t >> 2, C.ncell - 1);             // whole quads stay to the sum
  const int JK = gm_div(e >> 1, C.gmhx, C.gshx), I = e - JK * C.nx;
  const int K = gm_div(JK, C.gmny, C.gsny), J = JK - K * C.ny;
  const auto u = gfield<const T>((const void*)F.u);
  const auto f = gfield<const T>((const void*)F.f);
  const auto co = coefs<T>(F);
  const auto vx = gp(F.vol), vy = vx + F.nx, vz = vy + F.ny;
  const int k = 2 * K + (q >> 1), j = 2 * J + (q & 1);
  const double vyz = vz[k] * vy[j];
  const T v0 = T(vyz * vx[2 * I]), v1 = T(vyz * vx[2 * I + 1]);
  auto res = [&](int i) {
    const Nb n = neighbours(F, i, j, k);
    const T s = offsum<T>(co, F, i, j, k, u[n.xm], u[n.xp], u[n.ym], u[n.yp], u[n.zm], u[n.zp]);
    return f[n.c] - (s + diag_at<T>(co, F, i, j, k) * u[n.c]);
  };
  const int sk = use_skip ? x.rskip : kXferSkipNone;
  T acc;
  if (sk == kXferSkipNone) {
    acc = v0 * res(2 * I) + v1 * res(2 * I + 1);
  } else {
    // the row's cell of colour 0
    const int b = (sk == kXferSkipLine ? j : j + k) & 1;
    acc = (b ? v1 : v0) * res(2 * I + b);
  }
  acc = quad_sum(acc);
  const T vs = quad_sum(v0 + v1);
  if (q == 0 && (t >> 2) < C.ncell)
    gfield<T>(C.f)[cidx(I >> 1, J, K, (I + J) & 1, C.hx, C.ny)] = acc / vs;
}

// Residual + restriction of a transfer with factor 2 in every direction and
// fine sizes exactly twice the coarse ones, marching in z.  A thread owns
// coarse column (I, J) over a slab of restrict222_k coarse planes: fine
// columns i in {2I, 2I+1}, j in {2J, 2J+1}.  It walks their fine planes
// upward with the centre values of the planes below, at and above in
// registers; per coarse cell it loads the centres of the two planes above,
// b of its two planes and the eight in-plane neighbours outside its 2x2
// block (16 loads per fine plane, against 32 for restrict_elem).  The
// neighbours inside the block are its own centres, at the indices
// neighbours() gives, and the outside ones take its wraps.  Each fine
// residual is formed with offsum/diag_at as in restrict_elem, and the coarse
// value sums its eight in the same order (z, then y, then x), so the result
// is restrict_elem's.
//
// SK (DevXfer::rskip): after the fine level's pre-smoothing, whose last
// half-sweep solved the equations of its colour-1 cells from their
// neighbours, those cells' residuals are zero but for rounding; they are
// taken as zero, and the loads only they need (their b and their outside
// neighbours) are not in the code.  Colour 1 of cell (2I+cx, 2J+cy, 2K+h):
// (cx+cy) odd for the z-line sweep, (cx+cy+h) odd for the point sweep.
template <int SK>
__device__ __forceinline__ constexpr bool restrict_keeps(int cx, int cy, int h) {
  return SK == kXferSkipLine ? ((cx + cy) & 1) == 0
       : SK == kXferSkipPoint ? ((cx + cy + h) & 1) == 0 : true;
}

template <class T, int SK>
__device__ __forceinline__ void restrict222_cols(const LevelHead& F, const LevelHead& C, int I, int J,
                                                 int K0, int K1) {
  const auto u = gfield<const T>((const void*)F.u);
  const auto f = gfield<const T>((const void*)F.f);
  const auto co = coefs<T>(F);
  const auto vx = gp(F.vol);
  const auto vy = vx + F.nx;
  const auto vz = vy + F.ny;
  const int hx = F.hx, ny = F.ny, nz = F.nz;
  const int plane = 2 * hx * ny;
  // in-plane offsets: own cells o[cy][cx], outside neighbours
  int o[2][2], oxm[2], oxp[2], oym[2], oyp[2];
#pragma unroll
  for (int cy = 0; cy < 2; ++cy)
#pragma unroll
    for (int cx = 0; cx < 2; ++cx) {
      const int i = 2 * I + cx, j = 2 * J + cy;
      o[cy][cx] = cidx(i >> 1, j, 0, (i + j) & 1, hx, ny);
    }
#pragma unroll
  for (int cy = 0; cy < 2; ++cy) {
    const int j = 2 * J + cy;
    // x- of i = 2I (r = 0: m - 1, wrapped) and x+ of i = 2I+1 (r = 1: m + 1, wrapped)
    const int ml = I == 0 ? hx - 1 : I - 1, mr = I + 1 >= hx ? 0 : I + 1;
    oxm[cy] = cidx(0, j, 0, ((2 * I + j) & 1) ^ 1, hx, ny) + ml;
    oxp[cy] = cidx(0, j, 0, ((2 * I + 1 + j) & 1) ^ 1, hx, ny) + mr;
  }
#pragma unroll
  for (int cx = 0; cx < 2; ++cx) {
    const int i = 2 * I + cx;
    const int j0 = 2 * J, j1 = 2 * J + 1;
    const int jm = j0 == 0 ? ny - 1 : j0 - 1, jp = j1 == ny - 1 ? 0 : j1 + 1;
    oym[cx] = cidx(i >> 1, jm, 0, ((i + j0) & 1) ^ 1, hx, ny);
    oyp[cx] = cidx(i >> 1, jp, 0, ((i + j1) & 1) ^ 1, hx, ny);
  }
  auto ld4 = [&](int k, T (&v)[2][2]) {
#pragma unroll
    for (int cy = 0; cy < 2; ++cy)
#pragma unroll
      for (int cx = 0; cx < 2; ++cx) v[cy][cx] = u[k * plane + o[cy][cx]];
  };
  T um[2][2], uc[2][2];
  const int k00 = 2 * K0;
  ld4(k00 == 0 ? nz - 1 : k00 - 1, um);
  ld4(k00, uc);
  for (int K = K0; K < K1; ++K) {
    const int ka = 2 * K, kb = ka + 1, kc = kb == nz - 1 ? 0 : kb + 1;
    // every load of the coarse cell first
    T ua[2][2], ub[2][2], fv[2][2][2], xm[2][2], xp[2][2], ym[2][2], yp[2][2];
    ld4(kb, ua);
    ld4(kc, ub);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int kk = ka + h;
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        // fv[h][cy][cx]; xm/xp[h][cy] serve cells (0, cy)/(1, cy), ym/yp[h][cx]
        // cells (cx, 0)/(cx, 1)
        fv[h][q][0] = restrict_keeps<SK>(0, q, h) ? f[kk * plane + o[q][0]] : T(0);
        fv[h][q][1] = restrict_keeps<SK>(1, q, h) ? f[kk * plane + o[q][1]] : T(0);
        xm[h][q] = restrict_keeps<SK>(0, q, h) ? u[kk * plane + oxm[q]] : T(0);
        xp[h][q] = restrict_keeps<SK>(1, q, h) ? u[kk * plane + oxp[q]] : T(0);
        ym[h][q] = restrict_keeps<SK>(q, 0, h) ? u[kk * plane + oym[q]] : T(0);
        yp[h][q] = restrict_keeps<SK>(q, 1, h) ? u[kk * plane + oyp[q]] : T(0);
      }
    }
    T acc = T(0), vs = T(0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int k = ka + h;
      const T (&zm)[2][2] = h ? uc : um;
      const T (&cc)[2][2] = h ? ua : uc;
      const T (&zp)[2][2] = h ? ub : ua;
#pragma unroll
      for (int cy = 0; cy < 2; ++cy) {
        const int j = 2 * J + cy;
#pragma unroll
        for (int cx = 0; cx < 2; ++cx) {
          const int i = 2 * I + cx;
          const T v = T(vz[k] * vy[j] * vx[i]);
          if (restrict_keeps<SK>(cx, cy, h)) {
            const T uxm = cx ? cc[cy][0] : xm[h][cy];
            const T uxp = cx ? xp[h][cy] : cc[cy][1];
            const T uym = cy ? cc[0][cx] : ym[h][cx];
            const T uyp = cy ? yp[h][cx] : cc[1][cx];
            const T s = offsum<T>(co, F, i, j, k, uxm, uxp, uym, uyp, zm[cy][cx], zp[cy][cx]);
            const T rr = fv[h][cy][cx] - (s + diag_at<T>(co, F, i, j, k) * cc[cy][cx]);
            acc += v * rr;
          }
          vs += v;
        }
      }
    }
    gfield<T>(C.f)[cidx(I >> 1, J, K, (I + J) & 1, C.hx, C.ny)] = acc / vs;
#pragma unroll
    for (int cy = 0; cy < 2; ++cy)
#pragma unroll
      for (int cx = 0; cx < 2; ++cx) {
        um[cy][cx] = ua[cy][cx];
        uc[cy][cx] = ub[cy][cx];
      }
  }
}

// use_skip: take the transfer's rskip rule (the V-cycle's restriction after
// pre-smoothing); 0 forms every residual.
template <class T>
__global__ __launch_bounds__(kBlock) void k_restrict222(const DevLevel* __restrict__ Lt,
                                                        const DevXfer* __restrict__ X, LIST_PARAMS,
                                                        int use_skip, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevXfer x = xfer_of(X[wk.idx]);
  LevelHead F, C;
  level_heads(Lt[x.fine], Lt[x.coarse], F, C);
  if (level_off(F)) return;
  const int cols = C.nx * C.ny;
  const int ncb = (cols + kBlock - 1) / kBlock;
  const int lb = wk.lb;
  const int bk = lb / ncb, col = (lb - bk * ncb) * kBlock + threadIdx.x;
  if (col >= cols) return;
  const int J = gm_div(col >> 1, C.gmhx, C.gshx), I = col - J * C.nx;   // col / nx, nx = 2 hx
  const int kr = restrict222_k(C);
  const int K0 = bk * kr, K1 = min(K0 + kr, C.nz);
  const int sk = use_skip ? x.rskip : kXferSkipNone;
  if (sk == kXferSkipLine) restrict222_cols<T, kXferSkipLine>(F, C, I, J, K0, K1);
  else if (sk == kXferSkipPoint) restrict222_cols<T, kXferSkipPoint>(F, C, I, J, K0, K1);
  else restrict222_cols<T, kXferSkipNone>(F, C, I, J, K0, K1);
}

// ---------------------------------------------------------------------------
// Trilinear prolongation-add (mgMK/mg_cor.F90:102-159): fine u += sum of
// 27,9,9,3,9,3,3,1 /64 of the eight nearest coarse cells; coarse ghosts are
// periodic wraps, Neumann copies or Dirichlet zeros.
//
// One thread per dual cell (prolong_duals): the fine cells between coarse
// centres I and I+1 in each direction share the same eight coarse values,
// which are loaded once.  Per factor-2 direction the dual d covers fine
// cells 2I+1 (weights 3/4 on I, 1/4 on I+1) and 2I+2 (3/4 on I+1, 1/4 on I)
// with I = d (periodic, I+1 and 2I+2 wrapped) or I = d-1 (walls: the half
// duals d = 0 and d = nc hold one fine cell; the missing coarse value is
// the ghost -- the neighbour's value for Neumann, zero for Dirichlet).  A
// factor-1 direction maps cell to cell with weight 1.  Each fine value is
// summed nearest-first: x, then y, then z.
//
// skip (DevXfer::skip, kXferSkip*): the cells that the fine level's first
// post-smoothing half-sweep rewrites from the other colour and b alone are
// neither read nor written -- their correction would be overwritten unread,
// so the result of that half-sweep, and of everything after it, is the same.
struct PDir {
  int fi0, fi1;     // fine indices (fine cell 0 is nearest to coarse centre 0)
  bool fv0, fv1;    // fine cell exists
  int ci0, ci1;     // coarse indices
  bool cz0, cz1;    // coarse value is a Dirichlet zero ghost
  __device__ int fi(int h) const { return h ? fi1 : fi0; }
  __device__ bool fv(int h) const { return h ? fv1 : fv0; }
  __device__ int ci(int h) const { return h ? ci1 : ci0; }
  __device__ bool cz(int h) const { return h ? cz1 : cz0; }
};

template <int F>
__device__ __forceinline__ PDir pdir(int d, int nc, int per, int bc0, int bc1) {
  PDir r;
  if (F == 1) {
    r.fi0 = r.fi1 = d;
    r.fv0 = true; r.fv1 = false;
    r.ci0 = r.ci1 = d;
    r.cz0 = r.cz1 = false;
    return r;
  }
  const int nf = 2 * nc;
  if (per) {
    const int I = d;
    r.fi0 = 2 * I + 1;
    r.fi1 = (2 * I + 2 == nf) ? 0 : 2 * I + 2;
    r.fv0 = r.fv1 = true;
    r.ci0 = I;
    r.ci1 = (d + 1 == nc) ? 0 : d + 1;
    r.cz0 = r.cz1 = false;
  } else {
    const int I = d - 1;
    r.fi0 = 2 * I + 1;
    r.fi1 = 2 * I + 2;
    r.fv0 = I >= 0;
    r.fv1 = I + 1 < nc;
    // a missing coarse centre takes the ghost rule of its wall
    r.ci0 = (I >= 0) ? I : 0;
    r.ci1 = (I + 1 < nc) ? I + 1 : nc - 1;
    r.cz0 = (I < 0) && bc0 == 2;
    r.cz1 = (I + 1 >= nc) && bc1 == 2;
  }
  return r;
}

// Whether fine cell (h, q, a) of a 2:2:2 dual is corrected under skip rule
// SK.  Fine cell 0 of a factor-2 direction has an odd index (2I+1) and cell
// 1 an even one (2I+2, or 0 wrapped), so the colour of each cell is fixed by
// its position in the dual: the skipped cells are known at compile time,
// and their loads and stores are not in the code.
template <int SK>
__device__ __forceinline__ constexpr bool prolong_keeps(int h, int q, int a) {
  return SK == kXferSkipNone ? true
       : (SK == kXferSkipLine || SK == kXferSkipLineWrap) ? (((1 - h) + (1 - q)) & 1) != 0
       : (((1 - h) + (1 - q) + (1 - a)) & 1) != 0;
}

template <class T, int FX, int FY, int FZ, int SK = kXferSkipNone, class UP, class CUP>
__device__ __forceinline__ void prolong_dual(const DevLevel& F, UP u, const LevelHead& C, CUP uc,
                                             const DevXfer& x, int e) {
  static_assert(SK == kXferSkipNone || (FX == 2 && FY == 2 && FZ == 2), "skip: 2:2:2 duals only");
  constexpr int NX = FX == 2 ? 2 : 1, NY = FY == 2 ? 2 : 1, NZ = FZ == 2 ? 2 : 1;
  const int ndx = prolong_duals_dir(C.nx, FX, F.px), ndy = prolong_duals_dir(C.ny, FY, F.py);
  // e = (dz * ndy + dy) * ndx + dx, divided by the transfer's invariant divisors
  const int dyz = gm_div(e, x.pmx, x.psx), dx = e - dyz * ndx;
  const int dz = gm_div(dyz, x.pmy, x.psy), dy = dyz - dz * ndy;
  const PDir X = pdir<FX>(dx, C.nx, F.px, F.bcx0, F.bcx1);
  const PDir Y = pdir<FY>(dy, C.ny, F.py, F.bcy0, F.bcy1);
  const PDir Z = pdir<FZ>(dz, C.nz, F.pz, F.bcz0, F.bcz1);
  // every load first: the coarse values v[z][y][x] (index 0: the near
  // centre of fine cell 0) and the fine cells' old values (a missing cell's
  // index is clamped to its partner; it is not stored; a skipped cell is
  // neither loaded nor stored)
  T v[NZ][NY][NX], fold[NZ][NY][NX];
  int fid[NZ][NY][NX];
  bool keep[NZ][NY][NX];
  // with periodic z the z-line sweep's lagged wrap reads its own colour at
  // rows 0 and nz-1: both are cells of the last z dual
  const bool zwrap = SK == kXferSkipLineWrap && Z.fi(NZ - 1) == 0;
#pragma unroll
  for (int a = 0; a < NZ; ++a)
#pragma unroll
    for (int q = 0; q < NY; ++q)
#pragma unroll
      for (int h = 0; h < NX; ++h) {
        const int I = X.ci(h), J = Y.ci(q), K = Z.ci(a);
        // a Dirichlet ghost contributes zero: a 0/1 factor, not a branch,
        // so that all loads stay in one batch (the same 0*value as a zero
        // interpolation weight)
        const T c = uc[cidx(I >> 1, J, K, (I + J) & 1, C.hx, C.ny)];
        v[a][q][h] = c * ((X.cz(h) || Y.cz(q) || Z.cz(a)) ? T(0) : T(1));
        const int i = X.fv(h) ? X.fi(h) : X.fi(h ^ (NX - 1));
        const int j = Y.fv(q) ? Y.fi(q) : Y.fi(q ^ (NY - 1));
        const int k = Z.fv(a) ? Z.fi(a) : Z.fi(a ^ (NZ - 1));
        fid[a][q][h] = cidx(i >> 1, j, k, (i + j) & 1, F.hx, F.ny);
        keep[a][q][h] = X.fv(h) && Y.fv(q) && Z.fv(a) && (prolong_keeps<SK>(h, q, a) || zwrap);
        fold[a][q][h] = (prolong_keeps<SK>(h, q, a) || zwrap) ? u[fid[a][q][h]] : T(0);
      }
  // keep the old values' loads in the batch above (an empty register
  // constraint: otherwise a load is sunk into its predicated store)
#pragma unroll
  for (int a = 0; a < NZ; ++a)
#pragma unroll
    for (int q = 0; q < NY; ++q)
#pragma unroll
      for (int h = 0; h < NX; ++h) asm volatile("" : "+v"(fold[a][q][h]));
  // separable interpolation, nearest first: along x, then y, then z
  T ix[NZ][NY][NX], iy[NZ][NY][NX];
#pragma unroll
  for (int a = 0; a < NZ; ++a)
#pragma unroll
    for (int q = 0; q < NY; ++q)
#pragma unroll
      for (int h = 0; h < NX; ++h)
        ix[a][q][h] = (NX == 2) ? T(0.75) * v[a][q][h] + T(0.25) * v[a][q][h ^ (NX - 1)] : v[a][q][h];
#pragma unroll
  for (int a = 0; a < NZ; ++a)
#pragma unroll
    for (int q = 0; q < NY; ++q)
#pragma unroll
      for (int h = 0; h < NX; ++h)
        iy[a][q][h] = (NY == 2) ? T(0.75) * ix[a][q][h] + T(0.25) * ix[a][q ^ (NY - 1)][h] : ix[a][q][h];
#pragma unroll
  for (int a = 0; a < NZ; ++a)
#pragma unroll
    for (int q = 0; q < NY; ++q)
#pragma unroll
      for (int h = 0; h < NX; ++h) {
        const T add = (NZ == 2) ? T(0.75) * iy[a][q][h] + T(0.25) * iy[a ^ (NZ - 1)][q][h] : iy[a][q][h];
        if (keep[a][q][h]) u[fid[a][q][h]] = fold[a][q][h] + add;
      }
}

template <class T, class UP, class CUP>
__device__ __forceinline__ void prolong_any(const DevLevel& F, UP u, const LevelHead& C, CUP uc,
                                            const DevXfer& x, int e, int skip = kXferSkipNone) {
  const int code = (x.fx - 1) * 4 + (x.fy - 1) * 2 + (x.fz - 1);
  switch (code) {
    case 7:
      // the skip rules apply to 2:2:2 transfers (DevXfer::skip)
      if (skip == kXferSkipLine) prolong_dual<T, 2, 2, 2, kXferSkipLine>(F, u, C, uc, x, e);
      else if (skip == kXferSkipLineWrap) prolong_dual<T, 2, 2, 2, kXferSkipLineWrap>(F, u, C, uc, x, e);
      else if (skip == kXferSkipPoint) prolong_dual<T, 2, 2, 2, kXferSkipPoint>(F, u, C, uc, x, e);
      else prolong_dual<T, 2, 2, 2>(F, u, C, uc, x, e);
      break;
    case 6: prolong_dual<T, 2, 2, 1>(F, u, C, uc, x, e); break;
    case 5: prolong_dual<T, 2, 1, 2>(F, u, C, uc, x, e); break;
    case 4: prolong_dual<T, 2, 1, 1>(F, u, C, uc, x, e); break;
    case 3: prolong_dual<T, 1, 2, 2>(F, u, C, uc, x, e); break;
    case 2: prolong_dual<T, 1, 2, 1>(F, u, C, uc, x, e); break;
    case 1: prolong_dual<T, 1, 1, 2>(F, u, C, uc, x, e); break;
    default: prolong_dual<T, 1, 1, 1>(F, u, C, uc, x, e); break;
  }
}

// use_skip: leave the cells of the transfer's skip rule (the V-cycle's
// prolongation, followed by the fine level's post-smoothing); 0 corrects
// every cell.
template <class T>
__global__ __launch_bounds__(kBlock) void k_prolong(const DevLevel* __restrict__ Lt,
                                                    const DevXfer* __restrict__ X, LIST_PARAMS,
                                                    int use_skip, LaunchList ll) {
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevXfer x = xfer_of(X[wk.idx]);
  DevLevel F = Lt[x.fine];
  LevelHead C;
  pin_s(F.bcx0, F.bcx1, F.bcy0, F.bcy1, F.bcz0, F.bcz1);
  level_heads(F, Lt[x.coarse], F, C);
  if (level_off(F)) return;
  const int e = wk.lb * kBlock + threadIdx.x;
  const int nd = prolong_duals_dir(C.nx, x.fx, F.px) * prolong_duals_dir(C.ny, x.fy, F.py) *
                 prolong_duals_dir(C.nz, x.fz, F.pz);
  if (e < nd)
    prolong_any<T>(F, gfield<T>(F.u), C, gfield<const T>((const void*)C.u), x, e,
                   use_skip ? x.skip : kXferSkipNone);
}

// ---------------------------------------------------------------------------
// Coarsest level: u = Minv f with a precomputed FP64 (pseudo-)inverse
// stored transposed (row r of the product reads column r: coalesced), FP64
// accumulation in eight independent partial sums.
template <class T, class UP, class FP, class MP>
__device__ __forceinline__ void coarse_row(const DevLevel& L, UP u, FP f, MP Mt, int r) {
  const int n = L.ncell;
  const auto M = Mt + r;
  double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int s = 0;
  // 16 matrix loads in flight per row: a large coarsest level (an 8 MB
  // inverse at 1024 cells) is read by one workgroup, and with fewer loads
  // per thread its rate is set by the memory latency.  Element s+q adds to
  // acc[(s+q) & 7] in increasing s, as in the 8-wide loop below.
  for (; s + 16 <= n; s += 16) {
    double m[16];
    T fv[16];
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      m[q] = M[(s + q) * n];
      fv[q] = f[s + q];
    }
#pragma unroll
    for (int q = 0; q < 16; ++q) acc[q & 7] += m[q] * (double)fv[q];
  }
  for (; s + 8 <= n; s += 8) {
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] += M[(s + q) * n] * (double)f[s + q];
  }
  for (; s < n; ++s) acc[0] += M[s * n] * (double)f[s];
  const double sum = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  u[r] = (T)sum;
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_coarse(const DevLevel* __restrict__ Lt, LaunchList ll) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  if (level_off(L)) return;
  const int r = (b - ll.prefix[t]) * kBlock + threadIdx.x;
  if (r < L.ncell) coarse_row<T>(L, gfield<T>(L.u), gfield<const T>((const void*)L.f), gp(L.minvT), r);
}

// ---------------------------------------------------------------------------
// Coarse tail: the whole sub-V-cycle below a level (pre-smoothing and
// residual restriction down to the coarsest level, its exact solve, then
// prolongation and post-smoothing back up -- the order of
// mgMK/mg_cycle.F90) for one instance in one workgroup of 64*kTailWaves
// threads, with workgroup barriers between the steps instead of dependent
// launches.  The tail levels' u, f, coefficient tables and cell widths live
// in LDS (the first level's f, and u when it is an input, are copied in,
// its u copied out); the element routines are the standalone kernels' ones
// instantiated with LDS pointers.  One workgroup per item (DevTail).
// Global -> LDS copy of n values (converted to D) by `nthr` threads: each
// thread issues its (up to) 8 loads before any store, so a copy costs one
// memory round trip per 8*nthr values instead of one per nthr.
template <class D, class SRC, class DST>
__device__ __forceinline__ void stage_copy(DST dst, SRC src, int n, int t, int nthr) {
  for (int e0 = t; e0 < n; e0 += 8 * nthr) {
    D v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = (D)src[min(e0 + q * nthr, n - 1)];
#pragma unroll
    for (int q = 0; q < 8; ++q)
      if (e0 + q * nthr < n) dst[e0 + q * nthr] = v[q];
  }
}

template <class T, int NZ, bool ALL222>
// NZ = 0 is the point-smoother variant: no line-solve code (whose column
// registers would cap the workgroup at 512 lanes), and 1024 lanes.
// phase 0: the whole step list; 1: the steps before the coarse solve, then
// every level's u and f saved to its global arrays; 2: those restored, the
// steps after the coarse solve (run by k_coarse_wide in between).
__global__ __launch_bounds__(NZ == 0 ? 64 * kTailWavesPoint : 64 * kTailWaves) void k_tail(const DevLevel* __restrict__ Lt,
                                                          const DevXfer* __restrict__ X,
                                                          const DevTail* __restrict__ Tt,
                                                          LaunchList ll, int phase) {
  extern __shared__ unsigned char lds_raw[];
  __shared__ DevLevel Ls[kTailMaxLevels];
  const DevTail& tl = Tt[ll.items[blockIdx.x]];
  if (level_off(Lt[tl.lev[0]])) return;
  const int tid = threadIdx.y * 64 + threadIdx.x, nthr = 64 * blockDim.y;
  const int nl = tl.nlev;
  const sp<kS, unsigned char> base = (sp<kS, unsigned char>)lds_raw;
  auto U = [&](int d) { return (sp<kS, T>)(base + tl.lds_u[d]); };
  auto Fv = [&](int d) { return (sp<kS, T>)(base + tl.lds_f[d]); };
  auto CO = [&](int d) { return (sp<kS, const T>)(base + tl.lds_co[d]); };
  auto VOL = [&](int d) { return (sp<kS, const double>)(base + tl.lds_vol[d]); };
  if (tid < nl) Ls[tid] = Lt[tl.lev[tid]];
  // stage the tables of every tail level (one wave per level, in parallel),
  // the coarsest inverse when it fits, and the first level's fields
  const int wv = threadIdx.y, ln = threadIdx.x;
  for (int d = wv; d < nl; d += blockDim.y) {
    const DevLevel& G = Lt[tl.lev[d]];
    const int nco = 3 * (G.nx + G.ny + G.nz), nv = G.nx + G.ny + G.nz;
    stage_copy<T>((sp<kS, T>)(base + tl.lds_co[d]), coefs<T>(G), nco, ln, 64);
    if (d + 1 < nl) stage_copy<double>((sp<kS, double>)(base + tl.lds_vol[d]), gp(G.vol), nv, ln, 64);
  }
  if (tl.lds_minv >= 0) {
    const DevLevel& G = Lt[tl.lev[nl - 1]];
    stage_copy<T>((sp<kS, T>)(base + tl.lds_minv), gp(G.minvT), G.ncell * G.ncell, tid, nthr);
  }
  const DevLevel& G0 = Lt[tl.lev[0]];
  if (phase == 2) {
    for (int d = 0; d < nl; ++d) {
      const DevLevel& G = Lt[tl.lev[d]];
      stage_copy<T>(U(d), gfield<const T>((const void*)G.u), G.ncell, tid, nthr);
      if (d + 1 < nl) stage_copy<T>(Fv(d), gfield<const T>((const void*)G.f), G.ncell, tid, nthr);
    }
  } else {
    stage_copy<T>(Fv(0), gfield<const T>((const void*)G0.f), G0.ncell, tid, nthr);
    if (tl.copy_u_in) stage_copy<T>(U(0), gfield<const T>((const void*)G0.u), G0.ncell, tid, nthr);
  }
  __syncthreads();
  // the coarse solve's place in the step list (phases 1 and 2 stop or start there)
  int ci = 0;
  while (ci < tl.nsteps && (tl.steps[ci] & 7) != kStepCoarse) ++ci;
  const int st0 = phase == 2 ? ci + 1 : 0, st1 = phase == 1 ? ci : tl.nsteps;
  // one routine per step type, so that each element routine is instantiated
  // once (the kernel stays small enough for the instruction cache)
  for (int st = st0; st < st1; ++st) {
    const int code = tl.steps[st];
    const int type = code & 7, d = (code >> 3) & 15, par = (code >> 7) & 1, zg = (code >> 8) & 3;
    const DevLevel& L = Ls[d];
    if (type == kStepHalf) {
      if (NZ > 0 && tl.zline) {
        if constexpr (NZ > 0) {
          const int n = L.hx * L.ny;
          for (int e = tid; e < n; e += nthr) zline_column_n<T, NZ>(L, U(d), Fv(d), CO(d), par, zg, e);
        }
      } else {
        const int n = L.hx * L.ny * L.nz;
        for (int e = tid; e < n; e += nthr) rb_point_small<T>(L, U(d), Fv(d), CO(d), e, par, zg);
      }
    } else if (type == kStepRestrict) {
      const DevXfer x = X[tl.xf[d]];
      const DevLevel& C = Ls[d + 1];
      for (int e = tid; e < C.ncell; e += nthr) {
        if (ALL222) restrict_elem<T, 2, 2, 2>(L, U(d), Fv(d), CO(d), VOL(d), C, Fv(d + 1), e);
        else restrict_any<T>(L, U(d), Fv(d), CO(d), VOL(d), C, Fv(d + 1), x, e);
      }
    } else if (type == kStepCoarse) {
      if (tl.lds_minv >= 0) {
        const sp<kS, const T> M = (sp<kS, const T>)(base + tl.lds_minv);
        for (int r = tid; r < L.ncell; r += nthr) coarse_row<T>(L, U(d), Fv(d), M, r);
      } else {
        for (int r = tid; r < L.ncell; r += nthr) coarse_row<T>(L, U(d), Fv(d), gp(L.minvT), r);
      }
    } else if (type == kStepProlong) {
      const DevXfer x = X[tl.xf[d]];
      const DevLevel& C = Ls[d + 1];
      const int nd = prolong_duals(L, C, x);
      for (int e = tid; e < nd; e += nthr) {
        if (ALL222) prolong_dual<T, 2, 2, 2>(L, U(d), C, U(d + 1), x, e);
        else prolong_any<T>(L, U(d), C, U(d + 1), x, e);
      }
    } else {
      const sp<kS, T> u = U(d);
      for (int e = tid; e < L.ncell; e += nthr) u[e] = T(0);
    }
    __syncthreads();
  }
  if (phase == 1) {
    for (int d = 0; d < nl; ++d) {
      const DevLevel& G = Lt[tl.lev[d]];
      const sp<kG, T> gu = gfield<T>(G.u), gf = gfield<T>(G.f);
      const sp<kS, T> lu = U(d), lf = Fv(d);
      for (int e = tid; e < G.ncell; e += nthr) {
        gu[e] = lu[e];
        gf[e] = lf[e];
      }
    }
    return;
  }
  const sp<kG, T> gu = gfield<T>(G0.u);
  const sp<kS, T> lu = U(0);
  for (int e = tid; e < G0.ncell; e += nthr) gu[e] = lu[e];
}

// ---------------------------------------------------------------------------
// The coarse tail of an FP32 z-line V-cycle whose levels' columns share one
// matrix (DevLevel::zt), with walls in z, 2:2:2 transfers and smoothing on
// both ways on every level: the same sub-V-cycle as k_tail's, in one
// workgroup, but with the fields in LDS column by column (tail_stride), so
// that every step reads and writes four rows at a time:
//  - a half-sweep is one column per lane with the column's eliminated matrix
//    in scalar registers: no reciprocal, two dependent operations per row down
//    and one up (k_tail: a reciprocal per row and 130 four-byte LDS reads);
//  - the restriction forms the residuals of the colour-0 cells only, the
//    others being solved by the pre-smoothing (as k_restrict222), a task being
//    two coarse cells of a column;
//  - the prolongation corrects the colour-1 cells only, the others being
//    rewritten by the post-smoothing (as k_prolong), a task being eight rows
//    of a column;
//  - the coarsest level is solved by eigenvector transforms held in LDS.
// Bound by the steps' LDS and dependent latencies (one CU).  32x24x16 and
// below: 27 us against k_tail's 53; 24x24x24 and below: 32 against 45;
// 20x14x10 and 10x7x5: 17 against 44 (k_tail split around the dense product).
template <class T> using cst = const __attribute__((address_space(4))) T*;
template <class T> __device__ __forceinline__ cst<T> cp4(const T* p) { return (cst<T>)p; }

__device__ __forceinline__ float4& lds4(float* p) { return *reinterpret_cast<float4*>(p); }

// A smoothing phase, columns of 4*NC rows (rows past nz have zero table rows).
template <int NC>
__device__ __forceinline__ void line_smooth(float* __restrict__ lds, const LineLevel& L, cst<float> tabs,
                                            int sweeps, bool zero_first, int tid) {
  const int ncol = L.hx * L.ny, st = L.st, hx = L.hx;
  const cst<float> tab = tabs + L.col;
  for (int half = 0; half < 2 * sweeps; ++half) {
    const int parity = half & 1;
    const bool from_zero = zero_first && half == 0;
    if (half > 0) __syncthreads();
    for (int col = tid; col < ncol; col += 64 * kLineWaves) {
      const int j = gm_div(col, L.gmhx, L.gshx), m = col - j * hx;
      const int oth = parity ^ 1, r = (parity + j) & 1, i = 2 * m + r;
      float* const own = lds + L.u + ((j * 2 + parity) * hx + m) * st;
      const float* const fo = lds + L.f + ((j * 2 + parity) * hx + m) * st;
      float g[4 * NC];
#pragma unroll
      for (int q = 0; q < NC; ++q) {
        const float4 v = *reinterpret_cast<const float4*>(fo + 4 * q);
        g[4 * q] = v.x; g[4 * q + 1] = v.y; g[4 * q + 2] = v.z; g[4 * q + 3] = v.w;
      }
      if (!from_zero) {
        int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
        int mr = m + r;     if (mr >= hx) mr = 0;
        const int jm = (j == 0) ? L.ny - 1 : j - 1, jp = (j == L.ny - 1) ? 0 : j + 1;
        const float* const t = lds + L.xy;
        const float wxl = t[i], wxr = t[L.nx + i], wys = t[2 * L.nx + j], wyn = t[2 * L.nx + L.ny + j];
        const float* const ub = lds + L.u;
        const float* const xl = ub + ((j * 2 + oth) * hx + ml) * st;
        const float* const xr = ub + ((j * 2 + oth) * hx + mr) * st;
        const float* const ys = ub + ((jm * 2 + oth) * hx + m) * st;
        const float* const yn = ub + ((jp * 2 + oth) * hx + m) * st;
#pragma unroll
        for (int q = 0; q < NC; ++q) {
          const float4 a = *reinterpret_cast<const float4*>(xl + 4 * q);
          const float4 b = *reinterpret_cast<const float4*>(xr + 4 * q);
          const float4 c = *reinterpret_cast<const float4*>(ys + 4 * q);
          const float4 d = *reinterpret_cast<const float4*>(yn + 4 * q);
          g[4 * q] -= zline_nbr(wxl, wxr, wys, wyn, a.x, b.x, c.x, d.x);
          g[4 * q + 1] -= zline_nbr(wxl, wxr, wys, wyn, a.y, b.y, c.y, d.y);
          g[4 * q + 2] -= zline_nbr(wxl, wxr, wys, wyn, a.z, b.z, c.z, d.z);
          g[4 * q + 3] -= zline_nbr(wxl, wxr, wys, wyn, a.w, b.w, c.w, d.w);
        }
      }
      float y = 0.0f;
#pragma unroll
      for (int q = 0; q < 4 * NC; ++q) {
        y = fm(-tab[q], y, g[q]) * tab[kTailNz + q];
        g[q] = y;
      }
      float x = 0.0f;
#pragma unroll
      for (int q = 4 * NC - 1; q >= 0; --q) {
        x = fm(-tab[2 * kTailNz + q], x, g[q]);
        g[q] = x;
      }
#pragma unroll
      for (int q = 0; q < NC; ++q)
        lds4(own + 4 * q) = make_float4(g[4 * q], g[4 * q + 1], g[4 * q + 2], g[4 * q + 3]);
    }
  }
}

// Residuals of the colour-0 cells, weighted into the coarse right-hand side.
// Each 1-D weight is a cell's share of its coarse cell's width, formed in FP64.
// The x and y shares are 1/2 where columns share a matrix, so a cell's weight is
// its z share rounded once: 2e-8 of itself off, where the FP32 volume over the
// FP32 sum of volumes (restrict_elem) is 4e-8 to 9e-8.
__device__ __forceinline__ void line_restrict(float* __restrict__ lds, const LineLevel& F,
                                              const LineLevel& C, int tid) {
  const int ncc = C.nx * C.ny, kp = (C.nz + 1) >> 1, st = F.st, hx = F.hx;
  const float* const t = lds + F.xy;
  const float* const wnx = t + 2 * F.nx + 2 * F.ny;
  const float* const wny = wnx + F.nx;
  const float* const zt = lds + F.z;
  const int nzp = tail_rows(F.nz);
  for (int e = tid; e < ncc * kp; e += 64 * kLineWaves) {
    const int q0 = e / ncc, cc = e - q0 * ncc, J = gm_div(cc >> 1, C.gmhx, C.gshx), I = cc - J * C.nx;
    const int k0 = 4 * q0;
    const float4 za = *reinterpret_cast<const float4*>(zt + k0);
    const float4 ze = *reinterpret_cast<const float4*>(zt + nzp + k0);
    const float4 zd = *reinterpret_cast<const float4*>(zt + 2 * nzp + k0);
    const float4 zw = *reinterpret_cast<const float4*>(zt + 3 * nzp + k0);
    float lo = 0.0f, hi = 0.0f;
#pragma unroll
    for (int h = 0; h < 2; ++h) {                 // fine columns (2I, 2J) and (2I+1, 2J+1)
      const int i = 2 * I + h, j = 2 * J + h;
      const int jm = (j == 0) ? F.ny - 1 : j - 1, jp = (j == F.ny - 1) ? 0 : j + 1;
      const int ml = h ? I : (I == 0 ? hx - 1 : I - 1), mr = h ? (I + 1 == hx ? 0 : I + 1) : I;
      const float* const ub = lds + F.u;
      const int own = (j * 2 * hx + I) * st + k0;
      const float4 c4 = *reinterpret_cast<const float4*>(ub + own);
      const float um = ub[own - (k0 > 0 ? 1 : 0)], up = ub[own + (k0 + 4 < nzp ? 4 : 3)];
      const float4 f4 = *reinterpret_cast<const float4*>(lds + F.f + own);
      const float4 a = *reinterpret_cast<const float4*>(ub + ((j * 2 + 1) * hx + ml) * st + k0);
      const float4 b = *reinterpret_cast<const float4*>(ub + ((j * 2 + 1) * hx + mr) * st + k0);
      const float4 c = *reinterpret_cast<const float4*>(ub + ((jm * 2 + 1) * hx + I) * st + k0);
      const float4 d = *reinterpret_cast<const float4*>(ub + ((jp * 2 + 1) * hx + I) * st + k0);
      const float wxl = t[i], wxr = t[F.nx + i], wys = t[2 * F.nx + j], wyn = t[2 * F.nx + F.ny + j];
      auto res = [&](float fv, float xl, float xr, float ys, float yn, float dn, float upv, float cc0,
                     float A, float E, float D) {
        return fv - fm(D, cc0, fm(E, upv, fm(A, dn, zline_nbr(wxl, wxr, wys, wyn, xl, xr, ys, yn))));
      };
      const float r0 = res(f4.x, a.x, b.x, c.x, d.x, um, c4.y, c4.x, za.x, ze.x, zd.x);
      const float r1 = res(f4.y, a.y, b.y, c.y, d.y, c4.x, c4.z, c4.y, za.y, ze.y, zd.y);
      const float r2 = res(f4.z, a.z, b.z, c.z, d.z, c4.y, c4.w, c4.z, za.z, ze.z, zd.z);
      const float r3 = res(f4.w, a.w, b.w, c.w, d.w, c4.z, up, c4.w, za.w, ze.w, zd.w);
      const float wxy = wnx[i] * wny[j];
      lo = fm(wxy, fm(zw.y, r1, zw.x * r0), lo);
      hi = fm(wxy, fm(zw.w, r3, zw.z * r2), hi);
    }
    float* const fc = lds + C.f + ((J * 2 + ((I + J) & 1)) * C.hx + (I >> 1)) * C.st + 2 * q0;
    *reinterpret_cast<float2*>(fc) = make_float2(lo, hi);
  }
}

// Trilinear prolongation-add to the colour-1 cells (at a Dirichlet wall the
// correction vanishes at the ghost, at a Neumann wall it is copied).
__device__ __forceinline__ void line_prolong(float* __restrict__ lds, const LineLevel& F,
                                             const LineLevel& C, int tid) {
  const int bx0 = F.bc[0], bx1 = F.bc[1], by0 = F.bc[2], by1 = F.bc[3], bz0 = F.bc[4], bz1 = F.bc[5];
  const int ncol = F.hx * F.ny, nch = (C.nz + 3) >> 2, hx = F.hx, nzc = C.nz;
  for (int e = tid; e < ncol * nch; e += 64 * kLineWaves) {
    const int ch = e / ncol, col = e - ch * ncol;
    const int j = gm_div(col, F.gmhx, F.gshx), m = col - j * hx;
    const int r = (1 + j) & 1, I = m, J = j >> 1, K0 = 4 * ch;
    int I2 = r ? I + 1 : I - 1, J2 = (j & 1) ? J + 1 : J - 1;
    float fx = 1.0f, fy = 1.0f;
    if (I2 < 0) { if (F.px) I2 = C.nx - 1; else { I2 = 0; if (bx0 == 2) fx = 0.0f; } }
    if (I2 >= C.nx) { if (F.px) I2 = 0; else { I2 = C.nx - 1; if (bx1 == 2) fx = 0.0f; } }
    if (J2 < 0) { if (F.py) J2 = C.ny - 1; else { J2 = 0; if (by0 == 2) fy = 0.0f; } }
    if (J2 >= C.ny) { if (F.py) J2 = 0; else { J2 = C.ny - 1; if (by1 == 2) fy = 0.0f; } }
    const float* const ub = lds + C.u;
    auto at = [&](int a, int b) { return ub + ((b * 2 + ((a + b) & 1)) * C.hx + (a >> 1)) * C.st; };
    const float* const c0 = at(I, J);
    const float* const c1 = at(I2, J);
    const float* const c2 = at(I, J2);
    const float* const c3 = at(I2, J2);
    const float w0 = 0.5625f, w1 = 0.1875f * fx, w2 = 0.1875f * fy, w3 = 0.0625f * fx * fy;
    auto mix = [&](float a, float b, float c, float d) { return fm(w3, d, fm(w2, c, fm(w1, b, w0 * a))); };
    // coarse rows K0-1 .. K0+4
    float t[6];
    const int kb = max(K0 - 1, 0), ka = min(K0 + 4, nzc - 1);
    const float4 a4 = *reinterpret_cast<const float4*>(c0 + K0), b4 = *reinterpret_cast<const float4*>(c1 + K0);
    const float4 d4 = *reinterpret_cast<const float4*>(c2 + K0), e4 = *reinterpret_cast<const float4*>(c3 + K0);
    t[0] = mix(c0[kb], c1[kb], c2[kb], c3[kb]);
    t[1] = mix(a4.x, b4.x, d4.x, e4.x);
    t[2] = mix(a4.y, b4.y, d4.y, e4.y);
    t[3] = mix(a4.z, b4.z, d4.z, e4.z);
    t[4] = mix(a4.w, b4.w, d4.w, e4.w);
    t[5] = mix(c0[ka], c1[ka], c2[ka], c3[ka]);
    if (K0 == 0) t[0] = bz0 == 2 ? 0.0f : t[1];
#pragma unroll
    for (int q = 2; q < 6; ++q)
      if (K0 - 1 + q >= nzc) t[q] = bz1 == 2 ? 0.0f : t[q - 1];
    float* const uo = lds + F.u + ((j * 2 + 1) * hx + m) * F.st + 8 * ch;
#pragma unroll
    for (int h = 0; h < 2; ++h) {                  // fine rows 8ch + 4h ..: coarse rows K0+2h, +1
      if (K0 + 2 * h >= nzc) break;
      float4 v = lds4(uo + 4 * h);
      v.x += fm(0.75f, t[1 + 2 * h], 0.25f * t[2 * h]);
      v.y += fm(0.75f, t[1 + 2 * h], 0.25f * t[2 + 2 * h]);
      v.z += fm(0.75f, t[2 + 2 * h], 0.25f * t[1 + 2 * h]);
      v.w += fm(0.75f, t[2 + 2 * h], 0.25f * t[3 + 2 * h]);
      lds4(uo + 4 * h) = v;
    }
  }
}

// Separable solve of the coarsest level (direct_setup's tables in LDS, FP64):
// transforms in x, y and z, the inverse eigenvalue sums, and back, one value
// per lane and stage.  (Multiplying by the dense inverse took 5 us at 192
// cells and 14 at 350: one CU reads it at its L2 rate.)
__device__ __forceinline__ void line_coarse(float* __restrict__ lds, const LineLevel& L, int m0, int w0,
                                            int tid) {
  const int nx = L.nx, ny = L.ny, nz = L.nz, nxy = nx * ny, n = nxy * nz;
  const double* const xi = reinterpret_cast<const double*>(lds + m0);
  const double *const xv = xi + nx * nx, *const yi = xv + nx * nx, *const yv = yi + ny * ny;
  const double *const zi = yv + ny * ny, *const zv = zi + nz * nz, *const inv = zv + nz * nz;
  double* const A = reinterpret_cast<double*>(lds + w0);
  double* const B = A + n;
  const bool on = tid < n;
  const int k = tid / nxy, q = tid - k * nxy, j = q / nx, i = q - j * nx;
  const int col = ((j * 2 + ((i + j) & 1)) * L.hx + (i >> 1)) * L.st + k;
  // sum over c < len of a[c * sa] * b[c * sb]
  auto dot = [](const double* a, int sa, const double* b, int sb, int len) {
    double s = 0.0;
#pragma unroll 4
    for (int c = 0; c < len; ++c) s = fm(a[c * sa], b[c * sb], s);
    return s;
  };
  if (on) A[tid] = (double)lds[L.f + col];
  __syncthreads();
  if (on) B[tid] = dot(A + tid - i, 1, xi + i, nx, nx);
  __syncthreads();
  if (on) A[tid] = dot(yi + j * ny, 1, B + k * nxy + i, nx, ny);
  __syncthreads();
  if (on) B[tid] = dot(zi + k * nz, 1, A + q, nxy, nz) * inv[tid];
  __syncthreads();
  if (on) A[tid] = dot(zv + k * nz, 1, B + q, nxy, nz);
  __syncthreads();
  if (on) B[tid] = dot(yv + j * ny, 1, A + k * nxy + i, nx, ny);
  __syncthreads();
  if (on) lds[L.u + col] = (float)dot(B + tid - i, 1, xv + i, nx, nx);
}

__global__ __launch_bounds__(64 * kLineWaves) void k_tail_line(const DevLevel* __restrict__ Lt,
                                                                const DevTail* __restrict__ Tt, LIST_PARAMS,
                                                                LaunchList ll) {
  extern __shared__ float lds[];
  const int tid = threadIdx.x;
  constexpr int nthr = 64 * kLineWaves;
  const cst<DevTail> tl = cp4(Tt + (ln == 1 ? li0 : ll.items[blockIdx.x]));
  const int nst = tl->lin_nsteps, words = tl->tab_words;
  const float* tabg = tl->tab;
  const LevelHead H0 = level_head(Lt[tl->lev[0]]);
  if (H0.stop) return;
  auto level = [&](int d) {
    const auto* l = &tl->lin[d];
    return LineLevel{l->nx, l->ny, l->nz, l->hx, l->st, l->px, l->py, l->gmhx, l->gshx, l->u, l->f, l->xy,
                     l->z, l->col, {l->bc[0], l->bc[1], l->bc[2], l->bc[3], l->bc[4], l->bc[5]}};
  };
  // the first level's right-hand side on its way while the LDS is cleared (the
  // rows past nz have to be finite) and the tables are copied
  constexpr int U = 16;
  const int plane = H0.nx * H0.ny, n0 = H0.ncell;
  const sp<kG, const float> f0 = gfield<const float>((const void*)H0.f);
  float fv[U];
#pragma unroll
  for (int q = 0; q < U; ++q) fv[q] = f0[min(tid + q * nthr, n0 - 1)];
  const int end = tl->lin_c;
  for (int e = words + 4 * tid; e < end; e += 4 * nthr) lds4(lds + e) = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int e = tid; e < words; e += nthr) lds[e] = gp(tabg)[e];
  __syncthreads();
  const LineLevel L0 = level(0);
  {
    const int dk = nthr / plane, dc = nthr - dk * plane;
    int k = tid / plane, c = tid - k * plane;
    for (int e0 = tid; e0 < n0; e0 += U * nthr) {
#pragma unroll
      for (int q = 0; q < U; ++q) {
        if (e0 + q * nthr < n0) lds[L0.f + c * L0.st + k] = fv[q];
        c += dc;
        k += dk;
        if (c >= plane) { c -= plane; ++k; }
      }
      if (e0 + U * nthr < n0) {
#pragma unroll
        for (int q = 0; q < U; ++q) fv[q] = f0[min(e0 + (U + q) * nthr, n0 - 1)];
      }
    }
  }
  __syncthreads();
  int code = tl->lin_steps[0];
  for (int st = 0; st < nst; ++st) {
    const int type = code & 7, d = (code >> 3) & 15, zf = (code >> 7) & 1, sweeps = code >> 8;
    code = tl->lin_steps[st + 1];                 // (one past the last is allocated)
    const LineLevel L = level(d);
    if (type == kStepHalf) {
      const cst<float> tabs = cp4(tabg);
      switch (tail_rows(L.nz) >> 2) {
        case 1: line_smooth<1>(lds, L, tabs, sweeps, zf, tid); break;
        case 2: line_smooth<2>(lds, L, tabs, sweeps, zf, tid); break;
        case 3: line_smooth<3>(lds, L, tabs, sweeps, zf, tid); break;
        case 4: line_smooth<4>(lds, L, tabs, sweeps, zf, tid); break;
        case 5: line_smooth<5>(lds, L, tabs, sweeps, zf, tid); break;
        case 6: line_smooth<6>(lds, L, tabs, sweeps, zf, tid); break;
        case 7: line_smooth<7>(lds, L, tabs, sweeps, zf, tid); break;
        default: line_smooth<8>(lds, L, tabs, sweeps, zf, tid); break;
      }
    } else if (type == kStepRestrict) {
      line_restrict(lds, L, level(d + 1), tid);
    } else if (type == kStepProlong) {
      line_prolong(lds, L, level(d + 1), tid);
    } else {
      line_coarse(lds, L, tl->lin_m, end, tid);
    }
    __syncthreads();
  }
  const sp<kG, float> u0 = gfield<float>(H0.u);
  const int dk = nthr / plane, dc = nthr - dk * plane;
  int k = tid / plane, c = tid - k * plane;
  for (int e = tid; e < n0; e += nthr) {
    u0[e] = lds[L0.u + c * L0.st + k];
    c += dc;
    k += dk;
    if (c >= plane) { c -= plane; ++k; }
  }
}

// Coarsest level of a split tail: u = M f with the row-major (pseudo-)inverse,
// one wave per row (FP64 partial sums over the lane's columns in a fixed
// order, then a fixed butterfly), so a large inverse is read by the whole
// device rather than by one workgroup.
template <class T>
__global__ __launch_bounds__(kBlock) void k_coarse_wide(const DevLevel* __restrict__ Lt, LaunchList ll) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  if (level_off(L)) return;
  const int n = L.ncell;
  const int r = (b - ll.prefix[t]) * (kBlock / 64) + (int)(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  if (r >= n) return;
  const sp<kG, const double> M = gp(L.minv) + (size_t)r * n;
  const sp<kG, const T> f = gfield<const T>((const void*)L.f);
  double acc[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  int s = lane;
  for (; s + 7 * 64 < n; s += 8 * 64) {
    double m[8], fv[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      m[q] = M[s + q * 64];
      fv[q] = (double)f[s + q * 64];
    }
#pragma unroll
    for (int q = 0; q < 8; ++q) acc[q] += m[q] * fv[q];
  }
  for (int q = 0; s < n; s += 64, ++q) acc[q & 7] += M[s] * (double)f[s];
  double sum = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
  sum = wave_sum(sum);
  if (lane == 0) gfield<T>(L.u)[r] = (T)sum;
}

// ---------------------------------------------------------------------------
// FP64 finest-level kernels.
// Each thread handles kFinePer cells e = e0 + s*kBlock (coalesced), keeps
// running maxima, and the block writes one partial per value; the finalize
// kernel folds the partials per item.
template <int NV, class F>
__device__ __forceinline__ void fine_loop(const DevLevel& L, int lb, double* __restrict__ partial,
                                          int b, F&& body) {
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.0;
  const int e0 = lb * kBlock * kFinePer + threadIdx.x;
#pragma unroll
  for (int s = 0; s < kFinePer; ++s) {
    const int e = e0 + s * kBlock;
    if (e < L.ncell) body(e, v);
  }
  block_reduce_store<NV, false>(v, partial + (size_t)b * NV);
}

// {max|u - u2|, max|u|}
__global__ __launch_bounds__(kBlock) void k_change_max(const DevLevel* __restrict__ Lt,
                                                       LaunchList ll, double* __restrict__ partial) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  if (level_off(L)) return;
  const auto u = gfield<const double>((const void*)L.u);
  const auto u2 = gfield<const double>((const void*)L.u2);
  fine_loop<2>(L, b - ll.prefix[t], partial, b, [&](int e, double* v) {
    v[0] = amax(v[0], u[e] - u2[e]);
    v[1] = amax(v[1], u[e]);
  });
}

// FP64 finest-level stencil kernels, marching in z.  A thread owns one
// position col = (j*2 + colour)*hx + m of a plane and walks D.mk planes,
// keeping the centre values at k-1, k, k+1 in registers: every value of the
// iterate is read from memory once per slab (plus one halo plane at each
// slab end), the four in-plane neighbours come from the cache, and the
// index arithmetic is done once per thread instead of once per cell.
//   kResMax:        {max|b - A u|, max|b|}
//   kDefect32:      r = b - A u -> FP32 right-hand side of the correction
//                   level; {max|r|, max|b|}
//   kCorrDefect32:  p_out = p_in + e, r = b - A p_out -> FP32; p_in is never
//                   written, so neighbouring threads read consistent values;
//                   {max|r|, max|e|, max|p_out|}
// The stencil sums are ordered as in offsum/diag_at.
enum { kResMax = 0, kDefect32 = 1, kCorrDefect32 = 2 };
#ifndef AMG_FINE_DEPTH
#define AMG_FINE_DEPTH 2
#endif
constexpr int kFineDepth = AMG_FINE_DEPTH;

// The marching loop of one thread.  Every field pointer is a __restrict__
// parameter (the outputs never alias the inputs), and the loop is
// software-pipelined by hand: the loads of plane k+1 are issued before plane
// k is computed and stored, so a thread keeps two planes of loads in flight.
// In mixed mode the centre column's p and e are carried separately (e for
// the correction norm).
template <int MODE, int NV, bool SHIFT>
__device__ __forceinline__ void fine_march(sp<kG, const double> __restrict__ u,
                                           sp<kG, const float> __restrict__ ev,
                                           sp<kG, double> __restrict__ f, double cs,
                                           sp<kG, double> __restrict__ pout,
                                           sp<kG, float> __restrict__ r32,
                                           sp<kG, const double> __restrict__ cz, int nz, int plane,
                                           int col, int oxm, int oxp, int oym, int oyp, double wxm,
                                           double wxp, double wym, double wyp, double dxy_y,
                                           double dxy_x, int k0, int k1, double (&v)[NV]) {
  constexpr bool MIXED = MODE == kCorrDefect32;
  // loads of plane k: the four in-plane neighbours, b, and the centre at k+1
  struct Plane {
    double xm, xp, ym, yp, fb, pu;
    float xme, xpe, yme, ype, pe;
  };
  // rows are addressed as a plane base plus per-lane byte offsets that are
  // the same in every plane (no vector address arithmetic per load)
  const unsigned dxm = (unsigned)oxm * 8u, dxp = (unsigned)oxp * 8u, dym = (unsigned)oym * 8u,
                 dyp = (unsigned)oyp * 8u, dc = (unsigned)col * 8u;
  const unsigned sxm = (unsigned)oxm * 4u, sxp = (unsigned)oxp * 4u, sym = (unsigned)oym * 4u,
                 syp = (unsigned)oyp * 4u, sc = (unsigned)col * 4u;
  auto load = [&](int k) {
    Plane q;
    const int pb = k * plane;
    const int kp = (k == nz - 1) ? 0 : k + 1;
    const sp<kG, const double> ur = u + pb;
    q.xm = ld_row<double>(ur, dxm); q.xp = ld_row<double>(ur, dxp);
    q.ym = ld_row<double>(ur, dym); q.yp = ld_row<double>(ur, dyp);
    // cs: the compatibility shift of b, subtracted as b is loaded (the
    // first defect; the mixed step, which keeps b as ingested).  The mixed
    // step reads b once per cell and nothing else reads it during the step:
    // a non-temporal load (it was measured slower in the FP64 residual)
    const sp<kG, const double> fr = (sp<kG, const double>)(f + pb);
    q.fb = (MIXED ? ld_row_nt<double>(fr, dc) : ld_row<double>(fr, dc)) - cs;
    q.pu = ld_row<double>(u + kp * plane, dc);
    if constexpr (MIXED) {
      const sp<kG, const float> er = ev + pb;
      q.xme = ld_row<float>(er, sxm); q.xpe = ld_row<float>(er, sxp);
      q.yme = ld_row<float>(er, sym); q.ype = ld_row<float>(er, syp);
      q.pe = ld_row<float>(ev + kp * plane, sc);
    } else {
      q.xme = q.xpe = q.yme = q.ype = q.pe = 0.0f;
    }
    return q;
  };
  auto sum = [&](double a, float b) -> double {
    if constexpr (MIXED) return a + (double)b;
    else return a;
  };
  const int km0 = (k0 == 0) ? nz - 1 : k0 - 1;
  double vm = sum(u[km0 * plane + col], MIXED ? ev[km0 * plane + col] : 0.0f);
  const float ec0 = MIXED ? ev[k0 * plane + col] : 0.0f;
  double vc = sum(u[k0 * plane + col], ec0);
  float ec = ec0;
  auto step = [&](int k, const Plane& cur) {
    const int pbk = k * plane;
    const double vp = sum(cur.pu, cur.pe);
    // explicit fma: a residual is the same bits whatever slab it is in
    double s = fm(wxp, sum(cur.xp, cur.xpe), wxm * sum(cur.xm, cur.xme));
    s = fm(wym, sum(cur.ym, cur.yme), s);
    s = fm(wyp, sum(cur.yp, cur.ype), s);
    s = fm(cz[k], vm, s);
    s = fm(cz[nz + k], vp, s);
    const double diag = (cz[2 * nz + k] + dxy_y) + dxy_x;
    const double res = cur.fb - fm(diag, vc, s);
    // the shifted b (FP64: the V-cycle's finest right-hand side) and the
    // FP32 defect are read by later kernels only
    if constexpr (SHIFT && MODE == kResMax) st_row_nt<double>(f + pbk, dc, cur.fb);
    if constexpr (MODE == kCorrDefect32) {
      // the new p is read in the next cycle and the FP32 defect by the next
      // V-cycle's first sweep, both after many more bytes than the L2 holds
      st_row_nt<double>(pout + pbk, dc, vc);
      st_row_nt<float>(r32 + pbk, sc, (float)res);
      v[0] = amax(v[0], res);
      v[1] = amax(v[1], (double)ec);
      v[2] = amax(v[2], vc);
    } else {
      if constexpr (MODE == kDefect32) st_row_nt<float>(r32 + pbk, sc, (float)res);
      v[0] = amax(v[0], res);
      v[1] = amax(v[1], cur.fb);
    }
    vm = vc;
    vc = vp;
    ec = cur.pe;
  };
  // a ring of kFineDepth plane buffers, indexed statically (the loop is
  // unrolled by the ring size, so no register copies): the loads of plane
  // k + kFineDepth - 1 are issued before plane k is computed, and the
  // prefetch is unconditional (past the slab it reloads the last plane).
  // Loads complete in issue order, so the wait before a plane's arithmetic
  // leaves the kFineDepth - 1 younger planes in flight.
  // A full slab is unrolled completely and has no branch, so the ring needs
  // no register copies at a loop back edge (they would wait for the loads in
  // flight) and no load is sunk past a branch toward its use.
  constexpr int D = kFineDepth;
  auto slab = [&](auto planes) {
    constexpr int K = decltype(planes)::value;
    Plane R[D];
#pragma unroll
    for (int s = 0; s < D - 1; ++s) R[s] = load(k0 + s);
#pragma unroll
    for (int s = 0; s < K; ++s) {
      if (s + D - 1 < K) R[(s + D - 1) % D] = load(k0 + s + D - 1);
      // keep the prefetch ahead of the arithmetic: the scheduler would
      // otherwise move the loads toward their use
      __builtin_amdgcn_sched_barrier(0);
      step(k0 + s, R[s % D]);
    }
  };
  if (k1 - k0 == kMarchK) {
    slab(std::integral_constant<int, kMarchK>());
  } else if (k1 - k0 == 4) {
    slab(std::integral_constant<int, 4>());
  } else if (k1 - k0 == 2) {
    slab(std::integral_constant<int, 2>());
  } else {
    // other lengths: a short last slab
    Plane a = load(k0);
    for (int k = k0; k < k1; ++k) {
      const Plane n = load(min(k + 1, k1 - 1));
      step(k, a);
      a = n;
    }
  }
}

// SHIFT: the first defect of a solve, which takes the compatibility shift
// of a singular instance from csum (sum V b per item); FP64 writes the
// shifted b back, mixed keeps b and records the shift in the instance's
// bshift word, which its outer steps subtract as they load b.
template <int MODE, bool SHIFT>
__global__ __launch_bounds__(kBlock) void k_fine(DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                 const double* __restrict__ csum,
                                                 double* __restrict__ partial, LaunchList ll) {
  constexpr int NV = MODE == kCorrDefect32 ? 3 : 2;
  const Work wk = work_item(ln, lnb, li0, ll);
  const int b = wk.b, t = wk.t;
  const DevLevel& D = Lt[wk.idx];
  // the FP32 finest level's fields (mixed; an FP64 solve has none)
  const float* e32 = D.e32;
  float* r32 = D.r32;
  double bshift = D.bshift, vsum = D.vsum;
  int nullsp = D.nullsp, mk = D.mk;
  pin_s(e32, r32, bshift, vsum, nullsp, mk);
  const LevelHead L = level_head(D);
  if (level_off(L)) return;
  // the first cycle of a pair: no correction (its gate reads no norms)
  if (MODE == kCorrDefect32 && L.skipc) return;
  const int hx = L.hx, nx = L.nx, ny = L.ny, nz = L.nz;
  // the current FP64 pressure and its ping-pong partner
  const void* pin = L.pcur ? L.u2 : L.u;
  void* pout = L.pcur ? L.u : L.u2;
  const int plane = 2 * hx * ny;
  const int ncb = (plane + kBlock - 1) / kBlock;
  const int lb = wk.lb;
  const int bk = lb / ncb, bc = lb - bk * ncb;
  const int col = bc * kBlock + threadIdx.x;
  const int k0 = bk * mk, k1 = min(k0 + mk, nz);
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.0;
  if (col < plane) {
    const int row = gm_div(col, L.gmhx, L.gshx), m = col - row * hx, c = row & 1, j = row >> 1;
    const int i = 2 * m + ((c + j) & 1), r = i & 1, oth = c ^ 1;
    int ml = m - 1 + r; if (ml < 0) ml = hx - 1;
    int mr = m + r;     if (mr >= hx) mr = 0;
    const int jm = (j == 0) ? ny - 1 : j - 1, jp = (j == ny - 1) ? 0 : j + 1;
    const auto co = gp(L.co64);
    const auto cy = co + 3 * nx;
    const auto cz = cy + 3 * ny;
    const double cs = MODE == kCorrDefect32 ? bshift : (SHIFT && nullsp) ? csum[t] / vsum : 0.0;
    if (SHIFT && MODE == kDefect32 && lb == 0 && threadIdx.x == 0) Lt[wk.idx].bshift = cs;
    fine_march<MODE, NV, SHIFT>(gfield<const double>(pin),
                         gp(e32), gfield<double>(L.f), cs,
                         gfield<double>(pout),
                         gp(r32), cz, nz, plane, col, (j * 2 + oth) * hx + ml,
                         (j * 2 + oth) * hx + mr, (jm * 2 + oth) * hx + m, (jp * 2 + oth) * hx + m,
                         co[i], co[nx + i], cy[j], cy[ny + j], cy[2 * ny + j], co[2 * nx + i], k0, k1, v);
  }
  block_reduce_store<NV, false>(v, partial + (size_t)b * NV);
}

// State words an instance's levels take at the end of a cycle (a negative
// value leaves that word as it is; pflip toggles pcur).
struct GateWords {
  int stop, warm, skipc, pflip;
};

// Writes w on the levels of instance inst among entries l0, l0+step, ...
// of the table (the threads of a block split the table between them).  The
// entries' instance numbers are read eight at a time before any write, so
// a walk pays a memory round trip per eight entries, not per entry.
__device__ void set_words(DevLevel* Lt, int nL, int inst, GateWords w, int l0, int step) {
  constexpr int U = 8;
  for (int lb = l0; lb < nL; lb += U * step) {
    int iv[U];
#pragma unroll
    for (int j = 0; j < U; ++j) iv[j] = lb + j * step < nL ? Lt[lb + j * step].inst : -1;
#pragma unroll
    for (int j = 0; j < U; ++j) {
      if (iv[j] != inst) continue;
      DevLevel& d = Lt[lb + j * step];
      if (w.stop >= 0) d.stop = w.stop;
      if (w.warm >= 0) d.warm = w.warm;
      if (w.skipc >= 0) d.skipc = w.skipc;
      if (w.pflip) d.pcur ^= 1;
    }
  }
}

// What a gate check reads besides the norms of its own fold: the gate, the
// instance's state words and the norms in memory.  k_finalize loads it
// before it folds, so these round trips overlap the fold's.
struct GatePre {
  double o[4], oc[2];
  double bnorm, tol, rprev;
  int gstop, cycles, n, maxcy, rule, fp64, report, gpair, skipc, warm;
  int gslot, inst;
};
__device__ __forceinline__ GatePre gate_pre(const ItemGate* g, const double* out, const double* outc,
                                            const DevLevel& L, int slot, int inst) {
  GatePre P;
  for (int q = 0; q < 4; ++q) P.o[q] = out[q];
  P.oc[0] = outc[0];
  P.oc[1] = outc[1];
  P.gstop = g->stop;
  P.cycles = g->cycles;
  P.n = g->count;
  P.maxcy = g->maxcy;
  P.rule = g->rule;
  P.fp64 = g->fp64;
  P.report = g->report;
  P.gpair = g->pair;
  P.bnorm = g->bnorm;
  P.tol = g->tol;
  P.rprev = g->rprev;
  P.skipc = L.skipc;
  P.warm = L.warm;
  P.gslot = slot;
  P.inst = inst;
  return P;
}

// End of a gated cycle of one instance (its item's level is the FP64
// finest): the first cycle of a pair only hands over to the
// second; otherwise the correction's norms are recorded and the stop rule
// of the host's norm step (Context::post_norms) applied to them with the
// same double operations, so the host's replay reaches the same decision;
// then the next cycle is planned (paired or not).  Returns the state words
// the instance's levels take.
// P holds what it reads (gate_pre, with the norms of the calling fold put
// in); only stores remain here, and only the thread with `keep` makes them:
// the others take the same words from the same values.
__device__ __forceinline__ GateWords item_gate_check(ItemGate* g, const GatePre& P, bool keep) {
  const double* o = P.o;
  const double* oc = P.oc;
  const int gstop = P.gstop, cycles = P.cycles + 1, n = P.n, maxcy = P.maxcy;
  const int rule = P.rule, fp64 = P.fp64, report = P.report, gpair = P.gpair;
  const double bnorm = P.bnorm, tol = P.tol, rprev = P.rprev;
  const int skipc = P.skipc, warm = P.warm;
  if (gstop) return {-1, -1, -1, 0};
  if (keep) g->cycles = cycles;
  if (skipc) return {-1, 1, 0, 0};
  const int m = warm ? 2 : 1;
  if (keep) {
    double* h = g->hist[n % kItemRing];
    for (int q = 0; q < 4; ++q) h[q] = o[q];
    h[4] = report ? oc[0] : 0.0;
    h[5] = report ? oc[1] : 0.0;
    g->hcyc[n % kItemRing] = m;
    g->count = n + 1;
  }
  const double rmax = o[0];
  double relmax;
  if (fp64) relmax = report ? (oc[1] > 0.0 ? oc[0] / oc[1] : 0.0) : __longlong_as_double(0x7ff8000000000000ll);
  else relmax = o[2] > 0.0 ? o[1] / o[2] : 0.0;
  const double relres = bnorm > 0.0 ? rmax / bnorm : rmax;
  int stop = 0;
  if (!isfinite(rmax)) {
    stop = 1;
  } else {
    const double crit = (rule == AMG_STOP_RELMAX) ? relmax : relres;
    if (crit <= tol || cycles >= maxcy) stop = 1;
  }
  const bool pair = !stop && gpair && cycles + 2 <= maxcy && pair_next(relres, rprev, m, tol);
  if (keep) {
    g->rprev = relres;
    g->stop = stop;
  }
  return {stop, 0, pair ? 1 : 0, fp64 ? 0 : 1};
}

// One thread per item: the gate of a starting solve, from its first defect
// (the decisions the host's replay, Context::absorb_gate, takes with the
// same operations), and the plan of its first cycle.
__global__ void k_gate_init(LaunchList ll, const double* __restrict__ out, ItemGate* ig,
                            DevLevel* Lt, int nL, int maxcy, int rule, double tol, int report) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= ll.nitems) return;
  const DevLevel& L = Lt[ll.items[t]];
  ItemGate* g = ig + L.gslot;
  const double r = out[(size_t)t * 4], b = out[(size_t)t * 4 + 1];
  const int fp64 = L.link < 0;
  g->count = 0;
  g->cycles = 0;
  g->maxcy = maxcy;
  g->rule = rule;
  g->fp64 = fp64;
  g->report = fp64 && report;
  g->pair = L.pairok;
  g->tol = tol;
  g->bnorm = b;
  g->res0 = b > 0.0 ? r / b : r;
  g->rprev = g->res0;
  int stop = 0;
  if (!isfinite(r) || !isfinite(b)) stop = 1;
  else if (rule == AMG_STOP_RESIDUAL && (b == 0.0 || g->res0 <= tol)) stop = 1;
  g->stop = stop;
  const bool pair = !stop && g->pair && maxcy >= 2 && g->res0 * kPairRho0 > tol;
  set_words(Lt, nL, L.inst, {stop, 0, pair ? 1 : 0, 0}, 0, 1);
}

// One block per item: thread t folds partials b0+t, b0+t+kFinBlock, ... in
// order, then a fixed-shape tree combines the threads (deterministic).  With
// per-instance gates, the block then ends its item's cycle and writes the
// resulting state words, one table entry per thread.
//
// The kernel is one chain of waits: a store before a barrier is one (the
// barrier waits until it has arrived), a load after it another.  So the gate
// and the entries' own words are loaded before the fold, all values meet at
// one barrier, the waves' values are read from LDS together (a loop of
// read-and-fold costs 0.8 us per value), every thread with a table entry then
// takes the decision for itself, and all stores come last.  4096 partials of
// three values: 6.3 us (9.7 with two barriers per value, the decision passed
// on by another and pcur read to toggle it); 1024: 5.7 (8.9); 64: 4.6 (6.3).
// SUM: the values are summed; otherwise they are magnitudes (or NaN) and the
// largest is taken.
constexpr int kFinBlock = 1024;
template <bool SUM>
__global__ __launch_bounds__(kFinBlock) void k_finalize(LIST_PARAMS, int nvals,
                                                        const double* __restrict__ partial,
                                                        double* __restrict__ out, int ostride,
                                                        GateArgs ga, LaunchList ll) {
  constexpr int kWaves = kFinBlock / 64;
  __shared__ double sm[4][kWaves];
  const int t = blockIdx.x;
  const bool one = ln == 1;
  const int b0 = one ? 0 : ll.prefix[t], b1 = one ? lnb : ll.prefix[t + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // the threads that see the folded values: one per table entry with gates
  const int nsee = ga.ig ? max(64, ga.nL) : 64;
  // a launch of one item knows its gate's place; a thread's first entry (its
  // instance never changes on the device, its pcur only here)
  GatePre gpre;
  int inst0 = -1, pcur0 = 0;
  if (ga.ig && (int)threadIdx.x < nsee) {
    if ((int)threadIdx.x < ga.nL) {
      inst0 = ga.Lt[threadIdx.x].inst;
      pcur0 = ga.Lt[threadIdx.x].pcur;
    }
    const DevLevel& L = ga.Lt[one ? li0 : ll.items[t]];
    const int slot = one ? ga.slot : L.gslot, inst = one ? ga.inst : L.inst;
    gpre = gate_pre(ga.ig + slot, ga.out + (size_t)t * 4, ga.outc + (size_t)t * 2, L, slot, inst);
  }
  // one pass over the partials for every value (nvals <= 4), kFinU
  // partials per thread and round: their loads (clamped into the item, so
  // unconditional) are issued before they are folded, in order
  constexpr int kFinU = 4;
  double acc[4] = {0.0, 0.0, 0.0, 0.0};
  for (int b = b0 + threadIdx.x; b < b1; b += kFinBlock * kFinU) {
    double x[kFinU][4];
#pragma unroll
    for (int r = 0; r < kFinU; ++r) {
      const int bb = min(b + r * kFinBlock, b1 - 1);
#pragma unroll
      for (int q = 0; q < 4; ++q) x[r][q] = partial[(size_t)bb * nvals + min(q, nvals - 1)];
    }
#pragma unroll
    for (int r = 0; r < kFinU; ++r) {
      if (b + r * kFinBlock < b1) {
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < nvals) acc[q] = SUM ? acc[q] + x[r][q] : amax(acc[q], x[r][q]);
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= nvals) break;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const double o = __shfl_xor(acc[q], off, 64);
      acc[q] = SUM ? acc[q] + o : amax(acc[q], o);
    }
    if (lane == 0) sm[q][w] = acc[q];
  }
  __syncthreads();
  if ((int)threadIdx.x >= nsee) return;
  double fr[4];   // the folded values
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= nvals) break;
    double x[kWaves];
#pragma unroll
    for (int i = 0; i < kWaves; ++i) x[i] = sm[q][i];
#pragma unroll
    for (int i = 1; i < kWaves; ++i) x[0] = SUM ? x[0] + x[i] : amax(x[0], x[i]);
    fr[q] = x[0];
  }
  if (threadIdx.x == 0) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q < nvals) out[(size_t)t * ostride + q] = fr[q];
  }
  if (!ga.ig) return;
  // the gate's norms that this fold wrote: its values, not the loads made
  // before it
  const bool norms = out == ga.out, change = out == ga.outc;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    if (q >= nvals) break;
    if (norms) gpre.o[q] = fr[q];
    if (change && q < 2) gpre.oc[q] = fr[q];
  }
  const GateWords wv = item_gate_check(ga.ig + gpre.gslot, gpre, threadIdx.x == 0);
  if (inst0 == gpre.inst) {
    DevLevel& d = ga.Lt[threadIdx.x];
    if (wv.stop >= 0) d.stop = wv.stop;
    if (wv.warm >= 0) d.warm = wv.warm;
    if (wv.skipc >= 0) d.skipc = wv.skipc;
    if (wv.pflip) d.pcur = pcur0 ^ 1;
  }
  set_words(ga.Lt, ga.nL, gpre.inst, wv, threadIdx.x + kFinBlock, kFinBlock);
}

// ---------------------------------------------------------------------------
// Layout conversions (FP64).
__device__ __forceinline__ size_t fidx(int i, int j, int k, int nx, int ny) {
  return ((size_t)(k + 1) * (ny + 2) + (j + 1)) * (nx + 2) + (i + 1);
}

__global__ __launch_bounds__(kBlock) void k_from_fortran(const DevLevel* __restrict__ Lt,
                                                         LaunchList ll, PtrList ptr,
                                                         int which, int add_fold) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  const int e = (b - ll.prefix[t]) * kBlock + threadIdx.x;
  if (e >= L.ncell) return;
  int i, j, k;
  decode(L, e, i, j, k);
  double v = gp(ptr.p[t])[fidx(i, j, k, L.nx, L.ny)];
  if (add_fold) {
    const auto bf = gp(L.bcfold);
    v += (bf[i] + bf[L.nx + j]) + bf[L.nx + L.ny + k];
  }
  gfield<double>(which == 0 ? L.u : L.f)[e] = v;
}

// Ingest of a solve: b = rhs + boundary fold and u = phi (reference layout
// -> chequer), with the partial sum of V*b of the block's cells.  A thread
// takes cell pairs (2m, j, k), (2m+1, j, k): one decode per pair, the pair's
// two reference-layout values are adjacent (a wave reads contiguous rows),
// and the two cells go to the two colours' half-rows at position m.  Each
// thread folds kWsumPer cells (kWsumPer/2 pairs) in a fixed order.
__global__ __launch_bounds__(kBlock) void k_ingest(const DevLevel* __restrict__ Lt, LaunchList ll,
                                                   PtrList rhs, PtrList phi,
                                                   double* __restrict__ partial) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  constexpr int kPairs = kWsumPer / 2;
  const int np = L.ncell >> 1;                        // pairs: hx * ny * nz
  const int p0 = (b - ll.prefix[t]) * kBlock * kPairs + threadIdx.x;
  const auto vol = gp(L.vol);
  const auto bf = gp(L.bcfold);
  const auto src = gp(rhs.p[t]);
  const auto ph = gp(phi.p[t]);
  const auto f = gfield<double>(L.f);
  const auto u = gfield<double>(L.u);
  const int nx = L.nx, ny = L.ny, hx = L.hx;
  double v[1] = {0.0};
  // every load is unconditional (pair indices clamped into the item), so
  // each chunk of kIngestU pairs issues its loads before their uses; pairs
  // past the item's end are masked at the stores and the sum
  constexpr int kIngestU = 4;
#pragma unroll
  for (int s0 = 0; s0 < kPairs; s0 += kIngestU) {
    if (s0 > 0) __builtin_amdgcn_sched_barrier(0);
    double s0v[kIngestU], s1v[kIngestU], q0v[kIngestU], q1v[kIngestU], fb0[kIngestU], fb1[kIngestU];
    double w0[kIngestU], w1[kIngestU];
    int e0[kIngestU], e1[kIngestU];
#pragma unroll
    for (int q = 0; q < kIngestU; ++q) {
      const int pp = p0 + (s0 + q) * kBlock;
      const int pc = pp < np ? pp : np - 1;
      const int row = gm_div(pc, L.gmhx, L.gshx), m = pc - row * hx;
      const int k = gm_div(row, L.gmny, L.gsny), j = row - k * ny;
      const int i = 2 * m;
      const size_t fi = fidx(i, j, k, nx, ny);
      s0v[q] = src[fi];
      s1v[q] = src[fi + 1];
      q0v[q] = ph[fi];
      q1v[q] = ph[fi + 1];
      fb0[q] = (bf[i] + bf[nx + j]) + bf[nx + ny + k];
      fb1[q] = (bf[i + 1] + bf[nx + j]) + bf[nx + ny + k];
      const double wyz = vol[nx + ny + k] * vol[nx + j];
      w0[q] = wyz * vol[i];
      w1[q] = wyz * vol[i + 1];
      const int rb = (k * ny + j) * 2;
      e0[q] = (rb + (j & 1)) * hx + m;                 // colour of (2m, j): j & 1
      e1[q] = (rb + ((j + 1) & 1)) * hx + m;
    }
#pragma unroll
    for (int q = 0; q < kIngestU; ++q) {
      const bool in = p0 + (s0 + q) * kBlock < np;
      const double bv0 = s0v[q] + fb0[q], bv1 = s1v[q] + fb1[q];
      // the first defect reads b and p back only after the whole ingest,
      // more than the caches hold: non-temporal stores (the ingest takes 6
      // us longer at 256^3, the first defect 9-13 us less)
      if (in) {
        __builtin_nontemporal_store(bv0, (double*)(f + e0[q]));
        __builtin_nontemporal_store(bv1, (double*)(f + e1[q]));
        __builtin_nontemporal_store(q0v[q], (double*)(u + e0[q]));
        __builtin_nontemporal_store(q1v[q], (double*)(u + e1[q]));
      }
      v[0] += in ? w0[q] * bv0 : 0.0;
      v[0] += in ? w1[q] * bv1 : 0.0;
    }
  }
  block_reduce_store<1, true>(v, partial + b);
}

// Weighted sums sum V x (V = dx_i dy_j dz_k), marching in z like the
// finest-level stencil kernels (march_blocks per item): a thread owns
// position col of a plane and kMarchK planes, sums dz_k x_k over them in
// order and weights that sum by dx_i dy_j; one partial per block.  The dz_k
// are wave-uniform (scalar loads), so a cell costs one vector load.
__global__ __launch_bounds__(kBlock) void k_wsum(const DevLevel* __restrict__ Lt, LaunchList ll,
                                                 int which, double* __restrict__ partial) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  const int hx = L.hx, ny = L.ny, nz = L.nz, nx = L.nx;
  const int plane = 2 * hx * ny;
  const int ncb = (plane + kBlock - 1) / kBlock;
  const int lb = b - ll.prefix[t];
  const int bk = lb / ncb, col = (lb - bk * ncb) * kBlock + threadIdx.x;
  const int k0 = bk * kMarchK, k1 = min(k0 + kMarchK, nz);
  const auto vol = gp(L.vol);
  const auto rho = gp(L.rho);
  // which 0: the current pressure of an FP64 finest entry (its ping-pong
  // state word pcur says which buffer holds it); 1: f; 2: rho(z)
  const auto x = gfield<const double>((const void*)(which == 0 ? (L.pcur ? L.u2 : L.u) : L.f));
  double v[1] = {0.0};
  if (col < plane) {
    const int row = gm_div(col, L.gmhx, L.gshx), m = col - row * hx, j = row >> 1;
    const int i = 2 * m + (((row & 1) + j) & 1);
    const auto vz = vol + nx + ny;
    double s = 0.0;
    if (k1 - k0 == kMarchK) {
      double xv[kMarchK];
#pragma unroll
      for (int q = 0; q < kMarchK; ++q)
        xv[q] = which == 2 ? rho[k0 + q] : x[(size_t)(k0 + q) * plane + col];
#pragma unroll
      for (int q = 0; q < kMarchK; ++q) s += vz[k0 + q] * xv[q];
    } else {
      for (int k = k0; k < k1; ++k) s += vz[k] * (which == 2 ? rho[k] : x[(size_t)k * plane + col]);
    }
    v[0] = (vol[i] * vol[nx + j]) * s;
  }
  block_reduce_store<1, true>(v, partial + b);
}

__global__ void k_zero(double* __restrict__ a, int n) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e < n) a[e] = 0.0;
}

// dst interior = u, minus the null-space component (c[t]/vrsum) rho(z) of
// singular items when c is given
__global__ __launch_bounds__(kBlock) void k_to_fortran(const DevLevel* __restrict__ Lt,
                                                       LaunchList ll, PtrList ptr,
                                                       const double* __restrict__ c) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  const int e = (b - ll.prefix[t]) * kBlock + threadIdx.x;
  if (e >= L.ncell) return;
  int i, j, k;
  decode(L, e, i, j, k);
  // the current pressure (pcur: which buffer of the ping-pong pair holds it)
  double x = gfield<const double>((const void*)(L.pcur ? L.u2 : L.u))[e];
  if (c && L.nullsp) x -= (c[t] / L.vrsum) * gp(L.rho)[k];
  gp(ptr.p[t])[fidx(i, j, k, L.nx, L.ny)] = x;
}

__global__ __launch_bounds__(kBlock) void k_copy_u(const DevLevel* __restrict__ Lt, LaunchList ll,
                                                   const int* __restrict__ active) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  if (level_off(L)) return;
  if (active && !active[L.inst]) return;
  const int e = (b - ll.prefix[t]) * kBlock + threadIdx.x;
  if (e >= L.ncell) return;
  gfield<double>(L.u2)[e] = gfield<const double>((const void*)L.u)[e];
}

template <class T>
__global__ __launch_bounds__(kBlock) void k_fill_zero(const DevLevel* __restrict__ Lt, LaunchList ll) {
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int t = find_item(ll.prefix, ll.nitems, b);
  const DevLevel& L = Lt[ll.items[t]];
  if (level_off(L)) return;
  const int e = (b - ll.prefix[t]) * kBlock + threadIdx.x;
  if (e < L.ncell) gfield<T>(L.u)[e] = T(0);
}

// ---------------------------------------------------------------------------
// Ghost layers (serial path of mgMK/mg_bdry.F90:71-190).
__global__ void k_ghost_wrap(double* __restrict__ a, int nx, int ny, int nz, int dir) {
  const int sx = nx + 2, sy = ny + 2, sz = nz + 2;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (dir == 0) {
    if (e >= sy * sz) return;
    const size_t base = (size_t)e * sx;
    a[base + 0] = a[base + nx];
    a[base + nx + 1] = a[base + 1];
  } else if (dir == 1) {
    if (e >= sx * sz) return;
    const int i = e % sx, k = e / sx;
    const size_t pl = (size_t)k * sy * sx;
    a[pl + i] = a[pl + (size_t)ny * sx + i];
    a[pl + (size_t)(ny + 1) * sx + i] = a[pl + (size_t)sx + i];
  } else {
    if (e >= sx * sy) return;
    const size_t pl = (size_t)sx * sy;
    a[e] = a[(size_t)nz * pl + e];
    a[(size_t)(nz + 1) * pl + e] = a[pl + e];
  }
}

// Every ghost cell of a ghosted field in one pass, with the values of the
// serial sequence (mgMK/mg_bdry.F90:71-190): the three periodic wraps over
// full planes, then the non-periodic faces in the order 1 X2max, 2 X3min,
// 3 X2min, 4 X3max, 5 X1min, 6 X1max, each from the layer inside it as the
// earlier passes left it.  A wrap only copies, so after the wraps a ghost
// cell holds the interior value at its coordinates wrapped one by one.  A
// face rule reads the cell one step inside its face, which the last earlier
// face whose layer holds that cell wrote, and so on: walking the faces from
// the last down and stepping inside each face whose layer holds the current
// cell gives that chain, whose rules are then applied forward to the
// wrapped interior value.  Interior cells are only read, and a cell on an
// edge or corner is computed alike by every thread that owns it.
// GhostBC: per face 1..6, type (0 periodic: no rule, 1 Neumann, 2
// Dirichlet), the value v and v*dxc(edge cell) (the Neumann offset, a
// product made on the host so the rule is one rounding, x -/+ vd).
__global__ __launch_bounds__(kBlock) void k_ghost_fill(double* __restrict__ a, int nx, int ny, int nz,
                                                       GhostBC bc) {
  // (32-bit index arithmetic: the ghost cells of any grid this library
  // accepts number far below 2^31)
  const int sx = nx + 2, sy = ny + 2, sz = nz + 2;
  const int nxf = 2 * sy * sz, nyf = 2 * sx * sz, nzf = 2 * sx * sy;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  int i, j, k;
  if (e < nxf) {
    const int r = e >> 1;
    i = (e & 1) ? nx + 1 : 0; k = r / sy; j = r - k * sy;
  } else if (e < nxf + nyf) {
    const int r = (e - nxf) >> 1;
    j = ((e - nxf) & 1) ? ny + 1 : 0; k = r / sx; i = r - k * sx;
  } else if (e < nxf + nyf + nzf) {
    const int r = (e - nxf - nyf) >> 1;
    k = ((e - nxf - nyf) & 1) ? nz + 1 : 0; j = r / sx; i = r - j * sx;
  } else {
    return;
  }
  int chain[6], nc = 0;
  int ci = i, cj = j, ck = k;
  for (int f = 6; f >= 1; --f) {
    if (!bc.type[f]) continue;
    bool in = false;
    switch (f) {
      case 1: in = cj == ny + 1; if (in) cj = ny; break;
      case 2: in = ck == 0; if (in) ck = 1; break;
      case 3: in = cj == 0; if (in) cj = 1; break;
      case 4: in = ck == nz + 1; if (in) ck = nz; break;
      case 5: in = ci == 0; if (in) ci = 1; break;
      default: in = ci == nx + 1; if (in) ci = nx; break;
    }
    if (in) chain[nc++] = f;
  }
  auto wrap = [](int c, int n) { return c == 0 ? n : (c == n + 1 ? 1 : c); };
  double x = a[((size_t)wrap(ck, nz) * sy + wrap(cj, ny)) * sx + wrap(ci, nx)];
  for (int q = nc - 1; q >= 0; --q) {
    const int f = chain[q];
    if (bc.type[f] == 2) x = bc.v[f];
    else if (f == 1 || f == 4 || f == 6) x = x + bc.vd[f];
    else x = x - bc.vd[f];
  }
  a[((size_t)k * sy + j) * sx + i] = x;
}

// ---------------------------------------------------------------------------
// Projection step (dns/NSsolver.F90:2204-2219, :2057-2082; dns/Routines.F90:123-144).
//
// The source and the divergence march in z: a thread owns one position of a
// plane and kProjK planes (the source of a small grid two or one), so W below
// a plane is the value it has just used (with one cell per thread the plane
// below was read by another XCD, a second time from memory) and the position
// is divided once per slab.  Bound by
// memory: at 512x256x256 the source takes 216 us (271 with one cell per
// thread) for 1.09 GB.
template <int K>
__global__ __launch_bounds__(kBlock) void k_psource(const double* __restrict__ U,
                                                    const double* __restrict__ V,
                                                    const double* __restrict__ W,
                                                    double* __restrict__ S,
                                                    const double* __restrict__ rho,
                                                    const double* __restrict__ rdxc,
                                                    const double* __restrict__ rdyc,
                                                    const double* __restrict__ rdzc, int nx, int ny,
                                                    int nz, double rdt) {
  const int sx = nx + 2, sy = ny + 2, sxy = sx * sy, npb = (sxy + kBlock - 1) / kBlock;
  const int b = xcd_swizzle(blockIdx.x, gridDim.x);
  const int bk = b / npb, pos = (b - bk * npb) * kBlock + threadIdx.x;
  if (pos >= sxy) return;
  const int j = pos / sx, i = pos - j * sx;
  const bool in = i > 0 && j > 0 && i <= nx && j <= ny;
  const int k0 = bk * K, ic = in ? i : 1, jc = in ? j : 1;
  const size_t c0 = (size_t)jc * sx + ic;               // a ghost column reads the first interior one
  const double rx = rdxc[ic], ry = rdyc[jc];
  double u[K], um[K], v[K], vm[K], w[K + 1];
  w[0] = W[(size_t)max(k0 - 1, 0) * sxy + c0];
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const size_t e = (size_t)min(k0 + q, nz + 1) * sxy + c0;
    u[q] = U[e];
    um[q] = U[e - 1];
    v[q] = V[e];
    vm[q] = V[e - sx];
    w[q + 1] = W[e];
  }
#pragma unroll
  for (int q = 0; q < K; ++q) {
    const int k = k0 + q;
    if (k > nz + 1) break;
    double r = 0.0;
    if (in && k > 0 && k <= nz) {
      const double rk = rho[k], rp = rho[k + 1], rm = rho[k - 1];
      r = ((rk * u[q] - rk * um[q]) * rx + (rk * v[q] - rk * vm[q]) * ry +
           (0.5 * (rp + rk) * w[q + 1] - 0.5 * (rk + rm) * w[q]) * rdzc[k]) * rdt;
    }
    S[(size_t)k * sxy + pos] = r;
  }
}

__global__ __launch_bounds__(kBlock) void k_pgrad(const double* __restrict__ p,
                                                  double* __restrict__ U, double* __restrict__ V,
                                                  double* __restrict__ W,
                                                  const double* __restrict__ rho,
                                                  const double* __restrict__ rdxe,
                                                  const double* __restrict__ rdye,
                                                  const double* __restrict__ rdze, int nx, int ny,
                                                  int nz, double dt, int wallmask) {
  const int e0 = blockIdx.x * kBlock + threadIdx.x;
  if (e0 >= nx * ny * nz) return;
  const int i = e0 % nx + 1, jk = e0 / nx, j = jk % ny + 1, k = jk / ny + 1;
  const int sx = nx + 2, sy = ny + 2;
  const size_t sxy = (size_t)sx * sy;
  const size_t e = (size_t)k * sxy + (size_t)j * sx + i;
  const double rk = rho[k], rp = rho[k + 1];
  const double pc = p[e];
  // the last face of a direction with a pressure-Neumann upper wall is the
  // wall itself: its normal velocity is the velocity boundary condition
  if (!((wallmask & 1) && i == nx)) U[e] = U[e] - (p[e + 1] / rk - pc / rk) * rdxe[i] * dt;
  if (!((wallmask & 2) && j == ny)) V[e] = V[e] - (p[e + sx] / rk - pc / rk) * rdye[j] * dt;
  if (!((wallmask & 4) && k == nz)) W[e] = W[e] - (p[e + sxy] / rp - pc / rk) * rdze[k] * dt;
}

// Divergence report (dns/Routines.F90:123-173): tiles of kBlock positions of
// a plane by kProjK planes, a block taking every gridDim-th tile (at most
// kDivBlocks blocks); a thread folds its cells in a fixed order.  Per block:
// {sum |div| V, max |div|, its cell index}; the maximum keeps the smallest
// index on ties (the reference's first-found order).  V = dx dy dz from the
// widths: two FP64 divisions and a 64-bit index division per cell bound the
// earlier form by arithmetic (256x128x77: 22.2 us, now 16.9).
__device__ __forceinline__ void div_better(double& b, long long& bi, double ob, long long oi) {
  if (ob > b || (ob == b && oi < bi)) { b = ob; bi = oi; }
}

__global__ __launch_bounds__(kBlock) void k_divergence(const double* __restrict__ U,
                                                       const double* __restrict__ V,
                                                       const double* __restrict__ W,
                                                       double* __restrict__ div,
                                                       const double* __restrict__ rdxc,
                                                       const double* __restrict__ rdyc,
                                                       const double* __restrict__ rdzc,
                                                       const double* __restrict__ dxc,
                                                       const double* __restrict__ dyc,
                                                       const double* __restrict__ dzc, int nx,
                                                       int ny, int nz, double* __restrict__ partial) {
  const int np = nx * ny, npb = (np + kBlock - 1) / kBlock, tiles = npb * ((nz + kProjK - 1) / kProjK);
  const int sx = nx + 2, sy = ny + 2;
  const size_t sxy = (size_t)sx * sy;
  double s[1] = {0.0};
  double best = -1.0;
  long long bidx = (long long)1 << 62;
  for (int tile = xcd_swizzle(blockIdx.x, gridDim.x); tile < tiles; tile += gridDim.x) {
    const int bk = tile / npb, pos = (tile - bk * npb) * kBlock + threadIdx.x;
    if (pos >= np) continue;
    const int j = pos / nx, i = pos - j * nx;
    const int k0 = bk * kProjK;
    const size_t c0 = (size_t)(j + 1) * sx + (i + 1);
    const double rx = rdxc[i + 1], ry = rdyc[j + 1], wxy = dxc[i + 1] * dyc[j + 1];
    double u[kProjK], um[kProjK], v[kProjK], vm[kProjK], w[kProjK + 1];
    w[0] = W[(size_t)k0 * sxy + c0];
#pragma unroll
    for (int q = 0; q < kProjK; ++q) {
      const size_t e = (size_t)min(k0 + q + 1, nz) * sxy + c0;
      u[q] = U[e];
      um[q] = U[e - 1];
      v[q] = V[e];
      vm[q] = V[e - sx];
      w[q + 1] = W[e];
    }
#pragma unroll
    for (int q = 0; q < kProjK; ++q) {
      const int k = k0 + q;
      if (k >= nz) break;
      const double d = (u[q] - um[q]) * rx + (v[q] - vm[q]) * ry + (w[q + 1] - w[q]) * rdzc[k + 1];
      if (div) div[(size_t)(k + 1) * sxy + c0] = d;
      s[0] += fabs(d) * (wxy * dzc[k + 1]);
      div_better(best, bidx, fabs(d), (long long)k * np + pos);
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const double ob = __shfl_xor(best, off, 64);
    const long long oi = __shfl_xor(bidx, off, 64);
    div_better(best, bidx, ob, oi);
  }
  __shared__ double sb[kBlock / 64];
  __shared__ long long si[kBlock / 64];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { sb[w] = best; si[w] = bidx; }
  double* out = partial + (size_t)blockIdx.x * kDivVals;
  block_reduce_store<1, true>(s, out);   // contains __syncthreads
  if (threadIdx.x == 0) {
    double b = sb[0];
    long long bi = si[0];
    for (int q = 1; q < (int)(blockDim.x >> 6); ++q) div_better(b, bi, sb[q], si[q]);
    out[1] = b;
    out[2] = (double)bi;
  }
}

// One block of kDivFin threads: thread t folds partials t, t+kDivFin, ...
// in order, then a fixed-shape tree combines the threads (deterministic).
constexpr int kDivFin = 1024;
__global__ __launch_bounds__(kDivFin) void k_divergence_finalize(const double* __restrict__ partial,
                                                                 int nb, double* __restrict__ out) {
  __shared__ double s0s[kDivFin / 64], bs[kDivFin / 64];
  __shared__ long long is[kDivFin / 64];
  double s0 = 0.0, b = -1.0;
  long long bi = (long long)1 << 62;
  for (int q = threadIdx.x; q < nb; q += kDivFin) {
    const double* p = partial + (size_t)q * kDivVals;
    s0 += p[0];
    div_better(b, bi, p[1], (long long)p[2]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    s0 += __shfl_xor(s0, off, 64);
    const double ob = __shfl_xor(b, off, 64);
    const long long oi = __shfl_xor(bi, off, 64);
    div_better(b, bi, ob, oi);
  }
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (lane == 0) { s0s[w] = s0; bs[w] = b; is[w] = bi; }
  __syncthreads();
  if (threadIdx.x == 0) {
    double a0 = s0s[0], ab = bs[0];
    long long ai = is[0];
    for (int q = 1; q < kDivFin / 64; ++q) {
      a0 += s0s[q];
      div_better(ab, ai, bs[q], is[q]);
    }
    out[0] = a0; out[1] = ab; out[2] = (double)ai;
  }
}

// ---------------------------------------------------------------------------
// Separable direct solve of a coarse level (host set-up in amg_direct.cpp):
// u = A^-1 f with A = Ax + Ay + Az and every 1-D operator diagonalised,
// A_d = V_d diag(l_d) V_d^-1.  Three passes, all dense products on the
// matrix cores, in the compute type CT of the level's tables: FP64
// (v_mfma_f64_16x16x4f64) for an FP64 V-cycle, FP32 (v_mfma_f32_16x16x4f32)
// for the FP32 V-cycle of a mixed solve, whose coarse correction needs no
// more (at 64^3 the FP32 passes are the faster):
//   k_direct_xy<FWD>  per plane k:      f^ = Vy^-1 f_k Vx^-T          (-> dscr)
//   k_direct_z        per 16 modes:     x^ = Vz (inv .* (Vz^-1 f^))    (-> dscr + n)
//   k_direct_xy<inv>  per plane k:      u_k = Vy x^_k Vx^T
// with inv = 1/(lx + ly + lz) per eigenmode (0 for a singular operator's
// null mode: the solution then has sum V u = 0).
//
// Each pass is a few hundred short workgroups, so its time is its chain of
// waits, not its products (a wave's two products at 64^3 are 32 matrix
// instructions).  Every operand that comes from memory is therefore loaded
// straight into the lanes that feed it to the matrix core, all of them before
// the first product, and only the first product's result goes through LDS.
// The plane passes take 16 rows of the plane per workgroup, (My[rows] X) Mx,
// so that the elements of X and Mx lie across the lanes; the order of the sum
// over k is free, and a lane takes four consecutive k of a row of My.  The three
// launches take 11.4 us at 64^3 in FP32 and 9.4 at 32^3 in FP64 (22.0 and
// 20.2 with every operand staged through LDS, in passes of 48 loads per
// thread whatever the size); FP32 64x16x64 17.2 -> 9.4, FP64 64^3 28.2 -> 17.
typedef double dbl4 __attribute__((ext_vector_type(4)));
typedef float flt4 __attribute__((ext_vector_type(4)));

// The 16x16x4 product of each compute type: lane l holds A[i][k] and B[k][j]
// with i, j = l % 16 and k = l / 16; result register r of lane l holds
// D[row(l / 16, r)][l % 16] (the two types lay D out differently).
template <class CT> struct Mfma16;
template <> struct Mfma16<double> {
  typedef dbl4 V;
  static __device__ __forceinline__ V op(double a, double b, V c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return lk + 4 * r; }
};
template <> struct Mfma16<float> {
  typedef flt4 V;
  static __device__ __forceinline__ V op(float a, float b, V c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lk, int r) { return 4 * lk + r; }
};

constexpr int kDirectZs = 20;   // row stride of the z pass's LDS (kDirectCols modes)
__host__ __device__ inline int direct_nzp(int nz) { return (nz + 15) & ~15; }

// A lane's operands of up to 64 consecutive k (n groups of 16): value [g][q]
// belongs to k = k0 + 16 g + 4 (l / 16) + q of the lane's row or column.
template <class CT> struct DirectOps {
  typedef CT V4 __attribute__((ext_vector_type(4)));
  CT v[4][4];
  // f(k): the operand at k
  template <class F> __device__ __forceinline__ void load(int n, int k0, F&& f) {
    const int lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (g < n) {
#pragma unroll
        for (int q = 0; q < 4; ++q) v[g][q] = f(k0 + 16 * g + 4 * lk + q);
      }
  }
  // row: the lane's row of operands, 4-element aligned
  template <int AS, class E> __device__ __forceinline__ void load_row(int n, int k0, sp<AS, E> row) {
    const int lk = (threadIdx.x & 63) >> 4;
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (g < n) {
        const V4 t = *(sp<AS, const V4>)(row + k0 + 16 * g + 4 * lk);
#pragma unroll
        for (int q = 0; q < 4; ++q) v[g][q] = t[q];
      }
  }
};
template <class CT>
__device__ __forceinline__ typename Mfma16<CT>::V direct_mac(int n, const DirectOps<CT>& a,
                                                             const DirectOps<CT>& b,
                                                             typename Mfma16<CT>::V acc) {
#pragma unroll
  for (int g = 0; g < 4; ++g)
    if (g < n) {
#pragma unroll
      for (int q = 0; q < 4; ++q) acc = Mfma16<CT>::op(a.v[g][q], b.v[g][q], acc);
    }
  return acc;
}

// The plane passes, one workgroup per (plane k, 16 rows r0.. of it), a wave
// per 16 columns: FWD: rows of f^_k = Vy^-1 f_k Vx^-T into dscr, from plane k
// of f (level precision T); otherwise rows of u_k = Vy x^_k Vx^T from
// dscr + n.  Either is (My[rows] X) Mx.  The tables (dmat, dinv, dscr) hold
// CT values.
template <class T, class CT, bool FWD>
__global__ __launch_bounds__(kBlock) void k_direct_xy(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                      LaunchList ll) {
  extern __shared__ double dl[];
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevLevel& D = Lt[wk.idx];
  const double* dmat = D.dmat;
  double* dscr = D.dscr;
  pin_s(dmat, dscr);
  const LevelHead L = level_head(D);
  if (level_off(L)) return;
  const int nx = L.nx, ny = L.ny, hx = L.hx, sz = nx + 4;
  const int rs = ny / kDirectCols, k = wk.lb / rs, r0 = (wk.lb - k * rs) * kDirectCols;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), cstep = kBlock / 64 * 16;
  const sp<kS, CT> Z = (sp<kS, CT>)(sp<kS, double>)dl;   // My[rows] X (16 x nx, stride sz)
  const auto m = gp(reinterpret_cast<const CT*>(dmat));
  const auto Mx = m + (FWD ? 0 : nx * nx);               // Vx^-T or Vx^T
  const auto My = m + 2 * nx * nx + (FWD ? 0 : ny * ny) + (r0 + li) * ny;   // Vy^-1 or Vy
  const auto scr = gp(reinterpret_cast<CT*>(dscr));
  const auto f = gfield<const T>((const void*)L.f);
  const auto in = scr + (size_t)L.ncell + (size_t)k * ny * nx;
  auto x_at = [&](int j, int i) {
    if constexpr (FWD) return (CT)f[cidx(i >> 1, j, k, (i + j) & 1, hx, ny)];
    else return (CT)in[j * nx + i];
  };
  auto groups = [](int left) { return min(4, left >> 4); };
  DirectOps<CT> a, b, c;
  auto load1 = [&](int c0, int q0) {
    a.load_row(groups(ny - q0), q0, My);
    b.load(groups(ny - q0), q0, [&](int j) { return x_at(j, c0 + li); });
  };
  auto load2 = [&](int c0, int q0) {
    c.load(groups(nx - q0), q0, [&](int i) { return Mx[i * nx + c0 + li]; });
  };
  const int cw = 16 * wave;
  if (cw < nx) {
    load1(cw, 0);
    load2(cw, 0);
  }
  typedef typename Mfma16<CT>::V V;
  for (int c0 = cw; c0 < nx; c0 += cstep) {
    V acc = {CT(0), CT(0), CT(0), CT(0)};
    for (int q0 = 0; q0 < ny; q0 += 64) {
      if (c0 != cw || q0) load1(c0, q0);
      acc = direct_mac<CT>(groups(ny - q0), a, b, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) Z[Mfma16<CT>::row(lk, r) * sz + c0 + li] = acc[r];
  }
  __syncthreads();
  for (int c0 = cw; c0 < nx; c0 += cstep) {
    V acc = {CT(0), CT(0), CT(0), CT(0)};
    for (int q0 = 0; q0 < nx; q0 += 64) {
      if (c0 != cw || q0) load2(c0, q0);
      a.load_row(groups(nx - q0), q0, Z + li * sz);
      acc = direct_mac<CT>(groups(nx - q0), a, c, acc);
    }
    const int i = c0 + li;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int j = r0 + Mfma16<CT>::row(lk, r);
      if constexpr (FWD) scr[(size_t)k * ny * nx + j * nx + i] = acc[r];
      else gfield<T>(L.u)[cidx(i >> 1, j, k, (i + j) & 1, hx, ny)] = (T)acc[r];
    }
  }
}

// The z pass, one workgroup per slab of kDirectCols modes m0.. (all k), a
// wave per 16 of the nzp rows: x^ = Vz (inv .* (Vz^-1 f^)).
template <class CT>
__global__ __launch_bounds__(kBlock) void k_direct_z(const DevLevel* __restrict__ Lt, LIST_PARAMS,
                                                      LaunchList ll) {
  static_assert(kDirectMaxNz <= 16 * (kBlock / 64) && kDirectMaxNz <= 64, "one chunk of rows per wave");
  extern __shared__ double dl[];
  const Work wk = work_item(ln, lnb, li0, ll);
  const DevLevel& D = Lt[wk.idx];
  const double *dmat = D.dmat, *dinv = D.dinv;
  double* dscr = D.dscr;
  pin_s(dmat, dinv, dscr);
  const LevelHead L = level_head(D);
  if (level_off(L)) return;
  const int nx = L.nx, ny = L.ny, nz = L.nz, nzp = direct_nzp(nz), n = nzp >> 4;
  const int plane = nx * ny, m0 = wk.lb * kDirectCols;
  const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
  const int r0 = 16 * __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const sp<kS, CT> Tm = (sp<kS, CT>)(sp<kS, double>)dl;   // inv .* (Vz^-1 f^) (nzp x 16)
  const auto Wi = gp(reinterpret_cast<const CT*>(dmat)) + 2 * nx * nx + 2 * ny * ny + (r0 + li) * nzp;
  const auto W = Wi + nzp * nzp;                          // Vz, after Vz^-1
  const auto fh = gp(reinterpret_cast<const CT*>(dscr)) + m0 + li;
  const auto inv = gp(reinterpret_cast<const CT*>(dinv)) + m0 + li;
  typedef typename Mfma16<CT>::V V;
  DirectOps<CT> a, b, c;
  const V zero = {CT(0), CT(0), CT(0), CT(0)};
  const bool on = r0 < nzp;
  if (on) {
    CT iv[4];
    a.load_row(n, 0, Wi);
    b.load(n, 0, [&](int k) { return fh[min(k, nz - 1) * plane]; });
#pragma unroll
    for (int r = 0; r < 4; ++r) iv[r] = inv[min(r0 + Mfma16<CT>::row(lk, r), nz - 1) * plane];
    c.load_row(n, 0, W);
    // rows past nz are zero in the tables; the clamped data there may not be finite
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (16 * (e >> 2) + 4 * lk + (e & 3) >= nz) b.v[e >> 2][e & 3] = CT(0);
    const V acc = direct_mac<CT>(n, a, b, zero);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = r0 + Mfma16<CT>::row(lk, r);
      Tm[row * kDirectZs + li] = row < nz ? acc[r] * iv[r] : CT(0);
    }
  }
  __syncthreads();
  if (!on) return;
  b.load(n, 0, [&](int k) { return Tm[k * kDirectZs + li]; });
  const V acc = direct_mac<CT>(n, c, b, zero);
  const auto xo = gp(reinterpret_cast<CT*>(dscr)) + (size_t)L.ncell + m0 + li;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = r0 + Mfma16<CT>::row(lk, r);
    if (row < nz) xo[(size_t)row * plane] = acc[r];
  }
}

inline unsigned nb(size_t n, int bs = kBlock) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

// Clears the state words of the instances of the items of ll.
__global__ void k_gate_reset(DevLevel* __restrict__ Lt, int nL, LaunchList ll, int only_stopped) {
  for (int l = threadIdx.x; l < nL; l += blockDim.x) {
    bool mine = false;
    for (int t = 0; t < ll.nitems; ++t) mine = mine || Lt[ll.items[t]].inst == Lt[l].inst;
    if (only_stopped && !Lt[l].stop) mine = false;
    if (mine) {
      Lt[l].stop = 0;
      Lt[l].warm = 0;
      Lt[l].skipc = 0;
      Lt[l].pcur = 0;
    }
  }
}

// ---- launchers --------------------------------------------------------------
#define LAUNCH(kern, grid, blk, ...) hipLaunchKernelGGL(kern, dim3(grid), dim3(blk), 0, s, __VA_ARGS__)

// Compute units of the current device (cached per device).
static int device_cus() {
  static int cus[64] = {0};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  if (cus[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      n = 256;
    cus[dev] = n;
  }
  return cus[dev];
}

void launch_rb_march(bool fp64, const DevLevel* L, const LaunchList& ll, int parity, int zero_guess,
                     int planes, hipStream_t s) {
#define RM(T, K) LAUNCH((k_rb_march<T, K>), ll.nblocks, kBlock, L, LIST_ARGS(ll), parity, zero_guess, ll)
  if (fp64) {
    if (planes == 8) RM(double, 8); else if (planes == 4) RM(double, 4); else RM(double, 2);
  } else {
    if (planes == 8) RM(float, 8); else if (planes == 4) RM(float, 4); else RM(float, 2);
  }
#undef RM
}
RbPair rb_pair(bool fp64, int hx, int ny, int nz) {
  // Whole rows in a workgroup of at most 1024 threads, and halos that wrap
  // at most once.
  if ((kPairY + 2) * hx > 1024 || ny < kPairY || nz < 4) return {0, 0};
  // Three fields (u, w, b) that stay in the cache: past that the sweep waits
  // for HBM and the halos' extra reads lose (12 cycles of FP64 256x128x128
  // 2692 -> 2605 us, of 256x256x128 4158 -> 4486; FP32 256^3 4725 -> 4483,
  // 256x512x256 9598 -> 10117).
  if (2ll * hx * ny * nz > (fp64 ? 1ll << 22 : 1ll << 24)) return {0, 0};
  // Slabs of four planes, or of two where four leave CUs idle (32^3 FP64 932
  // -> 904 us, 64x32x32 FP32 1042 -> 1010; at 64^3, with as many workgroups
  // as CUs, 650 against 654).
  const int rows = (ny + kPairY - 1) / kPairY;
  const int tz = rows * ((nz + 3) / 4) < device_cus() ? 2 : 4;
  return {tz, rows * ((nz + tz - 1) / tz)};
}
void launch_rb_pair(bool fp64, const DevLevel* L, const LaunchList& ll, int zero_guess, int back,
                    int tz, int hx_max, hipStream_t s) {
  const int threads = ((kPairY + 2) * hx_max + 63) & ~63;
  const size_t lds = (size_t)(kPairY + 2) * (tz + 2) * hx_max * (fp64 ? 8 : 4);
#define RB(T, TZ)                                                                                \
  hipLaunchKernelGGL((k_rb_pair<T, TZ>), dim3(ll.nblocks), dim3(threads), lds, s, L, LIST_ARGS(ll), \
                     zero_guess, back, ll)
  if (fp64) {
    if (tz == 2) RB(double, 2);
    else RB(double, 4);
  } else {
    if (tz == 2) RB(float, 2);
    else RB(float, 4);
  }
#undef RB
}
void launch_rb_point(bool fp64, const DevLevel* L, const LaunchList& ll, int parity, int zero_guess,
                     hipStream_t s) {
  if (fp64) LAUNCH(k_rb_point<double>, ll.nblocks, kBlock, L, LIST_ARGS(ll), parity, zero_guess, ll);
  else LAUNCH(k_rb_point<float>, ll.nblocks, kBlock, L, LIST_ARGS(ll), parity, zero_guess, ll);
}
static void zline_variant(bool fp64, const DevLevel* L, const LaunchList& ll, int parity,
                          int zero_guess, int segs, hipStream_t s, bool lean, bool nbr, bool half) {
  // half: two segments of 32 columns per wave, segs rounded up to even
  const int wy = half ? (segs + 1) / 2 : segs, ps = half ? 2 * wy : segs, cw = half ? 32 : 64;
  const dim3 blk(64, wy);
  // reduced-system state (two buffers in FP32, one in FP64) + staged rows
  const size_t lds = (size_t)((fp64 ? 6 : 12) * cw + 3 * kZSeg) * ps * (fp64 ? 8 : 4);
#define ZL(T, CH, NBR, LEAN, H)                                                                   \
  hipLaunchKernelGGL((k_zline<T, kZSeg, CH, NBR, LEAN, H>), dim3(ll.nblocks), blk, lds, s, L, \
                     LIST_ARGS(ll), parity, zero_guess, ll)
  if (fp64) {
    if (!lean) {
      if (nbr) ZL(double, kZChunk64, true, false, true);
      else ZL(double, kZChunk64, false, false, true);
    } else if (half) {
      if (nbr) ZL(double, kZChunk64, true, true, true);
      else ZL(double, kZChunk64, false, true, true);
    } else {
      if (nbr) ZL(double, kZChunk64, true, true, false);
      else ZL(double, kZChunk64, false, true, false);
    }
  } else if (half) {
    if (nbr) ZL(float, kZChunk32, true, false, true);
    else ZL(float, kZChunk32, false, false, true);
  } else if (lean) {
    if (nbr) ZL(float, kZChunk32, true, true, false);
    else ZL(float, kZChunk32, false, true, false);
  } else {
    if (nbr) ZL(float, kZChunk32, true, false, false);
    else ZL(float, kZChunk32, false, false, false);
  }
#undef ZL
}
void launch_zline(bool fp64, const DevLevel* L, const LaunchList& ll, int parity, int zero_guess,
                  int segs, hipStream_t s, int form) {
  // The shape, from the count of 64-column groups (forced forms keep 64
  // columns):
  // - at most half as many as the device has CUs, and columns of two segments
  //   or more: 32 columns per workgroup, over twice the CUs, with the shorter
  //   dependent chains of the short form;
  // - up to the count of CUs: one group per CU is latency-bound too.  FP32
  //   takes the short form, FP64 (which the short form leaves no registers)
  //   the lean one;
  // - more: blocks pair up on the CUs, the lean form's registers allowing.
  //   FP64 needs the 32-column shape for that (256^3 48.4 -> 42.9 us, 4.16 ->
  //   4.69 TB/s, where the lone 16-wave group of a CU loaded and solved in
  //   turn; 512x256x128 41.0 -> 40.4; of 140 groups 11.2 -> 12.0).
  const int cus = device_cus();
  const bool few = form == 0 && segs >= 2 && 2 * ll.nblocks <= cus;
  const bool many = form == 0 && ll.nblocks > cus;
  const bool half = few || (many && fp64 && segs >= 2);
  const bool lean = !few && (fp64 || many || form == 2);
  LaunchList hl;
  if (half) {
    hl = ll;
    for (int t = 0; t <= ll.nitems; ++t) hl.prefix[t] = 2 * ll.prefix[t];
    hl.nblocks = 2 * ll.nblocks;
  }
  const LaunchList& l2 = half ? hl : ll;
  // kZgDyn with a zero other colour: the sweep from zero, then the ordinary
  // sweep for the instances whose cycle continues the iterate; each kernel
  // returns at once for the instances of the other
  if ((zero_guess & kZgDyn) && (zero_guess & 1)) {
    zline_variant(fp64, L, l2, parity, zero_guess, segs, s, lean, false, half);
    zline_variant(fp64, L, l2, parity, kZgWarm, segs, s, lean, true, half);
    return;
  }
  zline_variant(fp64, L, l2, parity, zero_guess, segs, s, lean, !(zero_guess & 1), half);
}
size_t zline_table_bytes(int nz) { return sizeof(float) * kZRec * (((nz + kZSeg - 1) / kZSeg + 1) & ~1); }
void launch_zline_table(const float* co32, int nx, int ny, int nz, float* zt, hipStream_t s) {
  LAUNCH(k_zline_table, 1, 64, co32, nx, ny, nz, zt);
}
void launch_zline_shared(const DevLevel* L, const LaunchList& ll, int parity, int zero_guess, int segs,
                         hipStream_t s) {
  // More column groups than CUs, and the other colour is read: two groups
  // share a CU, whose arithmetic hides behind the other's loads anyway, and
  // the general sweep's smaller start is the faster (256^3: 19.5 against
  // 20.3 us; 512x256x256: 36.0 against 37.5 us).
  if (ll.nblocks > device_cus() && !(zero_guess & 1)) {
    launch_zline(false, L, ll, parity, zero_guess, segs, s);
    return;
  }
  if (segs >= 2 && 2 * ll.nblocks <= device_cus()) {
    LaunchList hl = ll;
    for (int t = 0; t <= ll.nitems; ++t) hl.prefix[t] = 2 * ll.prefix[t];
    hl.nblocks = 2 * ll.nblocks;
    const int wy = (segs + 1) / 2;
    const size_t lds = (size_t)2 * wy * (4 * 32 + kZRec) * sizeof(float);
    hipLaunchKernelGGL(k_zline_shared<true>, dim3(hl.nblocks), dim3(64, wy), lds, s, L, LIST_ARGS(hl),
                       parity, zero_guess, hl);
    return;
  }
  const size_t lds = (size_t)4 * segs * 64 * sizeof(float);
  hipLaunchKernelGGL(k_zline_shared<false>, dim3(ll.nblocks), dim3(64, segs), lds, s, L, LIST_ARGS(ll),
                     parity, zero_guess, ll);
}
void launch_zline_col(bool fp64, const DevLevel* L, const LaunchList& ll, int parity,
                      int zero_guess, hipStream_t s) {
  if (fp64) LAUNCH(k_zline_col<double>, ll.nblocks, kBlock, L, LIST_ARGS(ll), parity, zero_guess, ll);
  else LAUNCH(k_zline_col<float>, ll.nblocks, kBlock, L, LIST_ARGS(ll), parity, zero_guess, ll);
}
void launch_restrict(bool fp64, const DevLevel* L, const DevXfer* X, const LaunchList& ll,
                     hipStream_t s) {
  if (fp64) LAUNCH(k_restrict<double>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), ll);
  else LAUNCH(k_restrict<float>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), ll);
}
void launch_restrict_quad(bool fp64, const DevLevel* L, const DevXfer* X, const LaunchList& ll,
                          hipStream_t s, bool use_skip) {
  if (fp64) LAUNCH(k_restrict_quad<double>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
  else LAUNCH(k_restrict_quad<float>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
}
void launch_restrict222(bool fp64, const DevLevel* L, const DevXfer* X, const LaunchList& ll,
                        hipStream_t s, bool use_skip) {
  if (fp64) LAUNCH(k_restrict222<double>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
  else LAUNCH(k_restrict222<float>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
}
void launch_prolong(bool fp64, const DevLevel* L, const DevXfer* X, const LaunchList& ll,
                    hipStream_t s, bool use_skip) {
  if (fp64) LAUNCH(k_prolong<double>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
  else LAUNCH(k_prolong<float>, ll.nblocks, kBlock, L, X, LIST_ARGS(ll), use_skip ? 1 : 0, ll);
}
static size_t direct_lds_limit() {
  static size_t limit = 0;
  if (limit) return limit;
  int dev = 0, v = 0;
  size_t lim = 64 * 1024;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
      v > 0)
    lim = (size_t)v;
  const void* kernels[] = {reinterpret_cast<const void*>(&k_direct_xy<double, double, true>),
                           reinterpret_cast<const void*>(&k_direct_xy<float, float, true>),
                           reinterpret_cast<const void*>(&k_direct_xy<double, double, false>),
                           reinterpret_cast<const void*>(&k_direct_xy<float, float, false>),
                           reinterpret_cast<const void*>(&k_direct_z<double>),
                           reinterpret_cast<const void*>(&k_direct_z<float>)};
  bool ok = true;
  for (const void* k : kernels)
    ok = ok && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lim) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    lim = 64 * 1024;
  }
  limit = lim;
  return limit;
}
size_t direct_lds(int nx, int nz, bool fp64) {
  const size_t es = fp64 ? sizeof(double) : sizeof(float);
  return es * std::max((size_t)kDirectCols * (nx + 4), (size_t)direct_nzp(nz) * kDirectZs);
}
bool direct_fits(int nx, int ny, int nz, bool fp64) {
  const size_t nzp = direct_nzp(nz), pad = kDirectCols + 1;
  const size_t xy = (size_t)ny * (nx + 1) + (size_t)ny * (ny + 1) + (size_t)(nx + ny) * pad;
  const size_t z = 2 * nzp * pad + 2 * nzp * (nzp + 1);
  return std::max(xy, z) * (fp64 ? sizeof(double) : sizeof(float)) <= direct_lds_limit();
}
void launch_direct(bool fp64, const DevLevel* L, const LaunchList& planes, const LaunchList& slabs,
                   size_t lds, hipStream_t s) {
  const dim3 blk(kBlock);
  if (fp64) {
    hipLaunchKernelGGL((k_direct_xy<double, double, true>), dim3(planes.nblocks), blk, lds, s, L, LIST_ARGS(planes), planes);
    hipLaunchKernelGGL(k_direct_z<double>, dim3(slabs.nblocks), blk, lds, s, L, LIST_ARGS(slabs), slabs);
    hipLaunchKernelGGL((k_direct_xy<double, double, false>), dim3(planes.nblocks), blk, lds, s, L, LIST_ARGS(planes), planes);
  } else {
    hipLaunchKernelGGL((k_direct_xy<float, float, true>), dim3(planes.nblocks), blk, lds, s, L, LIST_ARGS(planes), planes);
    hipLaunchKernelGGL(k_direct_z<float>, dim3(slabs.nblocks), blk, lds, s, L, LIST_ARGS(slabs), slabs);
    hipLaunchKernelGGL((k_direct_xy<float, float, false>), dim3(planes.nblocks), blk, lds, s, L, LIST_ARGS(planes), planes);
  }
}
void launch_coarse(bool fp64, const DevLevel* L, const LaunchList& ll, hipStream_t s) {
  if (fp64) LAUNCH(k_coarse<double>, ll.nblocks, kBlock, L, ll);
  else LAUNCH(k_coarse<float>, ll.nblocks, kBlock, L, ll);
}
int tail_nz_class(bool fp64, int nz_max, bool zline) {
  if (!zline) return 0;
  if (nz_max <= 8) return 8;
  if (nz_max <= 16 || fp64) return 16;
  return 32;
}

#define TAIL_KERNEL(T, NZ, F) (k_tail<T, NZ, F>)
void launch_tail(bool fp64, int nz_class, bool all222, const DevLevel* L, const DevXfer* X,
                 const DevTail* T, const LaunchList& ll, size_t lds_bytes, hipStream_t s, int phase) {
  const dim3 grd(ll.nitems);
#define GO(TT, NZ)                                                                                   \
  do {                                                                                               \
    const dim3 blk(64, NZ == 0 ? kTailWavesPoint : kTailWaves);                                      \
    if (all222) hipLaunchKernelGGL(TAIL_KERNEL(TT, NZ, true), grd, blk, lds_bytes, s, L, X, T, ll, phase); \
    else hipLaunchKernelGGL(TAIL_KERNEL(TT, NZ, false), grd, blk, lds_bytes, s, L, X, T, ll, phase);       \
  } while (0)
  if (fp64) {
    if (nz_class == 0) GO(double, 0); else if (nz_class <= 8) GO(double, 8); else GO(double, 16);
  } else {
    if (nz_class == 0) GO(float, 0);
    else if (nz_class <= 8) GO(float, 8);
    else if (nz_class <= 16) GO(float, 16);
    else GO(float, 32);
  }
#undef GO
}

void launch_tail_line(const DevLevel* L, const DevTail* T, const LaunchList& ll, size_t lds_bytes,
                      hipStream_t s) {
  hipLaunchKernelGGL(k_tail_line, dim3(ll.nitems), dim3(64 * kLineWaves), lds_bytes, s, L, T,
                     LIST_ARGS(ll), ll);
}

void launch_coarse_wide(bool fp64, const DevLevel* L, const LaunchList& ll, hipStream_t s) {
  if (fp64) LAUNCH(k_coarse_wide<double>, ll.nblocks, kBlock, L, ll);
  else LAUNCH(k_coarse_wide<float>, ll.nblocks, kBlock, L, ll);
}

size_t tail_lds_limit() {
  static size_t limit = 0;
  if (limit) return limit;
  int dev = 0, v = 0;
  size_t lim = 64 * 1024;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&v, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) == hipSuccess &&
      v > 0)
    lim = (size_t)v;
  // room for the static descriptor array of the kernel
  lim -= sizeof(DevLevel) * kTailMaxLevels + 256;
  const void* kernels[] = {
      reinterpret_cast<const void*>(&k_tail_line),
      reinterpret_cast<const void*>(&k_tail<double, 0, true>),
      reinterpret_cast<const void*>(&k_tail<double, 0, false>),
      reinterpret_cast<const void*>(&k_tail<float, 0, true>),
      reinterpret_cast<const void*>(&k_tail<float, 0, false>),
      reinterpret_cast<const void*>(&k_tail<double, 8, true>),
      reinterpret_cast<const void*>(&k_tail<double, 8, false>),
      reinterpret_cast<const void*>(&k_tail<double, 16, true>),
      reinterpret_cast<const void*>(&k_tail<double, 16, false>),
      reinterpret_cast<const void*>(&k_tail<float, 8, true>),
      reinterpret_cast<const void*>(&k_tail<float, 8, false>),
      reinterpret_cast<const void*>(&k_tail<float, 16, true>),
      reinterpret_cast<const void*>(&k_tail<float, 16, false>),
      reinterpret_cast<const void*>(&k_tail<float, 32, true>),
      reinterpret_cast<const void*>(&k_tail<float, 32, false>)};
  bool ok = true;
  for (const void* k : kernels)
    ok = ok && hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lim) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    lim = 64 * 1024 - sizeof(DevLevel) * kTailMaxLevels - 256;
  }
  limit = lim;
  return limit;
}
// (k_fine takes the table writable: the mixed first defect records bshift)
int march_planes(int hx, int ny, int nz) {
  // Slabs of 16 planes re-read the fewest planes; where they make fewer
  // workgroups than the device has CUs, shorter ones (a 64^3 residual has 64
  // workgroups of 16 planes: FP64 solve 4170 us, with 256 of four 3977;
  // 64x48x32 673 -> 655).  Past that, shorter slabs lose (256x64x256, 1024
  // workgroups of 16: 774 us, of four 808; 20 solves of up to 64x64x64 in the
  // same launches 3720, each with its own rule 3990).
  for (int K : {kMarchK, 4})
    if (march_blocks(hx, ny, nz, K) >= device_cus()) return K;
  return 2;
}
void launch_residual_max(const DevLevel* L, const LaunchList& ll, double* partial, hipStream_t s) {
  LAUNCH((k_fine<kResMax, false>), ll.nblocks, kBlock, const_cast<DevLevel*>(L), LIST_ARGS(ll), nullptr,
         partial, ll);
}
void launch_first_defect(bool fp64, const DevLevel* L, const LaunchList& ll, const double* c,
                         double* partial, hipStream_t s) {
  DevLevel* W = const_cast<DevLevel*>(L);
  if (fp64) LAUNCH((k_fine<kResMax, true>), ll.nblocks, kBlock, W, LIST_ARGS(ll), c, partial, ll);
  else LAUNCH((k_fine<kDefect32, true>), ll.nblocks, kBlock, W, LIST_ARGS(ll), c, partial, ll);
}
void launch_ingest(const DevLevel* L, const LaunchList& ll, const PtrList& rhs, const PtrList& phi,
                   double* partial, hipStream_t s) {
  LAUNCH(k_ingest, ll.nblocks, kBlock, L, ll, rhs, phi, partial);
}
void launch_change_max(const DevLevel* L, const LaunchList& ll, double* partial, hipStream_t s) {
  LAUNCH(k_change_max, ll.nblocks, kBlock, L, ll, partial);
}
void launch_correct_defect32(const DevLevel* L, const LaunchList& ll, double* partial,
                             hipStream_t s) {
  LAUNCH((k_fine<kCorrDefect32, false>), ll.nblocks, kBlock, const_cast<DevLevel*>(L), LIST_ARGS(ll), nullptr,
         partial, ll);
}
void launch_zero(double* a, int n, hipStream_t s) {
  LAUNCH(k_zero, nb((size_t)n), kBlock, a, n);
}
void launch_gate_reset(DevLevel* L, int nL, const LaunchList& ll, hipStream_t s, bool only_stopped) {
  hipLaunchKernelGGL(k_gate_reset, dim3(1), dim3(256), 0, s, L, nL, ll, only_stopped ? 1 : 0);
}
void launch_gate_init(const LaunchList& ll, const double* out, ItemGate* ig, DevLevel* L, int nL,
                      int maxcy, int rule, double tol, int report, hipStream_t s) {
  hipLaunchKernelGGL(k_gate_init, dim3(1), dim3(kMaxItems), 0, s, ll, out, ig, L, nL, maxcy, rule,
                     tol, report);
}
void launch_finalize(const LaunchList& ll, const double* partial, int nvals, int op_sum, double* out,
                     int ostride, hipStream_t s, const GateArgs* gate) {
  GateArgs ga{};
  if (gate) ga = *gate;
  if (op_sum) LAUNCH(k_finalize<true>, ll.nitems, kFinBlock, LIST_ARGS(ll), nvals, partial, out, ostride, ga, ll);
  else LAUNCH(k_finalize<false>, ll.nitems, kFinBlock, LIST_ARGS(ll), nvals, partial, out, ostride, ga, ll);
}
void launch_from_fortran(const DevLevel* L, const LaunchList& ll, const PtrList& ptr, int which,
                         int add_fold, hipStream_t s) {
  LAUNCH(k_from_fortran, ll.nblocks, kBlock, L, ll, ptr, which, add_fold);
}
void launch_wsum(const DevLevel* L, const LaunchList& ll, int which, double* partial, hipStream_t s) {
  LAUNCH(k_wsum, ll.nblocks, kBlock, L, ll, which, partial);
}
void launch_to_fortran(const DevLevel* L, const LaunchList& ll, const PtrList& ptr, const double* c,
                       hipStream_t s) {
  LAUNCH(k_to_fortran, ll.nblocks, kBlock, L, ll, ptr, c);
}
void launch_copy_u(const DevLevel* L, const LaunchList& ll, const int* active, hipStream_t s) {
  LAUNCH(k_copy_u, ll.nblocks, kBlock, L, ll, active);
}
void launch_fill_zero(bool fp64, const DevLevel* L, const LaunchList& ll, hipStream_t s) {
  if (fp64) LAUNCH(k_fill_zero<double>, ll.nblocks, kBlock, L, ll);
  else LAUNCH(k_fill_zero<float>, ll.nblocks, kBlock, L, ll);
}
void launch_ghost_wrap(double* a, int nx, int ny, int nz, int dir, hipStream_t s) {
  const size_t n = dir == 0 ? (size_t)(ny + 2) * (nz + 2)
                 : dir == 1 ? (size_t)(nx + 2) * (nz + 2) : (size_t)(nx + 2) * (ny + 2);
  LAUNCH(k_ghost_wrap, nb(n), kBlock, a, nx, ny, nz, dir);
}
void launch_ghost_fill(double* a, int nx, int ny, int nz, const GhostBC& bc, hipStream_t s) {
  const size_t n = 2 * ((size_t)(ny + 2) * (nz + 2) + (size_t)(nx + 2) * (nz + 2) +
                        (size_t)(nx + 2) * (ny + 2));
  LAUNCH(k_ghost_fill, nb(n), kBlock, a, nx, ny, nz, bc);
}
void launch_psource(const double* U, const double* V, const double* W, double* SRC, const double* rho,
                    const double* rdxc, const double* rdyc, const double* rdzc, int nx, int ny, int nz,
                    double rdt, hipStream_t s) {
  const unsigned plane = nb((size_t)(nx + 2) * (ny + 2));
  // Slabs of kProjK planes where they fill the device several times over (256^3
  // 123.5 us a call, with two planes 130.2).  Smaller grids are bound by a
  // thread's chain and take two planes, or one up to four workgroups per CU.
  // The kernel with one cell per thread and no march, with one plane, with two:
  // 24x24x14 2.68, 2.64, 2.80 us; 128x24x46 (672 workgroups of one plane) 3.40,
  // 3.24, 3.28; 96x96x64 (2508) 6.20, 5.32, 4.88; 160x112x80 11.96, 9.08, 8.64.
  const int K = plane * nb(nz + 2, kProjK) >= 4096 ? kProjK : plane * (unsigned)(nz + 2) > 1024 ? 2 : 1;
  const unsigned blocks = plane * nb(nz + 2, K);
#define PS(K) LAUNCH(k_psource<K>, blocks, kBlock, U, V, W, SRC, rho, rdxc, rdyc, rdzc, nx, ny, nz, rdt)
  if (K == kProjK) PS(kProjK);
  else if (K == 2) PS(2);
  else PS(1);
#undef PS
}
void launch_pgrad(const double* p, double* U, double* V, double* W, const double* rho,
                  const double* rdxe, const double* rdye, const double* rdze, int nx, int ny, int nz,
                  double dt, int wallmask, hipStream_t s) {
  LAUNCH(k_pgrad, nb((size_t)nx * ny * nz), kBlock, p, U, V, W, rho, rdxe, rdye, rdze, nx, ny, nz, dt,
         wallmask);
}
int divergence_blocks(int nx, int ny, int nz) {
  const long long tiles = (long long)nb((size_t)nx * ny) * nb(nz, kProjK);
  return (int)std::min<long long>(tiles, kDivBlocks);
}
void launch_divergence(const double* U, const double* V, const double* W, double* div,
                       const double* rdxc, const double* rdyc, const double* rdzc, const double* dxc,
                       const double* dyc, const double* dzc, int nx, int ny, int nz, double* partial,
                       hipStream_t s) {
  LAUNCH(k_divergence, divergence_blocks(nx, ny, nz), kBlock, U, V, W, div, rdxc, rdyc, rdzc, dxc, dyc,
         dzc, nx, ny, nz, partial);
}
void launch_divergence_finalize(const double* partial, int nblocks, double* out, hipStream_t s) {
  LAUNCH(k_divergence_finalize, 1, kDivFin, partial, nblocks, out);
}

}  // namespace amg
