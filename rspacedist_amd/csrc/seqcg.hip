// seqcg.hip — kscg_r (kscg8f.F90:98-472) and kscg_c (:492-1032) band by band, one code for real and
// complex bands.
//
// A band's iteration is a chain of vector operations on one band, a launch-bound workload: the
// plain sequence is about fifty launches and a host read per iteration.  Here it is eleven:
//   resid      eps, r = eps S psi - H psi, K r
//   dots       <S psi_j|K r> for the bands j <= l
//   apply      K r -= sum_j psi_j <S psi_j|K r>, with <r|K r>
//   gather     <p|K r>; expand: folded, times q, the projector part per list point
//   direction  S K r, P = K r + t P, S P and <p|P> alike
//   dots, apply  p = P - sum_j psi_j <S psi_j|P>, S p and <p|p> alike, with <p|S p>
//   expand     <p|p> times D, the projector part per list point
//   H          H p with its projector part, <p|H p> and <psi|H p>
//   update     the 2 x 2 step, psi, S psi, H psi, <p|psi>, with the next <psi|H psi>
// Scalars never leave the device: a kernel that needs a sum folds the partials of the launch
// before it, every work-group in the same order.  p is not normalised in memory; its norm enters
// the step's coefficients (H is linear).  A band that has converged is marked with the iteration
// it converged at, and the later launches of that band return at once.
// Each is bound by the time of a launch (3 to 9 us of device time; the bands' reads come from the
// caches).  One SCF step of four iterations: 40^3 points x 32 bands with S != 1 51.2 -> 10.6 ms,
// 32^3 x 24 complex bands 41.7 -> 7.9 ms (one launch per vector operation and a host read per
// iteration before).
#include "seqcg.hpp"

#include <algorithm>
#include <cmath>

namespace kukan {
namespace {

typedef double2 zt;
constexpr int NW = 256;  // threads of every kernel here
// Bands whose partials every work-group of k_seq_apply folds itself; with more a launch folds them
// first.  The two meet there: one / two arrays of 40^3 points take 19 / 33 us at 126 bands and
// 16 + 4 / 26 + 4 us at 130 with the fold launched.
constexpr int FOLD_MAX = 128;

// ---------------------------------------------------------------- arithmetic on double / double2
__device__ inline double re(double a) { return a; }
__device__ inline double re(zt a) { return a.x; }
__device__ inline void zero(double &a) { a = 0.0; }
__device__ inline void zero(zt &a) { a = make_double2(0.0, 0.0); }
__device__ inline double add(double a, double b) { return a + b; }
__device__ inline zt add(zt a, zt b) { return make_double2(a.x + b.x, a.y + b.y); }
__device__ inline double sub(double a, double b) { return a - b; }
__device__ inline zt sub(zt a, zt b) { return make_double2(a.x - b.x, a.y - b.y); }
__device__ inline double mul(double a, double b) { return a * b; }
__device__ inline zt mul(zt a, zt b) { return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
__device__ inline zt scl(double s, zt a) { return make_double2(s * a.x, s * a.y); }
__device__ inline double scl(double s, double a) { return s * a; }
__device__ inline double cmul(double a, double b) { return a * b; }  // conj(a) b
__device__ inline zt cmul(zt a, zt b) { return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x); }
__device__ inline double shfl(double v, int off) { return __shfl_down(v, off, 64); }
__device__ inline zt shfl(zt v, int off) { return make_double2(__shfl_down(v.x, off, 64), __shfl_down(v.y, off, 64)); }
__device__ inline double ratio(double a, double b) { return a / b; }  // a / b
__device__ inline zt ratio(zt a, zt b) {
  const double d = b.x * b.x + b.y * b.y;
  return scl(1.0 / d, cmul(b, a));
}
__device__ inline double mag(double a) { return a; }  // kscg_r's <r|K r>, kscg_c's modulus of it
__device__ inline double mag(zt a) { return hypot(a.x, a.y); }
template <class T>
__device__ inline T wave(T v) {
  for (int off = 32; off > 0; off >>= 1) v = add(v, shfl(v, off));
  return v;
}
// sum over the work-group, valid in thread 0
template <class T>
__device__ inline T group(T v, T *red4) {
  v = wave(v);
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = v;
  __syncthreads();
  const T s = add(add(add(red4[0], red4[1]), red4[2]), red4[3]);
  __syncthreads();
  return s;
}
// sum of np partials, the same in every thread of every work-group
template <class T>
__device__ inline T fold(const T *part, int np, T *red4) {
  T s;
  zero(s);
  for (int c = threadIdx.x; c < np; c += NW) s = add(s, part[c]);
  return group(s, red4);
}

// a norm that is an error, and 1 / sqrt of it: kscg_r stops at a NaN too, kscg_c does not
template <class T>
__device__ inline bool bad_norm(double v) { return sizeof(T) == 8 ? !(v > 0.0) : v <= 0.0; }
template <class T>
__device__ inline double rnorm(double v) { return bad_norm<T>(v) ? 0.0 : 1.0 / sqrt(v); }

// the band converged in an earlier iteration than `it`
__device__ inline bool over(const int *conv, int it) { return *conv != 0 && *conv < it; }

// ---------------------------------------------------------------- kernels
template <class T>
struct ResidArgs {
  int nx, ny, nz, px, py, pz, precon, npe, it;
  long n;
  double dv;
  const T *h, *s, *part_e;
  T *r, *k;
  double *eps;
  const int *conv;
};
template <class T>
__global__ __launch_bounds__(NW) void k_seq_resid(ResidArgs<T> a) {
  __shared__ T red[4];
  if (over(a.conv, a.it)) return;
  const double e = a.dv * re(fold(a.part_e, a.npe, red));
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.eps = e;
  const long plane = (long)a.nx * a.ny;
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n; i += (long)gridDim.x * NW) {
    const T c = sub(scl(e, a.s[i]), a.h[i]);
    a.r[i] = c;
    if (!a.precon) {
      a.k[i] = c;
      continue;
    }
    const unsigned u = (unsigned)i, row = u / (unsigned)a.nx;
    const int x = (int)(u - row * a.nx), y = (int)(row % (unsigned)a.ny), z = (int)(row / (unsigned)a.ny);
    auto at = [&](bool in, int per, long j) {
      T v;
      zero(v);
      if (in || per) v = sub(scl(e, a.s[j]), a.h[j]);
      return v;
    };
    const double w = 1.0 / 12.0;  // ksprecondition8f.F90:17-32
    T o = scl(w, at(x > 0, a.px, x > 0 ? i - 1 : i + a.nx - 1));
    o = add(o, scl(w, at(y > 0, a.py, y > 0 ? i - a.nx : i + plane - a.nx)));
    o = add(o, scl(w, at(z > 0, a.pz, z > 0 ? i - plane : i + plane * (a.nz - 1))));
    o = add(o, scl(0.5, c));
    o = add(o, scl(w, at(z < a.nz - 1, a.pz, z < a.nz - 1 ? i + plane : i - plane * (a.nz - 1))));
    o = add(o, scl(w, at(y < a.ny - 1, a.py, y < a.ny - 1 ? i + a.nx : i - plane + a.nx)));
    o = add(o, scl(w, at(x < a.nx - 1, a.px, x < a.nx - 1 ? i + 1 : i - a.nx + 1)));
    a.k[i] = o;
  }
}

// part[j][chunk] = sum over the chunk of conj(S_j) x, eight bands per work-group
template <class T>
__global__ __launch_bounds__(NW) void k_seq_dots(long n, long chunk, const T *S, int m, const T *x, T *part,
                                                 const int *conv, int it) {
  __shared__ T red[8][4];
  if (over(conv, it)) return;
  const int j0 = blockIdx.y * 8, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long i1 = min(n, (blockIdx.x + 1) * chunk);
  const T *col[8];
#pragma unroll
  for (int q = 0; q < 8; q++) col[q] = S + n * min(j0 + q, m - 1);
  T acc[8];
#pragma unroll
  for (int q = 0; q < 8; q++) zero(acc[q]);
  for (long i = blockIdx.x * chunk + threadIdx.x; i < i1; i += NW) {
    const T v = x[i];
#pragma unroll
    for (int q = 0; q < 8; q++) acc[q] = add(acc[q], cmul(col[q][i], v));
  }
#pragma unroll
  for (int q = 0; q < 8; q++) {
    const T s = wave(acc[q]);
    if (lane == 0) red[q][w] = s;
  }
  __syncthreads();
  if (threadIdx.x < 8 && j0 + (int)threadIdx.x < m) {
    const T *r = red[threadIdx.x];
    part[(long)(j0 + threadIdx.x) * gridDim.x + blockIdx.x] = add(add(add(r[0], r[1]), r[2]), r[3]);
  }
}
// one work-group per band: its partials folded, times dv (used where the bands are too many for
// every work-group of the next launch to fold them all)
template <class T>
__global__ __launch_bounds__(NW) void k_seq_fold(const T *part, int np, double dv, T *out, const int *conv, int it) {
  __shared__ T red[4];
  if (over(conv, it)) return;
  const T s = fold(part + (long)blockIdx.x * np, np, red);
  if (threadIdx.x == 0) out[blockIdx.x] = scl(dv, s);
}

// y -= sum_{j < m} B_j c_j for up to two arrays over the grid and the projections, with c_j the
// folded sums (FOLDED) or dv sum(part[j]); partials of conj(y0) z (z null: of the second array,
// or the first)
template <class T>
struct ApplyArgs {
  long n, n1;
  int m, np, two;
  double dv;
  const T *part, *B[2], *in[2], *cin, *cB, *z;
  T *out[2], *cout, *res;
  const int *conv;
  int it;
};
template <class T, bool FOLDED>
__global__ __launch_bounds__(NW) void k_seq_apply(ApplyArgs<T> a) {
  __shared__ T lds[FOLDED ? 1 : FOLD_MAX];
  __shared__ T red[4];
  if (over(a.conv, a.it)) return;
  const T *c = FOLDED ? a.part : lds;
  if constexpr (!FOLDED) {
    for (int j0 = 0; j0 < a.m; j0 += NW / 8) {  // eight threads per band: one round trip for 32 bands
      const int j = j0 + (threadIdx.x >> 3), q0 = threadIdx.x & 7;
      T s;
      zero(s);
      if (j < a.m)
        for (int q = q0; q < a.np; q += 8) s = add(s, a.part[(long)j * a.np + q]);
      for (int off = 4; off > 0; off >>= 1) s = add(s, shfl(s, off));
      if (j < a.m && q0 == 0) lds[j] = scl(a.dv, s);
    }
    __syncthreads();
  }
  T dot;
  zero(dot);
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n; i += (long)gridDim.x * NW) {
    T y0 = a.in[0][i], y1 = y0;
    const T *b0 = a.B[0] + i;
#pragma unroll 8
    for (int j = 0; j < a.m; j++) y0 = sub(y0, mul(b0[a.n * j], c[j]));
    a.out[0][i] = y0;
    if (a.two) {
      y1 = a.in[1][i];
      const T *b1 = a.B[1] + i;
#pragma unroll 8
      for (int j = 0; j < a.m; j++) y1 = sub(y1, mul(b1[a.n * j], c[j]));
      a.out[1][i] = y1;
    } else {
      y1 = y0;
    }
    dot = add(dot, cmul(y0, a.z ? a.z[i] : y1));
  }
  if (a.cout)
    for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n1; i += (long)gridDim.x * NW) {
      T y = a.cin[i];
#pragma unroll 8
      for (int j = 0; j < a.m; j++) y = sub(y, mul(a.cB[i + a.n1 * j], c[j]));
      a.cout[i] = y;
    }
  dot = group(dot, red);
  if (threadIdx.x == 0) a.res[blockIdx.x] = dot;
}

// v, S v and <p|v> times 1 / sqrt(dv Re sum(part)); a norm that is not positive raises the flag
template <class T>
__global__ __launch_bounds__(NW) void k_seq_scale(long n, long n1, double dv, const T *part, int np, T *v, T *sv, T *cv,
                                                  int band, int *flag) {
  __shared__ T red[4];
  const double t = dv * re(fold(part, np, red));
  if (blockIdx.x == 0 && threadIdx.x == 0 && bad_norm<T>(t) && !*flag) *flag = band;
  const double f = rnorm<T>(t);
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < n; i += (long)gridDim.x * NW) {
    v[i] = scl(f, v[i]);
    if (sv != v) sv[i] = scl(f, sv[i]);
  }
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < n1; i += (long)gridDim.x * NW) cv[i] = scl(f, cv[i]);
}

// projector tables of one call
struct Proj {
  const int *act, *lst, *row_ptr;
  const int2 *ent;
  const double *vnl;
  const zt *ph;
  int nact, num_list, nprjmx;
};
__device__ inline double phased(const Proj &, long, double u) { return u; }
__device__ inline zt phased(const Proj &p, long k, zt u) { return mul(p.ph[k], u); }
__device__ inline double unphased(const Proj &, long, double u) { return u; }
__device__ inline zt unphased(const Proj &p, long k, zt u) { return cmul(p.ph[k], u); }

// part[slot][j][chunk] of <p_j|u>: the list in gridDim.x chunks, nine projectors per sweep
template <class T>
__global__ __launch_bounds__(NW) void k_seq_gather(Proj p, const T *u, T *part, const int *conv, int it) {
  __shared__ T red[9][4];
  if (over(conv, it)) return;
  const int a = blockIdx.y, slot = p.act[5 * a], natinf = p.act[5 * a + 1], iprj = p.act[5 * a + 2];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const long lo = (long)p.num_list * slot;
  for (int j0 = 0; j0 < iprj; j0 += 9) {
    T acc[9];
#pragma unroll
    for (int j = 0; j < 9; j++) zero(acc[j]);
    for (int k = blockIdx.x * NW + threadIdx.x; k < natinf; k += gridDim.x * NW) {
      const T v = phased(p, lo + k, u[p.lst[lo + k] - 1]);
#pragma unroll
      for (int j = 0; j < 9; j++)
        if (j0 + j < iprj) acc[j] = add(acc[j], scl(p.vnl[lo * p.nprjmx + k + (long)p.num_list * (j0 + j)], v));
    }
#pragma unroll
    for (int j = 0; j < 9; j++) {
      const T s = wave(acc[j]);
      if (lane == 0) red[j][w] = s;
    }
    __syncthreads();
    if (threadIdx.x < 9 && j0 + (int)threadIdx.x < iprj) {
      const T *r = red[threadIdx.x];
      part[((long)p.nprjmx * slot + j0 + threadIdx.x) * gridDim.x + blockIdx.x] =
          add(add(add(r[0], r[1]), r[2]), r[3]);
    }
    __syncthreads();
  }
}

// Per active atom: cp = sum of its gather partials (nch > 0), coef = X cp / dV, and
// val(k) = conj(phase) sum_j coef_j vnl(k, j) for its list points (X null: cp alone).  Read along
// the list the projector values are contiguous; the kernels that add the projector part then load
// one value per grid point and entry instead of iprj scattered ones behind two index loads (40^3
// points, 12 atoms x 9 projectors: the H kernel 20.8 -> 8.9 us, the direction 10.1 -> 5.1 us).
// The real path multiplies by X^T (nonlocaloperation8f.F90:180-198), the complex one by X (:300-331).
template <class T>
__global__ __launch_bounds__(NW) void k_seq_expand(Proj p, const T *part, int nch, T *cp, const double *X, int per_atom,
                                                   int ns, int nums, double dvinv, T *val, const int *conv, int it) {
  extern __shared__ double shm[];
  T *c = (T *)shm, *coef = c + p.nprjmx;
  if (over(conv, it)) return;
  const int a = blockIdx.y, slot = p.act[5 * a], natinf = p.act[5 * a + 1], iprj = p.act[5 * a + 2];
  const int na = p.act[5 * a + 3], ispe = p.act[5 * a + 4], t = threadIdx.x;
  const long o = (long)p.nprjmx * slot, lo = (long)p.num_list * slot;
  for (int j = t; j < iprj; j += NW) {
    T s;
    if (nch > 0) {
      zero(s);
#pragma unroll 4
      for (int q = 0; q < nch; q++) s = add(s, part[(o + j) * nch + q]);
      if (blockIdx.x == 0) cp[o + j] = s;
    } else {
      s = cp[o + j];
    }
    c[j] = s;
  }
  if (!X) return;
  __syncthreads();
  const double *Xa = X + (long)p.nprjmx * p.nprjmx * (per_atom ? (ns - 1) + (long)nums * na : ispe);
  for (int j = t; j < iprj; j += NW) {
    T s;
    zero(s);
#pragma unroll 4
    for (int i = 0; i < iprj; i++)
      s = add(s, scl(sizeof(T) == 8 ? Xa[i + (long)p.nprjmx * j] : Xa[j + (long)p.nprjmx * i], c[i]));
    coef[j] = scl(dvinv, s);
  }
  __syncthreads();
  for (int k = blockIdx.x * NW + t; k < natinf; k += gridDim.x * NW) {
    const double *v = p.vnl + lo * p.nprjmx + k;
    T s;
    zero(s);
#pragma unroll 8
    for (int j = 0; j < iprj; j++) s = add(s, scl(v[(long)p.num_list * j], coef[j]));
    val[lo + k] = unphased(p, lo + k, s);
  }
}

// projector part at grid point r
template <class T>
__device__ inline T entries(const Proj &p, long r, const T *val) {
  T s;
  zero(s);
  const int e1 = p.row_ptr[r + 1];
  for (int e = p.row_ptr[r]; e < e1; e++) {
    const int2 en = p.ent[e];
    s = add(s, val[en.y + (long)p.num_list * en.x]);
  }
  return s;
}

// r2 = dv sum(part), t = r2 / r1 (0 at a reset); P = K r + t P, S P = S K r + t S P, <p|P> alike
template <class T>
struct DirArgs {
  long n, n1;
  int np, reset, slot, it;  // rr[slot] receives r2, rr[1 - slot] holds r1
  double dv;
  const T *part, *kr, *cr, *sproj;  // sproj (projector part of S K r) null: S = 1
  T *rr, *P, *SP, *cP;
  double *resid;
  const int *conv;
};
template <class T>
__global__ __launch_bounds__(NW) void k_seq_direction(DirArgs<T> a, Proj p) {
  __shared__ T red[4];
  if (over(a.conv, a.it)) return;
  const T r2 = scl(a.dv, fold(a.part, a.np, red));
  T t;
  zero(t);
  if (!a.reset) t = ratio(r2, a.rr[1 - a.slot]);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a.rr[a.slot] = r2;
    *a.resid = mag(r2);
  }
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n; i += (long)gridDim.x * NW) {
    const T k = a.kr[i];
    a.P[i] = a.reset ? k : add(k, mul(t, a.P[i]));
    if (a.SP != a.P) {
      const T sk = a.sproj ? add(k, entries(p, i, a.sproj)) : k;
      a.SP[i] = a.reset ? sk : add(sk, mul(t, a.SP[i]));
    }
  }
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n1; i += (long)gridDim.x * NW)
    a.cP[i] = a.reset ? a.cr[i] : add(a.cr[i], mul(t, a.cP[i]));
}

// out = H u (twisted by the Bloch phases for complex bands) on 16 x 16-column tiles of TZ planes,
// one batch of loads and one barrier per tile as the Hartree CG's direction kernel; partials of
// Re conj(u) out and conj(psi) out
template <class T>
struct HArgs {
  int nx, ny, nz, px, py, pz, ntx, nty, ntz, it;
  double cx[9], cy[9], cz[9], c0;
  zt ex[9], ey[9], ez[9];
  const double *veff;
  const T *u, *psi, *val;  // val null: no projectors
  T *out, *part_u, *part_psi;
  const int *conv;
};
__device__ inline int wrap(int i, int n) {  // also for an axis shorter than the stencil's reach
  i %= n;
  return i < 0 ? i + n : i;
}
__device__ inline double pair(double c, zt, double lo, double hi) { return c * (lo + hi); }
__device__ inline zt pair(double c, zt e, zt lo, zt hi) { return scl(c, add(cmul(e, lo), mul(e, hi))); }
template <class T, int NF, int TZ>
__global__ __launch_bounds__(NW) void k_seq_h(HArgs<T> a, Proj p) {
  constexpr int W = 16 + 2 * NF, NZ = TZ + 2 * NF;
  constexpr int NXH = (2 * NF * 16 * TZ + NW - 1) / NW, NYH = NXH;
  __shared__ T box[TZ][W][W];
  __shared__ T red[4];
  if (a.conv && over(a.conv, a.it)) return;
  const int t = threadIdx.x, lx = t & 15, ly = t >> 4;
  const long plane = (long)a.nx * a.ny;
  const int ntile = a.ntx * a.nty * a.ntz;
  T su, sp;
  zero(su);
  zero(sp);
  for (int tile = blockIdx.x; tile < ntile; tile += gridDim.x) {
    const int x0 = tile % a.ntx * 16, y0 = tile / a.ntx % a.nty * 16, z0 = tile / (a.ntx * a.nty) * TZ;
    const int ex = min(16, a.nx - x0), ey = min(16, a.ny - y0), ez = min(TZ, a.nz - z0);
    const bool act = lx < ex && ly < ey;
    const long col = act ? x0 + lx + (long)a.nx * (y0 + ly) : 0;
    T v[NZ], hx[NXH], hy[NYH];
    int ix[NXH], iy[NYH];
#pragma unroll
    for (int j = 0; j < NZ; j++) {
      int z = z0 + j - NF;
      bool ok = act && z < z0 + ez + NF;
      if (z < 0 || z >= a.nz) {
        ok = ok && a.pz;
        z = wrap(z, a.nz);
      }
      zero(v[j]);
      if (ok) v[j] = a.u[col + plane * z];
    }
#pragma unroll
    for (int h = 0; h < NXH; h++) {
      const int i = t + NW * h, c = i % (2 * NF), row = i / (2 * NF) % 16, pl = i / (2 * NF * 16);
      const int cx = c < NF ? c - NF : ex + c - NF;
      bool ok = pl < ez && row < ey;
      ix[h] = ok ? (pl * W + row + NF) * W + cx + NF : -1;
      int X = x0 + cx;
      if (X < 0 || X >= a.nx) {
        ok = ok && a.px;
        X = wrap(X, a.nx);
      }
      zero(hx[h]);
      if (ok) hx[h] = a.u[X + (long)a.nx * (y0 + row) + plane * (z0 + pl)];
    }
#pragma unroll
    for (int h = 0; h < NYH; h++) {
      const int i = t + NW * h, c = i % 16, row = i / 16 % (2 * NF), pl = i / (16 * 2 * NF);
      const int cy = row < NF ? row - NF : ey + row - NF;
      bool ok = pl < ez && c < ex;
      iy[h] = ok ? (pl * W + cy + NF) * W + c + NF : -1;
      int Y = y0 + cy;
      if (Y < 0 || Y >= a.ny) {
        ok = ok && a.py;
        Y = wrap(Y, a.ny);
      }
      zero(hy[h]);
      if (ok) hy[h] = a.u[x0 + c + (long)a.nx * Y + plane * (z0 + pl)];
    }
    if (tile != (int)blockIdx.x) __syncthreads();  // the previous tile's values have been read
    if (act) {
#pragma unroll
      for (int j = 0; j < TZ; j++) box[j][ly + NF][lx + NF] = v[j + NF];
    }
    T *flat = &box[0][0][0];
#pragma unroll
    for (int h = 0; h < NXH; h++)
      if (ix[h] >= 0) flat[ix[h]] = hx[h];
#pragma unroll
    for (int h = 0; h < NYH; h++)
      if (iy[h] >= 0) flat[iy[h]] = hy[h];
    __syncthreads();
    if (act) {
#pragma unroll
      for (int j = 0; j < TZ; j++) {
        if (j >= ez) break;
        const long r = col + plane * (z0 + j);
        const T *c = &box[j][ly + NF][lx + NF];
        T s = scl(a.c0 + (a.veff ? a.veff[r] : 0.0), v[j + NF]);
#pragma unroll
        for (int m = 1; m <= NF; m++) s = add(s, pair(a.cx[m], a.ex[m], c[-m], c[m]));
#pragma unroll
        for (int m = 1; m <= NF; m++) s = add(s, pair(a.cy[m], a.ey[m], c[-m * W], c[m * W]));
#pragma unroll
        for (int m = 1; m <= NF; m++) s = add(s, pair(a.cz[m], a.ez[m], v[j + NF - m], v[j + NF + m]));
        if (a.val) s = add(s, entries(p, r, a.val));
        a.out[r] = s;
        su = add(su, cmul(v[j + NF], s));
        sp = add(sp, cmul(a.psi[r], s));
      }
    }
  }
  su = group(su, red);
  sp = group(sp, red);
  if (t == 0) {
    a.part_u[blockIdx.x] = su;
    a.part_psi[blockIdx.x] = sp;
  }
}

// the 2 x 2 Rayleigh-Ritz step: kscg_r_05 (kscg8f.F90:1197-1230) and kscg_c_05 (:1233-1274)
__device__ inline void step(double sv, double pp, double sa, double &al, double &be) {
  const double eps = 1.0e-14;
  al = 1.0;
  be = 0.0;
  const double gamma = (sv + pp) * 0.5 - sqrt((sv - pp) * (sv - pp) * 0.25 + sa * sa);
  if (fabs((sv - gamma) / gamma) > eps) {
    const double d = sqrt(sa * sa + (sv - gamma) * (sv - gamma));
    al = sa / d;
    be = -(sv - gamma) / d;
  }
  if (al < eps) {
    al = -al;
    be = -be;
  }
}
__device__ inline void step(double sv, double pp, zt sa, double &al, zt &be) {
  const double eps = 1.0e-14, s2 = sa.x * sa.x + sa.y * sa.y;
  al = 1.0;
  zero(be);
  const double gamma = (sv + pp) * 0.5 - sqrt((sv - pp) * (sv - pp) * 0.25 + s2);
  if (fabs((sv - gamma) / gamma) > eps) {
    const double d = sqrt(s2 + (sv - gamma) * (sv - gamma));
    const zt ca = scl(1.0 / d, sa);
    be = make_double2(-(sv - gamma) / d, 0.0);
    al = hypot(ca.x, ca.y);
    if (al > eps) be = scl(al, ratio(be, ca));
  }
}
// the step with p / |p|; psi, S psi, H psi, <p|psi> and the partials of conj(psi) H psi
template <class T>
struct UpdArgs {
  long n, n1;
  int npn, nph, it, band;
  double dv, epssd;
  const T *part_n, *part_u, *part_psi;  // <p|S p>, <p|H p>, <psi|H p>
  const double *eps, *resid;
  const T *p, *sp, *hp, *cp;
  T *psi, *spsi, *hpsi, *cps, *part_e;
  int *conv, *flag;
};
template <class T>
__global__ __launch_bounds__(NW) void k_seq_update(UpdArgs<T> a) {
  __shared__ T red[4];
  if (over(a.conv, a.it)) return;
  const double nn = a.dv * re(fold(a.part_n, a.npn, red));
  const double f = rnorm<T>(nn);
  const double pap = a.dv * f * f * re(fold(a.part_u, a.nph, red));
  const T sap = scl(a.dv * f, fold(a.part_psi, a.nph, red));
  double al;
  T be;
  step(*a.eps, pap, sap, al, be);
  const T bf = scl(f, be);
  T dot;
  zero(dot);
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n; i += (long)gridDim.x * NW) {
    const T x = add(scl(al, a.psi[i]), mul(bf, a.p[i])), h = add(scl(al, a.hpsi[i]), mul(bf, a.hp[i]));
    a.psi[i] = x;
    a.hpsi[i] = h;
    if (a.spsi != a.psi) a.spsi[i] = add(scl(al, a.spsi[i]), mul(bf, a.sp[i]));
    dot = add(dot, cmul(x, h));
  }
  for (long i = blockIdx.x * (long)NW + threadIdx.x; i < a.n1; i += (long)gridDim.x * NW)
    a.cps[i] = add(scl(al, a.cps[i]), mul(bf, a.cp[i]));
  dot = group(dot, red);
  if (threadIdx.x == 0) {
    a.part_e[blockIdx.x] = dot;
    if (blockIdx.x == 0) {
      if (bad_norm<T>(nn) && !*a.flag) *a.flag = a.band;
      if (sqrt(*a.resid) < a.epssd) *a.conv = a.it;  // later iterations of this band do nothing
    }
  }
}
__global__ void k_seq_clear(int n, int *v) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) v[i] = 0;
}

template <class T, int TZ>
void launch_h_tz(int nf, const HArgs<T> &a, const Proj &p, int grid, hipStream_t s) {
  switch (nf) {
#define CASE(N) case N: hipLaunchKernelGGL((k_seq_h<T, N, TZ>), dim3(grid), dim3(NW), 0, s, a, p); break;
    CASE(1) CASE(2) CASE(3) CASE(4) CASE(5) CASE(6) CASE(7) CASE(8)
#undef CASE
    default: throw Error(1, "error in kslaplacian_r! This subroutine is for nf in 1-8.");
  }
}

// -------------------------------------------------------------------------------- driver
template <class T>
void run(Ctx &c, const SeqCgArgs<T> &a, const zt *ph, const double *k, const char *gs_msg, const char *p_msg) {
  const Grid &g = c.g;
  const NonlocalPlan &pl = c.pl;
  const long n = g.n(), n1 = (long)pl.nprjmx * pl.num_ppcell;
  const double dv = g.dv();
  hipStream_t s = c.s;
  const bool per[3] = {g.nperi >= 1, g.nperi >= 2, g.nperi >= 3};
  const bool real = sizeof(T) == 8;
  if (real && (g.nx < g.nf || g.ny < g.nf || g.nz < g.nf))
    throw Error(1, "grid smaller than the finite-difference radius");
  const bool gathers = pl.nact > 0 && a.M > 0 && (a.nsdmax > 0 || (a.recompute && a.northo > 0));
  if (gathers && real && pl.max_iprj > 32)
    throw Error(1, "nonlocal projectors: more than 32 per atom are not supported");
  if (gathers && !real && pl.max_iprj > 16) throw Error(1, "complex path: more than 16 projectors per atom");
  auto buf = [&](const char *tag, size_t cnt) {
    return (T *)c.buf((std::string(tag) + (sizeof(T) == 16 ? ".z" : ".r")).c_str(), std::max<size_t>(1, cnt) * sizeof(T) / 8);
  };
  const bool same = a.spsi == a.psi;  // S psi is psi: no array of its own
  T *r = buf("seq.r", n), *kr = buf("seq.kr", n), *P = buf("seq.P", n), *SP = same ? P : buf("seq.SP", n);
  T *p = buf("seq.p", n), *sp = same ? p : buf("seq.sp", n), *hp = buf("seq.hp", n);
  T *cr = buf("seq.cr", n1), *cP = buf("seq.cP", n1), *cp = buf("seq.cp", n1), *val = buf("seq.val", (size_t)pl.num_list * pl.num_ppcell);
  // work-groups of the elementwise kernels and of the dot products (fewer: their partials are
  // folded by every work-group of the next launch)
  const int nw = (int)std::max(1L, std::min(512L, (n + NW - 1) / NW));
  const long chunk = std::max(512L, (n + 63) / 64);
  const int nd = (int)((n + chunk - 1) / chunk);
  const int nch = std::max(1, std::min(16, 256 / std::max(1, pl.nact)));  // list chunks per atom
  HArgs<T> h{};
  h.nx = g.nx; h.ny = g.ny; h.nz = g.nz; h.px = per[0]; h.py = per[1]; h.pz = per[2];
  double w[9];
  fd_coefficients(g.nf, w);
  for (int m = 0; m < 9; m++) {
    h.cx[m] = w[m] / g.dx / g.dx * (-0.5);
    h.cy[m] = w[m] / g.dy / g.dy * (-0.5);
    h.cz[m] = w[m] / g.dz / g.dz * (-0.5);
    if (k) {
      h.ex[m] = make_double2(std::cos(k[0] * m * g.dx), std::sin(k[0] * m * g.dx));
      h.ey[m] = make_double2(std::cos(k[1] * m * g.dy), std::sin(k[1] * m * g.dy));
      h.ez[m] = make_double2(std::cos(k[2] * m * g.dz), std::sin(k[2] * m * g.dz));
    }
  }
  h.c0 = h.cx[0] + h.cy[0] + h.cz[0];
  h.ntx = (g.nx + 15) / 16;
  h.nty = (g.ny + 15) / 16;
  const int tz = (long)h.ntx * h.nty * ((g.nz + 1) / 2) <= 2048 ? 2 : 4;
  h.ntz = (g.nz + tz - 1) / tz;
  const int nt = (int)std::min(512L, (long)h.ntx * h.nty * h.ntz);
  h.veff = a.veff;
  T *part_d = buf("seq.part_d", (size_t)nd * a.M), *cfold = buf("seq.cfold", a.M);
  T *part_a = buf("seq.part_a", nw), *part_n = buf("seq.part_n", nw), *part_e = buf("seq.part_e", std::max(nw, nt));
  T *part_u = buf("seq.part_u", nt), *part_psi = buf("seq.part_psi", nt), *part_g = buf("seq.part_g", (size_t)n1 * nch);
  T *rr = buf("seq.rr", 4);
  int *conv = (int *)scratch("seq.conv", sizeof(int) * (a.M + 2)), *flag = conv + a.M;
  hipLaunchKernelGGL(k_seq_clear, dim3((a.M + 2 + 255) / 256), dim3(256), 0, s, a.M + 2, conv);
  launch_fill(n1 * (long)(sizeof(T) / 8), 0.0, (double *)cr, s);  // inactive slots stay zero
  launch_fill(n1 * (long)(sizeof(T) / 8), 0.0, (double *)cp, s);
  Proj q{};
  q.act = pl.act; q.lst = pl.lst; q.row_ptr = pl.row_ptr; q.ent = pl.ent; q.vnl = pl.vnl;
  q.ph = ph; q.nact = pl.nact; q.num_list = pl.num_list; q.nprjmx = pl.nprjmx;
  const bool proj = pl.nact > 0 && pl.nent > 0;  // some grid point has projectors

  // conj(S_j) x for the first m bands; afterwards `part` / `np` hold each band's partials
  auto dots = [&](int m, const T *x, const int *cv, int it, ApplyArgs<T> &ap) {
    hipLaunchKernelGGL((k_seq_dots<T>), dim3(nd, (m + 7) / 8), dim3(NW), 0, s, n, chunk, a.spsi, m, x, part_d, cv, it);
    ap.part = part_d;
    ap.np = nd;
    if (m > FOLD_MAX) {
      hipLaunchKernelGGL((k_seq_fold<T>), dim3(m), dim3(NW), 0, s, part_d, nd, dv, cfold, cv, it);
      ap.part = cfold;
    }
  };
  // y0 (and y1, and the projections) minus the projection on the first m bands
  auto apply = [&](int m, const T *x0, T *y0, const T *x1, T *y1, const T *cx, T *cy, const T *z, T *res, const int *cv,
                   int it) {
    ApplyArgs<T> ap{};
    if (m > 0) dots(m, x0, cv, it, ap);
    ap.n = n; ap.n1 = cy ? n1 : 0; ap.m = m; ap.two = y1 != nullptr; ap.dv = dv;
    ap.B[0] = a.psi; ap.B[1] = a.spsi; ap.in[0] = x0; ap.in[1] = x1; ap.out[0] = y0; ap.out[1] = y1;
    ap.cin = cx; ap.cB = a.cps; ap.cout = cy; ap.z = z; ap.res = res; ap.conv = cv; ap.it = it;
    if (m > FOLD_MAX) hipLaunchKernelGGL((k_seq_apply<T, true>), dim3(nw), dim3(NW), 0, s, ap);
    else hipLaunchKernelGGL((k_seq_apply<T, false>), dim3(nw), dim3(NW), 0, s, ap);
  };
  auto expand = [&](const T *pg, int chunks, T *cc, bool H, const int *cv, int it) {
    const double *X = H ? c.dij : c.q_zero ? nullptr : c.sss;
    if (pl.nact > 0 && (chunks > 0 || X))
      hipLaunchKernelGGL((k_seq_expand<T>), dim3(X ? std::max(1, (pl.max_natinf + NW - 1) / NW) : 1, pl.nact), dim3(NW),
                         2 * sizeof(T) * pl.nprjmx, s, q, pg, chunks, cc, X, H ? 1 : 0, a.ns, pl.nums, 1.0 / dv, val, cv,
                         it);
  };
  auto ham = [&](const T *u, T *out, const T *psi, T *pu, T *pp, const int *cv, int it) {
    h.u = u; h.out = out; h.psi = psi; h.val = proj ? val : nullptr; h.part_u = pu; h.part_psi = pp;
    h.conv = cv; h.it = it;
    if (tz == 2) launch_h_tz<T, 2>(g.nf, h, q, nt, s);
    else launch_h_tz<T, 4>(g.nf, h, q, nt, s);
  };

  std::vector<int> hc(a.M + 2);
  for (int l = 0; l < a.M; l++) {
    T *psi = a.psi + n * l, *spsi = a.spsi + n * l, *hpsi = a.hpsi + n * l, *cps = a.cps + n1 * l;
    int *cv = conv + l;
    // orthonormalise against the lower bands (orthogonalization8f.F90:316-369)
    for (int loop = 0; loop < a.northo; loop++) {
      if (a.recompute && !real) launch_fill(2 * n1, 0.0, (double *)cps, s);
      if (a.recompute && pl.nact > 0) {
        hipLaunchKernelGGL((k_seq_gather<T>), dim3(nch, pl.nact), dim3(NW), 0, s, q, psi, part_g, cv, 0);
        expand(part_g, nch, cps, false, cv, 0);
      }
      if (a.recompute && !same) {  // S psi = psi + q part, as a direction that starts afresh
        DirArgs<T> d{};
        d.n = n; d.part = part_a; d.reset = 1; d.kr = psi; d.sproj = proj && !c.q_zero ? val : nullptr;
        d.rr = rr; d.P = P; d.SP = spsi; d.resid = (double *)(rr + 2); d.conv = cv;
        hipLaunchKernelGGL((k_seq_direction<T>), dim3(nw), dim3(NW), 0, s, d, q);
      }
      apply(l, psi, psi, same ? nullptr : spsi, same ? nullptr : spsi, cps, n1 > 0 ? cps : nullptr, nullptr, part_a, cv, 0);
      hipLaunchKernelGGL((k_seq_scale<T>), dim3(nw), dim3(NW), 0, s, n, n1, dv, part_a, nw, psi, spsi, cps,
                         l + 1, flag);
    }
    expand(nullptr, 0, cps, true, cv, 0);
    ham(psi, hpsi, psi, part_e, part_psi, nullptr, 0);
    int npe = nt;
    for (int it = 1; it <= a.nsdmax; it++) {
      const bool reset = it == 1 || it == 10 || (it - 1) % 200 == 0 || a.nkscg != 1;
      ResidArgs<T> ra{};
      ra.nx = g.nx; ra.ny = g.ny; ra.nz = g.nz; ra.px = per[0]; ra.py = per[1]; ra.pz = per[2];
      ra.precon = a.nprecon_cg == 1; ra.npe = npe; ra.it = it; ra.n = n; ra.dv = dv; ra.h = hpsi; ra.s = spsi;
      ra.part_e = part_e; ra.r = r; ra.k = kr; ra.eps = a.sval + l; ra.conv = cv;
      hipLaunchKernelGGL((k_seq_resid<T>), dim3(nw), dim3(NW), 0, s, ra);
      for (int loop = 0; loop < std::max(1, a.northo); loop++)
        apply(a.northo > 0 ? l + 1 : 0, kr, kr, nullptr, nullptr, nullptr, nullptr, r, part_a, cv, it);
      if (pl.nact > 0) {
        hipLaunchKernelGGL((k_seq_gather<T>), dim3(nch, pl.nact), dim3(NW), 0, s, q, kr, part_g, cv, it);
        expand(part_g, nch, cr, false, cv, it);
      }
      DirArgs<T> d{};
      d.n = n; d.n1 = n1; d.np = nw; d.reset = reset; d.slot = it & 1; d.it = it; d.dv = dv; d.part = part_a;
      d.kr = kr; d.cr = cr; d.sproj = proj && !c.q_zero ? val : nullptr; d.rr = rr; d.P = P; d.SP = SP; d.cP = cP;
      d.resid = a.resid + l; d.conv = cv;
      hipLaunchKernelGGL((k_seq_direction<T>), dim3(nw), dim3(NW), 0, s, d, q);
      for (int loop = 0; loop < std::max(1, a.northo); loop++) {
        const bool first = loop == 0;
        apply(a.northo > 0 ? l + 1 : 0, first ? P : p, p, same ? nullptr : first ? SP : sp, same ? nullptr : sp, first ? cP : cp,
              n1 > 0 ? cp : nullptr, nullptr, part_n, cv, it);
      }
      expand(nullptr, 0, cp, true, cv, it);
      ham(p, hp, psi, part_u, part_psi, cv, it);
      UpdArgs<T> u{};
      u.n = n; u.n1 = n1; u.npn = nw; u.nph = nt; u.it = it; u.band = l + 1; u.dv = dv; u.epssd = a.epssd; u.part_n = part_n;
      u.part_u = part_u; u.part_psi = part_psi; u.eps = a.sval + l; u.resid = a.resid + l; u.p = p; u.sp = sp; u.hp = hp;
      u.cp = cp; u.psi = psi; u.spsi = spsi; u.hpsi = hpsi; u.cps = cps; u.part_e = part_e; u.conv = cv; u.flag = flag + 1;
      hipLaunchKernelGGL((k_seq_update<T>), dim3(nw), dim3(NW), 0, s, u);
      npe = nw;
      if (it % 8 == 0 && it < a.nsdmax) {  // long runs: stop launching for a band that is done
        int done = 0;
        HIPCK(hipMemcpyAsync(&done, cv, sizeof(int), hipMemcpyDeviceToHost, s));
        sync();
        if (done) break;
      }
    }
    HIPCK(hipGetLastError());
  }
  HIPCK(hipMemcpyAsync(hc.data(), conv, sizeof(int) * (a.M + 2), hipMemcpyDeviceToHost, s));
  sync();
  for (int l = 0; l < a.M; l++) {
    const int its = hc[l] ? hc[l] : a.nsdmax;
    // as the reference's per-iteration test: a band fails it in its last permitted iteration only
    *a.ksconv = *a.ksconv && (a.nsdmax < 1 || hc[l] != 0);
    *a.ksitmax = std::max(*a.ksitmax, its);
  }
  const int gs_bad = hc[a.M], p_bad = hc[a.M + 1];  // the first band of each error, or 0
  if (gs_bad && (real || !p_bad || gs_bad <= p_bad)) throw Error(2, gs_msg);
  if (p_bad) throw Error(2, p_msg);
}

}  // namespace

void seq_cg(Ctx &c, const SeqCgArgs<double> &a) {
  run<double>(c, a, nullptr, nullptr, "orthogonalization_r_01 (3): wf has negative norm", "kscg_r: pvec has negative norm");
}

void seq_cg(ZCtx &z, const SeqCgArgs<double2> &a) {
  const double k[3] = {z.kx, z.ky, z.kz};
  run<double2>(z.c, a, z.ph, k, "orthogonalization_c_01 (3): wf has negative norm", "kscg_c: pvec has negative norm");
}

}  // namespace kukan
