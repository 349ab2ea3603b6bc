// batch.hip — batching pattern: many independent periodic systems of different grid sizes
// advanced together.  Per system and step: H psi for all bands, one preconditioned
// steepest-descent band update with a 2x2 Rayleigh-Ritz per band (the first, reset iteration
// of kscg_r, kscg8f.F90:98-472 and :1197-1230), the orthonormalisation of the bands (FP64
// Cholesky-QR, the Q of orthogonalization8f.F90:93-376), then the Hartree CG solve of
// rho = sum_l psi_l^2 (scf_hartree8f.F90).
//
// Batched mode: every stencil pass of all systems is one persistent launch (the items of all
// systems in one work list), per-band arithmetic runs as launches over a global band table,
// the Hartree CG of all systems advances as device-side iteration blocks of two launches per
// iteration with per-system stop flags (hartree_cg.hip), and the band step and the Hartree block are captured once as HIP graphs and
// replayed.  Loop mode runs the same kernels system by system (one launch per system and
// pass, no graphs): the comparison the batching is measured against.  Both modes compute
// bit-identical results.  The stencil tile (points per thread) and the persistent grid size
// are chosen by timing the candidates on first use.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <memory>
#include <string>
#include <vector>

#include "hartree_cg.hpp"
#include "kukan_hip.h"
#include "kukan_internal.hpp"
#include "solvers.hpp"

namespace kukan {
namespace {

// One band of one system in the global band table.
struct BandRef {
  double *psi, *hpsi, *p, *hp;  // band columns
  const double *part;           // this band's stencil+projector partial sums
  long n;                       // grid points
  int nparts;
  double dv;
};
constexpr int BCH = 64;  // work-groups per band for band reductions

// which = 1: r0 = <psi|p>, r1 = <p|p>; which = 2: r0 = <psi|hp>  (times dV, fixed order)
__global__ __launch_bounds__(256) void k_band_dots(const BandRef *bands, int which, double *part) {
  __shared__ double red[2][4];
  const BandRef B = bands[blockIdx.y];
  const long chunk = (B.n + BCH - 1) / BCH;
  const long i0 = blockIdx.x * chunk, i1 = min(B.n, i0 + chunk);
  double s0 = 0.0, s1 = 0.0;
  for (long i = i0 + threadIdx.x; i < i1; i += 256) {
    const double x = B.psi[i];
    if (which == 1) {
      const double q = B.p[i];
      s0 += x * q;
      s1 += q * q;
    } else {
      s0 += x * B.hp[i];
    }
  }
  for (int off = 32; off > 0; off >>= 1) {
    s0 += __shfl_down(s0, off, 64);
    s1 += __shfl_down(s1, off, 64);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    red[0][w] = s0;
    red[1][w] = s1;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double *o = part + ((long)blockIdx.y * BCH + blockIdx.x) * 2;
    o[0] = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
    o[1] = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
  }
}
__global__ void k_band_fold(const BandRef *bands, int nbt, const double *part, double *r0,
                            double *r1) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbt) return;
  double s0 = 0.0, s1 = 0.0;
  for (int c = 0; c < BCH; c++) {
    s0 += part[((long)b * BCH + c) * 2];
    s1 += part[((long)b * BCH + c) * 2 + 1];
  }
  r0[b] = bands[b].dv * s0;
  if (r1) r1[b] = bands[b].dv * s1;
}
// res[b] = dV * sum of the band's stencil/projector partials (<in|H in>)
__global__ void k_band_parts(const BandRef *bands, int nbt, double *res) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbt) return;
  const BandRef B = bands[b];
  double s = 0.0;
  for (int c = 0; c < B.nparts; c++) s += B.part[c];
  res[b] = B.dv * s;
}
// p <- (p - d psi) / sqrt(<p|p> - d^2)  (S = 1, psi normalised)
__global__ __launch_bounds__(256) void k_band_orth(const BandRef *bands, const double *d,
                                                   const double *pp) {
  const BandRef B = bands[blockIdx.y];
  const double db = d[blockIdx.y], n2 = pp[blockIdx.y] - db * db;
  const double f = n2 > 0.0 ? 1.0 / sqrt(n2) : 0.0;
  const long stride = (long)gridDim.x * 256;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < B.n; i += stride) B.p[i] = f * (B.p[i] - db * B.psi[i]);
}
// 2x2 Rayleigh-Ritz of (psi, p) (kscg8f.F90:1197-1230, S = 1):
//   gamma = (eps + pap)/2 - sqrt(((eps - pap)/2)^2 + sap^2); lower eigenvector (a, c), a >= 0
__global__ void k_band_rr(int nbt, const double *eps, const double *pap, const double *sap,
                          double *ab, double *sval) {
  const int b = blockIdx.x * blockDim.x + threadIdx.x;
  if (b >= nbt) return;
  const double e = eps[b], q = pap[b], s = sap[b];
  const double g = 0.5 * (e + q) - sqrt(0.25 * (e - q) * (e - q) + s * s);
  double a, c;
  if (fabs(e - g) >= fabs(q - g)) {
    a = -s;
    c = e - g;
  } else {
    a = q - g;
    c = -s;
  }
  double nn = sqrt(a * a + c * c);
  if (nn == 0.0) {
    a = 1.0;
    c = 0.0;
    nn = 1.0;
  }
  a /= nn;
  c /= nn;
  if (a < 0.0) {
    a = -a;
    c = -c;
  }
  ab[2 * b] = a;
  ab[2 * b + 1] = c;
  sval[b] = g;
}
// psi <- a psi + c p ; hpsi <- a hpsi + c hp
__global__ __launch_bounds__(256) void k_band_update(const BandRef *bands, const double *ab) {
  const BandRef B = bands[blockIdx.y];
  const double a = ab[2 * blockIdx.y], c = ab[2 * blockIdx.y + 1];
  const long stride = (long)gridDim.x * 256;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < B.n; i += stride) {
    B.psi[i] = a * B.psi[i] + c * B.p[i];
    B.hpsi[i] = a * B.hpsi[i] + c * B.hp[i];
  }
}

// ------------------------------------------------------------------ batched Hartree CG
// The iteration is that of hartree_cg.hip over all systems (two launches); here are its start and
// the tables.  state = {done, iteration, iterations taken}, sc = {<r|r> of odd / even iterations,
// mean b}.
struct HSys {
  double *rho, *vh, *r, *p, *ap, *sc;
  int *state;
  long n;
};
constexpr int HCH = 64;

__global__ __launch_bounds__(256) void k_hb_sum(const HSys *hs, int which, double *part) {
  __shared__ double red[4];
  const HSys H = hs[blockIdx.y];
  const long chunk = (H.n + HCH - 1) / HCH;
  const long i0 = blockIdx.x * chunk, i1 = min(H.n, i0 + chunk);
  double s = 0.0;
  for (long i = i0 + threadIdx.x; i < i1; i += 256) {
    if (which == 0) {
      const double bi = 2.0 * M_PI * H.rho[i];
      H.r[i] = bi;
      s += bi;
    } else {
      s += H.r[i] * H.r[i];
    }
  }
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[(long)blockIdx.y * HCH + blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}
// mean: sc[2] = mean of the sums; else <r|r> of the start, and the iteration's state
__global__ void k_hb_fold(const HSys *hs, int ns, const double *part, int mean) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ns) return;
  double s = 0.0;
  for (int c = 0; c < HCH; c++) s += part[(long)i * HCH + c];
  hs[i].sc[mean ? 2 : 1] = mean ? s / (double)hs[i].n : s;
  if (!mean) {
    hs[i].state[0] = 0;
    hs[i].state[1] = 1;
    hs[i].state[2] = 0;
  }
}
// r = b - mean - A v (A v in ap, b in r); p = r
__global__ __launch_bounds__(256) void k_hb_init(const HSys *hs) {
  const HSys H = hs[blockIdx.y];
  const double m = H.sc[2];
  const long stride = (long)gridDim.x * 256;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < H.n; i += stride) {
    const double ri = H.r[i] - m - H.ap[i];
    H.r[i] = ri;
    H.p[i] = ri;
  }
}

inline unsigned nb_(long n, int t) { return (unsigned)((n + t - 1) / t); }

}  // namespace

// ============================================================================= Batch
// ---------------------------------------------------------------- orthonormalisation
// One FP64 Cholesky-QR per system after the band update (S = 1): G = dV Psi^T Psi = R^T R,
// Psi <- Psi R^-1, the same Q as the reference's Gram-Schmidt (orthogonalization8f.F90:93-376)
// in exact arithmetic.  The work of all systems runs in one launch per kernel over unit
// tables (system-major), so loop mode launches the same kernels on one system's units.
// The products run on the FP64 matrix cores straight from global memory; the sizes (at most 128
// bands) let a wave hold what a general product would stage.  12 cells of 27^3 to 62^3 points, 16
// to 126 bands: Gram 2.44 -> 0.53 ms, factor and inverse 1.18 -> 0.16 ms, apply 2.14 -> 0.47 ms
// (vector FMAs from LDS tiles, and a column of the inverse per thread, before).
constexpr int OMAX = 128;  // bands per system (the Cholesky runs in 128 KB of LDS)
typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d4u __attribute__((ext_vector_type(4), aligned(8)));
struct OSys {
  double *psi;
  long n, kc;  // points; points per Gram unit
  int M, nt, nchunk;
  double dv;
  double *G, *Rinv, *part;  // M x M, M x M (and 16 zeros), [pair of 16-band tiles][chunk][256]
  int *flag;                // 1: a pivot was not positive
};
struct GUnit {  // Gram: points [item kc, ...) and which part of the pairs; reduction: pair of tiles
  int sys, item, part;
};
struct AUnit {
  int sys;
  long p0;  // first point of the 128-point tile
};

// One wave: the upper tile pairs i <= j, J0 <= j < NT, of X^T X over points [k0, k1), all of them
// in registers (NT = 6: 21 x 4 doubles per lane), so every value is loaded once, 32 bytes per lane,
// and one 16-point step of loads is in flight while the products of the last run.  More than six
// tiles do not fit 512 registers: their last one or two columns of pairs are a wave's work of
// their own.  A lane's operand is the same for both sides: band l % 16 of its tile, points
// 4 (l / 16) + s at step s.
template <int NT, int J0>
__device__ inline void gram_unit(const OSys &S, long k0, long k1, int chunk) {
  const int lane = threadIdx.x, q = lane >> 4, c16 = lane & 15;
  const double *col[NT];
#pragma unroll
  for (int f = 0; f < NT; f++)  // bands past the last repeat it (results unused)
    col[f] = S.psi + S.n * min(16 * f + c16, S.M - 1) + k0 + 4 * q;
  constexpr int PR0 = J0 * (J0 + 1) / 2, NP = NT * (NT + 1) / 2 - PR0;
  d4 acc[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) acc[i] = d4{0.0, 0.0, 0.0, 0.0};
  auto mac = [&](const d4u *x) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
      int pr = 0;
#pragma unroll
      for (int j = J0; j < NT; j++)
#pragma unroll
        for (int i = 0; i <= j; i++, pr++)
          acc[pr] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], x[j][s], acc[pr], 0, 0, 0);
    }
  };
  const long nf = (k1 - k0) / 16;
  d4u x[NT], xn[NT];
  if (nf > 0) {
#pragma unroll
    for (int f = 0; f < NT; f++) x[f] = *(const d4u *)col[f];
    for (long st = 1; st < nf; st++) {
#pragma unroll
      for (int f = 0; f < NT; f++) xn[f] = *(const d4u *)(col[f] + 16 * st);
      mac(x);
#pragma unroll
      for (int f = 0; f < NT; f++) x[f] = xn[f];
    }
    mac(x);
  }
  const int rem = (int)(k1 - k0 - 16 * nf);
  if (rem > 0) {  // the last, partial step: points past k1 are zero
#pragma unroll
    for (int f = 0; f < NT; f++)
#pragma unroll
      for (int s = 0; s < 4; s++) x[f][s] = 4 * q + s < rem ? col[f][16 * nf + s] : 0.0;
    mac(x);
  }
#pragma unroll
  for (int pr = 0; pr < NP; pr++) {
    double *o = S.part + ((long)(PR0 + pr) * S.nchunk + chunk) * 256 + lane;
#pragma unroll
    for (int r = 0; r < 4; r++) o[64 * r] = acc[pr][r];
  }
}
__global__ __launch_bounds__(64, 1) void k_bgram_part(const OSys *os, const GUnit *units) {
  const GUnit u = units[blockIdx.x];
  const OSys S = os[u.sys];
  const long k0 = u.item * S.kc, k1 = min(S.n, k0 + S.kc);
  switch (S.nt) {
    case 1: gram_unit<1, 0>(S, k0, k1, u.item); break;
    case 2: gram_unit<2, 0>(S, k0, k1, u.item); break;
    case 3: gram_unit<3, 0>(S, k0, k1, u.item); break;
    case 4: gram_unit<4, 0>(S, k0, k1, u.item); break;
    case 5: gram_unit<5, 0>(S, k0, k1, u.item); break;
    case 6: gram_unit<6, 0>(S, k0, k1, u.item); break;
    default:
      if (u.part == 0) gram_unit<6, 0>(S, k0, k1, u.item);
      else if (S.nt == 7) gram_unit<7, 6>(S, k0, k1, u.item);
      else gram_unit<8, 6>(S, k0, k1, u.item);
  }
}

// G tile pair = dV sum over chunks in order; register r of lane l is row l / 16 + 4 r, column l % 16
__global__ __launch_bounds__(256) void k_bgram_reduce(const OSys *os, const GUnit *units) {
  const GUnit u = units[blockIdx.x];
  const OSys S = os[u.sys];
  int tj = 0, ti = u.item;
  while (ti > tj) ti -= ++tj;
  const int t = threadIdx.x, lane = t & 63;
  const int gi = 16 * ti + (lane >> 4) + 4 * (t >> 6), gj = 16 * tj + (lane & 15);
  const double *p = S.part + (long)u.item * S.nchunk * 256 + t;
  double s = 0.0;
#pragma unroll 8
  for (int c = 0; c < S.nchunk; c++) s += p[256L * c];
  if (gi < S.M && gj < S.M) S.G[gi + (long)S.M * gj] = S.dv * s;
}

// R^-1 of G = R^T R per system in LDS, by eliminating [G | 1]: the upper triangle holds what is
// left of G, the strictly lower one the rows of R^-T found so far.  Step k divides row k of both
// by its pivot's root (w) and subtracts w_i w_j from every row i > k; its work does not shrink
// with k, and no thread waits on a chain longer than a step.
__global__ __launch_bounds__(1024) void k_bchol_inv(const OSys *os) {
  __shared__ double A[OMAX * OMAX], w[2][OMAX], dinv[OMAX];
  __shared__ int bad;
  const OSys S = os[blockIdx.x];
  const int M = S.M, t = threadIdx.x, tx = t & 31, ty = t >> 5;
  for (int j = ty; j < M; j += 32)
    for (int i = tx; i < M; i += 32) A[i + M * j] = i <= j ? S.G[i + (long)M * j] : 0.0;
  if (t == 0) bad = 0;
  __syncthreads();
  for (int k = 0; k < M; k++) {
    double *wk = w[k & 1];
    if (t < M) {
      const double d = A[k + M * k], f = 1.0 / (d > 0.0 ? sqrt(d) : 1.0);
      if (t == k) {
        if (!(d > 0.0)) bad = 1;
        wk[t] = dinv[t] = f;
      } else {
        const double v = A[k + M * t] * f;
        wk[t] = v;
        if (t < k) A[k + M * t] = v;  // row k of R^-T
      }
    }
    __syncthreads();
    for (int j = ty; j < M; j += 32) {
      const double wj = wk[j];
      const int i0 = k + 1, i1 = j <= k ? M : j + 1;  // rows of R^-T, or the rows of G above j
      for (int i = i0 + tx; i < i1; i += 32) A[i + M * j] -= wk[i] * wj;
    }
    __syncthreads();
  }
  for (int j = ty; j < M; j += 32)
    for (int i = tx; i < M; i += 32) S.Rinv[i + (long)M * j] = i < j ? A[j + M * i] : i == j ? dinv[i] : 0.0;
  if (t == 0) *S.flag = bad;
}

// Psi <- Psi R^-1, a wave per 32 points: it loads all its bands (8 NT doubles per lane), then
// forms the rows of R^-T Psi^T tile by tile, so the update is in place without LDS.  Psi is the
// right operand (and the result's columns): loads and stores are 16 consecutive points each, and
// R^-1 (at most 128 KB) comes from the caches.
template <int NT>
__device__ inline void apply_unit(const OSys &S, long p0) {
  const int lane = threadIdx.x & 63, q = lane >> 4, c16 = lane & 15;
  double x[2][NT][4];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const long pt = min(p0 + 16 * h + c16, S.n - 1);
#pragma unroll
    for (int f = 0; f < NT; f++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const int b = 16 * f + 4 * q + s;
        x[h][f][s] = b < S.M ? S.psi[S.n * b + pt] : 0.0;
      }
  }
#pragma unroll
  for (int j = 0; j < NT; j++) {
    const double *rc = S.Rinv + (long)S.M * min(16 * j + c16, S.M - 1) + 4 * q;
    d4 acc[2] = {d4{0.0, 0.0, 0.0, 0.0}, d4{0.0, 0.0, 0.0, 0.0}};
#pragma unroll
    for (int f = 0; f <= j; f++) {
      const d4u a = *(const d4u *)(rc + 16 * f);  // past the last band: zero bands in x
#pragma unroll
      for (int s = 0; s < 4; s++)
#pragma unroll
        for (int h = 0; h < 2; h++)
          acc[h] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s], x[h][f][s], acc[h], 0, 0, 0);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const long pt = p0 + 16 * h + c16;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int b = 16 * j + q + 4 * r;
        if (b < S.M && pt < S.n) S.psi[S.n * b + pt] = acc[h][r];
      }
    }
  }
}
__global__ __launch_bounds__(256) void k_bortho_apply(const OSys *os, const AUnit *units) {
  const AUnit u = units[blockIdx.x];
  const OSys S = os[u.sys];
  const long p0 = u.p0 + 32 * (threadIdx.x >> 6);
  if (p0 >= S.n) return;
  switch (S.nt) {
    case 1: apply_unit<1>(S, p0); break;
    case 2: apply_unit<2>(S, p0); break;
    case 3: apply_unit<3>(S, p0); break;
    case 4: apply_unit<4>(S, p0); break;
    case 5: apply_unit<5>(S, p0); break;
    case 6: apply_unit<6>(S, p0); break;
    case 7: apply_unit<7>(S, p0); break;
    default: apply_unit<8>(S, p0); break;
  }
}

struct BatchSystem {
  int n = 0, M = 0, natom = 0, num_list = 0, band0 = 0;
  double h = 0;
  Grid g;
  std::unique_ptr<Ctx> ctx;  // projector plan and dij
  double *veff = nullptr, *vnl = nullptr, *dij = nullptr, *psi = nullptr, *hpsi = nullptr,
         *p = nullptr, *hp = nullptr, *rp = nullptr, *coef = nullptr, *part = nullptr,
         *ones = nullptr;
  int *lst = nullptr;
  double *rho = nullptr, *vh = nullptr, *hr = nullptr, *hpv = nullptr, *hpw = nullptr, *hap = nullptr;
  long nparts = 0, sparts = 0;
  std::vector<void *> owned;
  template <class T>
  T *alloc(size_t count) {
    void *q = nullptr;
    HIPCK(hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)));
    owned.push_back(q);
    return (T *)q;
  }
  ~BatchSystem() {
    for (void *q : owned) (void)hipFree(q);
  }
};

struct Batch {
  std::vector<std::unique_ptr<BatchSystem>> sys;
  int nbt = 0;
  BandRef *bands = nullptr, *pbands = nullptr;  // <psi|H psi> partials / <p|H p> partials
  double *bpart = nullptr, *eps = nullptr, *d = nullptr, *pp = nullptr, *sap = nullptr,
         *pap = nullptr, *ab = nullptr, *sval = nullptr, *hpart = nullptr;
  HSys *hs = nullptr;
  double *hsc = nullptr;     // 3 per system
  int *hstate = nullptr;     // 3 per system
  std::vector<HcgArgs> hcg;  // the Hartree iteration's arguments, their device copy and units
  HcgArgs *hcg_dev = nullptr;
  bool hcg_sent = false;     // hcg_dev holds hcg
  int2 *hdir = nullptr, *hupd = nullptr;
  std::vector<int> hd0, hu0;  // each system's first unit (ns + 1)
  std::vector<void *> owned;
  bool ready = false;
  int P = 2, grid = 1024;
  // plans over all systems [0] and per system [1 + i]; kinds: H psi, H p, precond, A v
  std::vector<StencilBatchPlan> plan[4];
  hipGraphExec_t g_band = nullptr, g_hart = nullptr;
  int hart_blk = 16;
  // orthonormalisation: per-system descriptors and unit tables (system-major) with each
  // system's first unit, so loop mode launches one system's range
  bool ortho = true;
  OSys *osys = nullptr;
  GUnit *gunits = nullptr, *runits = nullptr;
  AUnit *aunits = nullptr;
  std::vector<int> g0, r0, a0;  // ns + 1 offsets each
  int *oflag = nullptr;
  ~Batch() {
    if (g_band) (void)hipGraphExecDestroy(g_band);
    if (g_hart) (void)hipGraphExecDestroy(g_hart);
    for (void *q : owned) (void)hipFree(q);
  }
  template <class T>
  T *alloc(size_t count) {
    void *q = nullptr;
    HIPCK(hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T)));
    owned.push_back(q);
    return (T *)q;
  }
};

namespace {

std::vector<Batch *> &batches() {
  static std::vector<Batch *> b;
  return b;
}
Batch *get_batch(void *h) {
  for (Batch *b : batches())
    if (b == h) return b;
  throw Error(1, "batch: unknown handle");
}

StencilCall call_for(BatchSystem &S, int kind, const double *eps_band) {
  StencilCall c;
  c.g = &S.g;
  c.ld_in = c.ld_out = S.g.n();
  c.nb = S.M;
  if (kind == 0 || kind == 1) {  // H psi / H p with <in|H in> partials
    c.in = kind == 0 ? S.psi : S.p;
    c.out = kind == 0 ? S.hpsi : S.hp;
    c.veff = S.veff;
    c.dot_partial = S.part;
    c.dot_ld = S.nparts;
  } else if (kind == 2) {  // K r with r = -(H psi - eps psi)
    c.in = S.hpsi; c.in2 = S.psi; c.eps = eps_band; c.sign = -1.0; c.out = S.p;
  } else {  // Hartree start: A v
    c.in = S.vh; c.out = S.hap; c.nb = 1; c.nfh_coeffs = 4;
  }
  return c;
}

void build_plans(Batch &B) {
  const int ns = (int)B.sys.size();
  for (int kind = 0; kind < 4; kind++) {
    B.plan[kind].clear();
    std::vector<StencilCall> all;
    for (int i = 0; i < ns; i++) all.push_back(call_for(*B.sys[i], kind, B.eps + B.sys[i]->band0));
    const bool res = kind == 2;
    const std::string tag = "batch" + std::to_string((long)(intptr_t)&B) + ".k" + std::to_string(kind);
    B.plan[kind].push_back(plan_stencil_batch(all, res, B.P, tag + ".all"));
    for (int i = 0; i < ns; i++)
      B.plan[kind].push_back(plan_stencil_batch({all[i]}, res, B.P, tag + ".s" + std::to_string(i)));
  }
}

// ---------------------------------------------------------------- one band step
// systems [s0, s1); batched: one launch per pass over the whole range
void band_step(Batch &B, int s0, int s1, bool batched, hipStream_t s) {
  const int b0 = B.sys[s0]->band0;
  const int b1 = s1 < (int)B.sys.size() ? B.sys[s1]->band0 : B.nbt;
  const int nb = b1 - b0;
  auto pass = [&](int kind) {
    if (batched) {
      launch_stencil_batch(B.plan[kind][0], B.grid, s);
    } else {
      for (int i = s0; i < s1; i++) launch_stencil_batch(B.plan[kind][1 + i], B.grid, s);
    }
  };
  auto nonlocal = [&](bool on_p) {
    for (int i = s0; i < s1; i++) {
      BatchSystem &S = *B.sys[i];
      Ctx &c = *S.ctx;
      const long n1 = (long)c.pl.nprjmx * c.pl.num_ppcell;
      c.proj(on_p ? S.p : S.psi, S.g.n(), S.M, S.rp, n1);
      launch_coef(c.pl, S.rp, n1, S.M, c.dij, false, 1, 1.0 / S.g.dv(), S.coef, n1, s, true);
    }
  };
  auto expand = [&](bool on_p) {
    for (int i = s0; i < s1; i++) {
      BatchSystem &S = *B.sys[i];
      launch_expand_rows(S.ctx->pl, S.coef, S.M, on_p ? S.hp : S.hpsi, S.g.n(), on_p ? S.p : S.psi,
                         S.g.n(), S.part, S.nparts, (int)S.sparts, s);
    }
  };
  const dim3 gb(BCH, nb), gu(16, nb);
  // eps = dV <psi|H psi>
  nonlocal(false);
  pass(0);
  expand(false);
  hipLaunchKernelGGL(k_band_parts, dim3(nb_(nb, 64)), dim3(64), 0, s, B.bands + b0, nb, B.eps + b0);
  // p = K r, orthogonal to psi and normalised
  pass(2);
  hipLaunchKernelGGL(k_band_dots, gb, dim3(256), 0, s, B.bands + b0, 1, B.bpart + (long)b0 * BCH * 2);
  hipLaunchKernelGGL(k_band_fold, dim3(nb_(nb, 64)), dim3(64), 0, s, B.bands + b0, nb,
                     B.bpart + (long)b0 * BCH * 2, B.d + b0, B.pp + b0);
  hipLaunchKernelGGL(k_band_orth, gu, dim3(256), 0, s, B.bands + b0, B.d + b0, B.pp + b0);
  // H p, pap = dV <p|H p>, sap = dV <psi|H p>
  nonlocal(true);
  pass(1);
  expand(true);
  hipLaunchKernelGGL(k_band_parts, dim3(nb_(nb, 64)), dim3(64), 0, s, B.bands + b0, nb, B.pap + b0);
  hipLaunchKernelGGL(k_band_dots, gb, dim3(256), 0, s, B.bands + b0, 2, B.bpart + (long)b0 * BCH * 2);
  hipLaunchKernelGGL(k_band_fold, dim3(nb_(nb, 64)), dim3(64), 0, s, B.bands + b0, nb,
                     B.bpart + (long)b0 * BCH * 2, B.sap + b0, nullptr);
  // 2x2 Rayleigh-Ritz and the band update
  hipLaunchKernelGGL(k_band_rr, dim3(nb_(nb, 64)), dim3(64), 0, s, nb, B.eps + b0, B.pap + b0,
                     B.sap + b0, B.ab + 2L * b0, B.sval + b0);
  hipLaunchKernelGGL(k_band_update, gu, dim3(256), 0, s, B.bands + b0, B.ab + 2L * b0);
  // Cholesky-QR of each system's bands
  if (B.ortho) {
    const int ng = B.g0[s1] - B.g0[s0], nr = B.r0[s1] - B.r0[s0], na = B.a0[s1] - B.a0[s0];
    if (ng > 0) hipLaunchKernelGGL(k_bgram_part, dim3(ng), dim3(64), 0, s, B.osys, B.gunits + B.g0[s0]);
    if (nr > 0) hipLaunchKernelGGL(k_bgram_reduce, dim3(nr), dim3(256), 0, s, B.osys, B.runits + B.r0[s0]);
    hipLaunchKernelGGL(k_bchol_inv, dim3(s1 - s0), dim3(1024), 0, s, B.osys + s0);
    if (na > 0) hipLaunchKernelGGL(k_bortho_apply, dim3(na), dim3(256), 0, s, B.osys, B.aunits + B.a0[s0]);
  }
  HIPCK(hipGetLastError());
}

// ---------------------------------------------------------------- Hartree
void hartree_start(Batch &B, int s0, int s1, bool batched, hipStream_t s) {
  const int ns = s1 - s0;
  for (int i = s0; i < s1; i++) {
    BatchSystem &S = *B.sys[i];
    charge(S.g.n(), S.M, S.psi, S.ones, S.rho, false);
  }
  HSys *hs = B.hs + s0;
  double *part = B.hpart + (long)s0 * HCH;
  hipLaunchKernelGGL(k_hb_sum, dim3(HCH, ns), dim3(256), 0, s, hs, 0, part);
  hipLaunchKernelGGL(k_hb_fold, dim3(nb_(ns, 64)), dim3(64), 0, s, hs, ns, part, 1);
  if (batched) {
    launch_stencil_batch(B.plan[3][0], B.grid, s);
  } else {
    for (int i = s0; i < s1; i++) launch_stencil_batch(B.plan[3][1 + i], B.grid, s);
  }
  hipLaunchKernelGGL(k_hb_init, dim3(16, ns), dim3(256), 0, s, hs);
  hipLaunchKernelGGL(k_hb_sum, dim3(HCH, ns), dim3(256), 0, s, hs, 1, part);
  hipLaunchKernelGGL(k_hb_fold, dim3(nb_(ns, 64)), dim3(64), 0, s, hs, ns, part, 0);
  HIPCK(hipGetLastError());
}

// one iteration of systems [s0, s1), it = 0, 1, ...
void hartree_iter(Batch &B, int s0, int s1, int it, hipStream_t s) {
  hcg_iteration_batch(B.hcg_dev, B.hdir + B.hd0[s0], B.hd0[s1] - B.hd0[s0], B.hupd + B.hu0[s0], B.hu0[s1] - B.hu0[s0],
                      B.hcg[0].tx, B.hcg[0].tz, it & 1, s);
}

void hartree_solve(Batch &B, int s0, int s1, bool batched, int ncgmax, hipStream_t s) {
  hartree_start(B, s0, s1, batched, s);
  const int blk = B.hart_blk;  // even: a block starts with the same direction buffer
  std::vector<int> st(3 * (s1 - s0));
  // a solve that ends after ncgmax iterations is marked by the launch that follows them
  for (int done = 0, it = 0; !done && it <= ncgmax; it += blk) {
    if (batched) {
      HIPCK(hipGraphLaunch(B.g_hart, s));
    } else {
      for (int k = 0; k < blk; k++) hartree_iter(B, s0, s1, k, s);
    }
    HIPCK(hipMemcpyAsync(st.data(), B.hstate + 3 * s0, sizeof(int) * st.size(), hipMemcpyDeviceToHost, s));
    HIPCK(hipStreamSynchronize(s));
    done = 1;
    for (size_t i = 0; i < st.size(); i += 3) done = done && st[i];
  }
}

// The iteration's rule of this step into the device table
void hartree_rule(Batch &B, int ncgmax, double eps) {
  if (B.hcg_sent && B.hcg[0].ncgmax == ncgmax && B.hcg[0].eps == eps) return;
  B.hcg_sent = false;
  for (HcgArgs &a : B.hcg) {
    a.ncgmax = ncgmax;
    a.eps = eps;
  }
  HIPCK(hipMemcpy(B.hcg_dev, B.hcg.data(), sizeof(HcgArgs) * B.hcg.size(), hipMemcpyHostToDevice));
  B.hcg_sent = true;
}

template <class F>
hipGraphExec_t capture(hipStream_t s, F &&f) {
  hipGraph_t graph;
  lib().capturing = true;
  try {
    HIPCK(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
    f();
    HIPCK(hipStreamEndCapture(s, &graph));
  } catch (...) {
    lib().capturing = false;
    hipGraph_t g2;
    (void)hipStreamEndCapture(s, &g2);
    throw;
  }
  lib().capturing = false;
  hipGraphExec_t exec;
  HIPCK(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
  HIPCK(hipGraphDestroy(graph));
  return exec;
}

// Tile shape and persistent grid: time the batched H psi pass for each candidate.
void autotune(Batch &B, hipStream_t s) {
  const int Ps[3] = {1, 2, 4};
  const int grids[4] = {512, 1024, 2048, 4096};
  float best = 1e30f;
  int bp = 2, bg = 1024;
  hipEvent_t e0, e1;
  HIPCK(hipEventCreate(&e0));
  HIPCK(hipEventCreate(&e1));
  for (int P : Ps) {
    bool fits = true;
    for (auto &sp : B.sys) fits = fits && (long)sp->g.nx * std::max(1, std::min(sp->g.ny, 512 * P / sp->g.nx)) <= 512L * P;
    if (!fits) continue;
    B.P = P;
    std::vector<StencilCall> all;
    for (auto &sp : B.sys) all.push_back(call_for(*sp, 0, nullptr));
    StencilBatchPlan plan = plan_stencil_batch(all, false, P, "batch.tune");
    for (int G : grids) {
      launch_stencil_batch(plan, G, s);  // warm
      HIPCK(hipEventRecord(e0, s));
      for (int r = 0; r < 3; r++) launch_stencil_batch(plan, G, s);
      HIPCK(hipEventRecord(e1, s));
      HIPCK(hipEventSynchronize(e1));
      float ms = 0.f;
      HIPCK(hipEventElapsedTime(&ms, e0, e1));
      if (ms < best) {
        best = ms;
        bp = P;
        bg = G;
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  B.P = bp;
  B.grid = bg;
  lib().params["batch_tile_p"] = bp;
  lib().params["batch_grid"] = bg;
  lib().params["batch_tune_ms"] = best / 3.0;
}

void prepare(Batch &B) {
  if (B.ready) return;
  hipStream_t s = lib().stream;
  const int ns = (int)B.sys.size();
  if (ns == 0) throw Error(1, "batch: no systems");
  B.nbt = 0;
  for (auto &sp : B.sys) {
    sp->band0 = B.nbt;
    B.nbt += sp->M;
  }
  const int nbt = B.nbt;
  B.bands = B.alloc<BandRef>(nbt);
  B.bpart = B.alloc<double>((size_t)nbt * BCH * 2);
  B.eps = B.alloc<double>(nbt);
  B.d = B.alloc<double>(nbt);
  B.pp = B.alloc<double>(nbt);
  B.sap = B.alloc<double>(nbt);
  B.pap = B.alloc<double>(nbt);
  B.ab = B.alloc<double>(2L * nbt);
  B.sval = B.alloc<double>(nbt);
  B.hs = B.alloc<HSys>(ns);
  B.hpart = B.alloc<double>((size_t)ns * HCH);
  B.hsc = B.alloc<double>(3L * ns);
  B.hstate = B.alloc<int>(3L * ns);
  std::vector<int> st0(3L * ns, 0);
  HIPCK(hipMemcpy(B.hstate, st0.data(), sizeof(int) * st0.size(), hipMemcpyHostToDevice));
  autotune(B, s);
  B.hcg.clear();  // a preparation that failed part-way is repeated by the next step
  B.hcg_sent = false;
  std::vector<BandRef> br(nbt);
  std::vector<HSys> hs(ns);
  for (int i = 0; i < ns; i++) {
    BatchSystem &S = *B.sys[i];
    const long n = S.g.n();
    S.sparts = stencil_batch_parts(S.g, 4, S.M, B.P);
    S.nparts = S.sparts + expand_nparts(S.ctx->pl);
    S.part = S.alloc<double>((size_t)S.nparts * S.M);
    for (int l = 0; l < S.M; l++) {
      BandRef &r = br[S.band0 + l];
      r.psi = S.psi + n * l; r.hpsi = S.hpsi + n * l; r.p = S.p + n * l; r.hp = S.hp + n * l;
      r.part = S.part + (long)S.nparts * l; r.n = n; r.nparts = (int)S.nparts; r.dv = S.g.dv();
    }
    HSys &H = hs[i];
    H.rho = S.rho; H.vh = S.vh; H.r = S.hr; H.p = S.hpv; H.ap = S.hap; H.sc = B.hsc + 3 * i;
    H.state = B.hstate + 3 * i; H.n = n;
    HcgArgs a{};
    a.nx = S.g.nx; a.ny = S.g.ny; a.nz = S.g.nz; a.px = a.py = a.pz = 1;
    double w[9];
    fd_coefficients(4, w);
    for (int m = 0; m < 9; m++) {
      a.cx[m] = w[m] / S.g.dx / S.g.dx * (-0.5);
      a.cy[m] = w[m] / S.g.dy / S.g.dy * (-0.5);
      a.cz[m] = w[m] / S.g.dz / S.g.dz * (-0.5);
    }
    a.c0 = a.cx[0] + a.cy[0] + a.cz[0];
    a.n = n; a.vh = S.vh; a.r = S.hr; a.p[0] = S.hpv; a.p[1] = S.hpw; a.ap = S.hap; a.rr = H.sc; a.state = H.state;
    a.ncgres = 801;  // restart period of parameters.inp
    a.ncgmin = 1;
    a.dvo = 1.0 / (double)n;  // dV / Omega of the periodic cell
    B.hcg.push_back(a);
  }
  // the Hartree iteration's tiles, partial sums and units
  hcg_plan_batch(B.hcg.data(), ns);
  B.hd0.assign(1, 0);
  B.hu0.assign(1, 0);
  std::vector<int2> ud, uu;
  for (int i = 0; i < ns; i++) {
    HcgArgs &a = B.hcg[i];
    a.part_p = B.alloc<double>(a.np);
    a.part_r = B.alloc<double>(a.nr);
    for (int k = 0; k < a.np; k++) ud.push_back(make_int2(i, k));
    for (int k = 0; k < a.nr; k++) uu.push_back(make_int2(i, k));
    B.hd0.push_back((int)ud.size());
    B.hu0.push_back((int)uu.size());
  }
  B.hcg_dev = B.alloc<HcgArgs>(ns);
  B.hdir = B.alloc<int2>(ud.size());
  B.hupd = B.alloc<int2>(uu.size());
  HIPCK(hipMemcpy(B.hdir, ud.data(), sizeof(int2) * ud.size(), hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(B.hupd, uu.data(), sizeof(int2) * uu.size(), hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(B.bands, br.data(), sizeof(BandRef) * nbt, hipMemcpyHostToDevice));
  HIPCK(hipMemcpy(B.hs, hs.data(), sizeof(HSys) * ns, hipMemcpyHostToDevice));
  // orthonormalisation tables (param "batch_ortho", default 1, read once here)
  B.ortho = param("batch_ortho", 1.0) >= 1.0;
  if (B.ortho) {
    std::vector<OSys> os(ns);
    std::vector<GUnit> gu, ru;
    std::vector<AUnit> au;
    B.oflag = B.alloc<int>(ns);
    long points = 0;
    for (auto &sp : B.sys) points += sp->g.n();
    // points per Gram wave: about one wave per SIMD of the chip, and no shorter than the
    // partial sums it leaves are worth
    const long kc = std::min(8192L, std::max(512L, points / 1024 / 16 * 16));
    B.g0.assign(1, 0);
    B.r0.assign(1, 0);
    B.a0.assign(1, 0);
    for (int i = 0; i < ns; i++) {
      BatchSystem &S = *B.sys[i];
      if (S.M > OMAX) throw Error(1, "batch: at most 128 bands per system");
      OSys &o = os[i];
      o.psi = S.psi;
      o.n = S.g.n();
      o.M = S.M;
      o.nt = (S.M + 15) / 16;
      o.kc = kc;
      o.nchunk = (int)((o.n + kc - 1) / kc);
      const int ntp = o.nt * (o.nt + 1) / 2;
      o.dv = S.g.dv();
      o.G = S.alloc<double>((size_t)S.M * S.M);
      o.Rinv = S.alloc<double>((size_t)S.M * S.M + 16);
      launch_fill(16, 0.0, o.Rinv + (size_t)S.M * S.M, s);
      o.part = S.alloc<double>((size_t)ntp * o.nchunk * 256);
      o.flag = B.oflag + i;
      for (int c = 0; c < o.nchunk; c++)
        for (int part = 0; part < (o.nt > 6 ? 2 : 1); part++) gu.push_back({i, c, part});
      for (int tp = 0; tp < ntp; tp++) ru.push_back({i, tp, 0});
      for (long p0 = 0; p0 < o.n; p0 += 128) au.push_back({i, p0});
      B.g0.push_back((int)gu.size());
      B.r0.push_back((int)ru.size());
      B.a0.push_back((int)au.size());
    }
    B.osys = B.alloc<OSys>(ns);
    B.gunits = B.alloc<GUnit>(gu.size());
    B.runits = B.alloc<GUnit>(ru.size());
    B.aunits = B.alloc<AUnit>(au.size());
    HIPCK(hipMemcpy(B.osys, os.data(), sizeof(OSys) * ns, hipMemcpyHostToDevice));
    HIPCK(hipMemcpy(B.gunits, gu.data(), sizeof(GUnit) * gu.size(), hipMemcpyHostToDevice));
    HIPCK(hipMemcpy(B.runits, ru.data(), sizeof(GUnit) * ru.size(), hipMemcpyHostToDevice));
    HIPCK(hipMemcpy(B.aunits, au.data(), sizeof(AUnit) * au.size(), hipMemcpyHostToDevice));
  }
  build_plans(B);
  B.ready = true;
}

}  // namespace

// ============================================================================= C-ABI helpers
void *batch_create() {
  Batch *b = new Batch();
  batches().push_back(b);
  return b;
}

void batch_destroy(void *h) {
  Batch *b = get_batch(h);
  batches().erase(std::find(batches().begin(), batches().end(), b));
  sync();
  delete b;
}

int batch_add(void *h, int n, double hh, int nbands, int natom, int num_list, const int *lstvec2,
              const int *natinf, const double *vnlocp, const double *dij, const double *veff,
              const double *psi) {
  Batch *B = get_batch(h);
  if (B->ready) throw Error(1, "batch: systems can only be added before the first step");
  if (n < 8 || n > 256) throw Error(1, "batch: grid edge must be in 8..256");
  if (nbands < 1 || natom < 1 || num_list < 1) throw Error(1, "batch: empty system");
  hipStream_t s = lib().stream;
  auto S = std::make_unique<BatchSystem>();
  S->n = n; S->h = hh; S->M = nbands; S->natom = natom; S->num_list = num_list;
  S->g = Grid{n, n, n, 4, 3, hh, hh, hh};
  const long N = S->g.n();
  S->veff = S->alloc<double>(N);
  S->vnl = S->alloc<double>((size_t)num_list * 9 * natom);
  S->dij = S->alloc<double>((size_t)81 * natom);
  S->lst = S->alloc<int>((size_t)num_list * natom);
  S->psi = S->alloc<double>((size_t)N * nbands);
  S->hpsi = S->alloc<double>((size_t)N * nbands);
  S->p = S->alloc<double>((size_t)N * nbands);
  S->hp = S->alloc<double>((size_t)N * nbands);
  S->rp = S->alloc<double>((size_t)9 * natom * nbands);
  S->coef = S->alloc<double>((size_t)9 * natom * nbands);
  S->ones = S->alloc<double>(nbands);
  S->rho = S->alloc<double>(N);
  S->vh = S->alloc<double>(N);
  S->hr = S->alloc<double>(N);
  S->hpv = S->alloc<double>(N);
  S->hpw = S->alloc<double>(N);
  S->hap = S->alloc<double>(N);
  auto up = [&](void *dst, const void *src, size_t bytes) {
    Arr a(src, bytes, Arr::In);
    HIPCK(hipMemcpyAsync(dst, a.v(), bytes, hipMemcpyDeviceToDevice, s));
    HIPCK(hipStreamSynchronize(s));
  };
  up(S->veff, veff, sizeof(double) * N);
  up(S->vnl, vnlocp, sizeof(double) * num_list * 9 * natom);
  up(S->dij, dij, sizeof(double) * 81 * natom);
  up(S->lst, lstvec2, sizeof(int) * num_list * natom);
  up(S->psi, psi, sizeof(double) * N * nbands);
  launch_fill(nbands, 1.0, S->ones, s);
  launch_fill(N, 0.0, S->vh, s);
  // projector plan: one species, 9 projectors, every atom on this rank
  std::vector<int> nprj(1, 9), indspe(natom, 1), natpri(natom, 2), naps(natom);  // natpri: "in"
  std::vector<int> nat = host_ints(natinf, natom);
  for (int a = 0; a < natom; a++) naps[a] = a + 1;
  S->ctx = std::make_unique<Ctx>(S->g);
  build_plan(S->ctx->pl, S->g, natom, 9, 1, natom, num_list, 1, 2, 1, nprj.data(), indspe.data(),
             nat.data(), natpri.data(), naps.data(), S->vnl, S->lst,
             "batch" + std::to_string((long)(intptr_t)B) + ".p" + std::to_string(B->sys.size()));
  S->ctx->dij = S->dij;
  S->ctx->q_zero = true;
  B->sys.push_back(std::move(S));
  sync();
  return (int)B->sys.size() - 1;
}

void batch_step(void *h, int batched, int ncgmax, double epsvh) {
  Batch *B = get_batch(h);
  prepare(*B);
  hipStream_t s = lib().stream;
  const int ns = (int)B->sys.size();
  hartree_rule(*B, ncgmax, epsvh);
  if (batched) {
    Timed t("batch_step", 0.0);
    if (!B->g_band) B->g_band = capture(s, [&] { band_step(*B, 0, ns, true, s); });
    HIPCK(hipGraphLaunch(B->g_band, s));
    if (!B->g_hart)
      B->g_hart = capture(s, [&] {
        for (int k = 0; k < B->hart_blk; k++) hartree_iter(*B, 0, ns, k, s);
      });
    hartree_solve(*B, 0, ns, true, ncgmax, s);
  } else {
    Timed t("batch_loop", 0.0);
    for (int i = 0; i < ns; i++) {
      band_step(*B, i, i + 1, false, s);
      hartree_solve(*B, i, i + 1, false, ncgmax, s);
    }
  }
  sync();
  if (B->ortho) {
    std::vector<int> f(ns);
    HIPCK(hipMemcpy(f.data(), B->oflag, sizeof(int) * ns, hipMemcpyDeviceToHost));
    for (int i = 0; i < ns; i++)
      if (f[i]) throw Error(2, "batch: orthonormalisation of system " + std::to_string(i) + ": wf has negative norm");
  }
}

void batch_get(void *h, int i, double *psi, double *sval, double *vh, int *iters) {
  Batch *B = get_batch(h);
  if (i < 0 || i >= (int)B->sys.size()) throw Error(1, "batch: system index out of range");
  prepare(*B);
  BatchSystem &S = *B->sys[i];
  const long N = S.g.n();
  hipStream_t s = lib().stream;
  if (psi) {
    Arr a(psi, sizeof(double) * N * S.M, Arr::Out);
    HIPCK(hipMemcpyAsync(a.v(), S.psi, sizeof(double) * N * S.M, hipMemcpyDeviceToDevice, s));
    a.finish();
  }
  if (sval) {
    Arr a(sval, sizeof(double) * S.M, Arr::Out);
    HIPCK(hipMemcpyAsync(a.v(), B->sval + S.band0, sizeof(double) * S.M, hipMemcpyDeviceToDevice, s));
    a.finish();
  }
  if (vh) {
    Arr a(vh, sizeof(double) * N, Arr::Out);
    HIPCK(hipMemcpyAsync(a.v(), S.vh, sizeof(double) * N, hipMemcpyDeviceToDevice, s));
    a.finish();
  }
  if (iters) {
    int st[3];
    HIPCK(hipMemcpyAsync(st, B->hstate + 3 * i, sizeof(st), hipMemcpyDeviceToHost, s));
    sync();
    *iters = st[2];
  }
}

}  // namespace kukan
