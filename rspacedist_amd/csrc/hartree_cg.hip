// hartree_cg.hip — the Hartree CG iteration (scf_hartree8f.F90:611-1143) as two launches:
//   direction: beta and the stopping rule from <r|r>, p = r + beta p, A p and <p|A p>;
//   update:    alpha from <p|A p>, V += alpha p, r -= alpha A p and <r|r>.
// Ten passes over a grid vector per iteration (direction: r and p read, p and A p written;
// update: V, p, r, A p read, V and r written) against thirteen for the stencil, update, direction
// and control launches this replaces, and half the launches.  The residual follows
// r -= alpha A p, which in exact arithmetic is the reference's b - avhs with avhs += alpha A p;
// neither recomputes A V, so both drift from b - A V by the same rounding of the alpha A p.
// One iteration, four launches before and now (periodic, nfh 4):
//   40^3: 30 -> 11 us, 64^3: 34 -> 16, 96^3: 43 -> 24, 128^3: 55 -> 38, 256^3: 328 now.
// Small grids are bound by the launches and the two folds of partial sums, 128^3 by the passes
// (the update moves 100 MB in 16 us) and the tile halos.  Updating V one launch late, where its p
// is read anyway (nine passes), was no faster: 39 us at 128^3, 17 at 64^3.
// Twelve cells of 27^3 to 62^3 points in lock step (1.35 M points): 100 us with the stencil over a
// list of plane tiles, an update, a direction and four small control launches, 30 us here.
#include "hartree_cg.hpp"

#include <algorithm>

namespace kukan {
namespace {

// Sum of np partials by a 256-thread work-group in a fixed order (strided per thread, then
// wave shuffles, then the 4 wave sums in order); every thread gets the result.
__device__ inline double fold256(const double *part, int np, double *red4) {
  double s = 0.0;
  for (int c = threadIdx.x; c < np; c += 256) s += part[c];
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = s;
  __syncthreads();
  const double tot = ((red4[0] + red4[1]) + red4[2]) + red4[3];
  __syncthreads();
  return tot;
}
__device__ inline double sum256(double s, double *red4) {  // valid in thread 0
  for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
  if ((threadIdx.x & 63) == 0) red4[threadIdx.x >> 6] = s;
  __syncthreads();
  return ((red4[0] + red4[1]) + red4[2]) + red4[3];
}

// Work-group blk of nblk of one solve: p = r + beta p, A p and the <p|A p> partials (zero from a
// work-group without a tile).  A work-group owns a tile of TX x (256 / TX) columns and TZ planes; each thread loads its column's TZ + 2 NF values of r and p into
// registers and the work-group loads the tile's x and y halos, all in one batch of independent
// loads that is in flight while <r|r> is folded; the new p then goes through LDS for the x and y
// neighbours, with one barrier, and the z neighbours are in registers.  The tile has no serial
// march, so a small grid's iteration is one memory latency long, and the tile's halos (2 x its
// own points at 32 x 8 x 8) come from L2.
template <int NF, int TX, int TZ>
__device__ inline void hcg_direction(const HcgArgs &a, int par, int blk, int nblk) {
  constexpr int TY = 256 / TX, W = TX + 2 * NF, WY = TY + 2 * NF, NZ = TZ + 2 * NF;
  constexpr int NXH = (2 * NF * TY * TZ + 255) / 256, NYH = (2 * NF * TX * TZ + 255) / 256;
  __shared__ double box[TZ][WY][W];
  __shared__ double red[4];
  if (a.state[0]) return;  // uniform: the solve has finished
  const int t = threadIdx.x, lx = t % TX, ly = t / TX;
  const int k = a.state[1];
  // (not a.p[par]: an indexed member would put a copied argument struct into scratch memory)
  const double *pold = par ? a.p[1] : a.p[0];
  double *pnew = par ? a.p[0] : a.p[1];
  const long plane = (long)a.nx * a.ny;
  const int ntile = a.ntx * a.nty * a.ntz;
  double beta = 0.0, dsum = 0.0;
  bool folded = false;
  // each XCD takes a contiguous eighth of the tiles, so most halos are read by the XCD whose L2
  // holds them already (work-group g runs on XCD g mod 8; nblk is a multiple of 8, and so is the grid index
  // of the solve's first work-group)
  const int per = (ntile + 7) / 8, xcd = blk & 7, t1 = min(ntile, (xcd + 1) * per);
  for (int tile = xcd * per + (blk >> 3); tile < t1; tile += nblk >> 3) {
    const int x0 = tile % a.ntx * TX, y0 = tile / a.ntx % a.nty * TY, z0 = tile / (a.ntx * a.nty) * TZ;
    const int ex = min(TX, a.nx - x0), ey = min(TY, a.ny - y0), ez = min(TZ, a.nz - z0);
    const int x = x0 + lx, y = y0 + ly;
    const bool act = lx < ex && ly < ey;
    const long col = act ? x + (long)a.nx * y : 0;
    double rv[NZ], pv[NZ];
#pragma unroll
    for (int j = 0; j < NZ; j++) {
      int z = z0 + j - NF;
      bool ok = act && z < z0 + ez + NF;
      if (z < 0 || z >= a.nz) {
        ok = ok && a.pz;
        z = z < 0 ? z + a.nz : z - a.nz;
      }
      rv[j] = ok ? a.r[col + plane * z] : 0.0;
      pv[j] = ok ? pold[col + plane * z] : 0.0;
    }
    // x halo: NF values on either side of each row; y halo: NF rows above and below
    double rx[NXH], qx[NXH], ry[NYH], qy[NYH];
    int ix[NXH], iy[NYH];
#pragma unroll
    for (int h = 0; h < NXH; h++) {
      const int i = t + 256 * h, c = i % (2 * NF), row = i / (2 * NF) % TY, pl = i / (2 * NF * TY);
      const int cx = c < NF ? c - NF : ex + c - NF;
      bool ok = pl < ez && row < ey;
      ix[h] = ok ? (pl * WY + row + NF) * W + cx + NF : -1;
      int X = x0 + cx;
      if (X < 0 || X >= a.nx) {
        ok = ok && a.px;
        X = X < 0 ? X + a.nx : X - a.nx;
      }
      const long o = X + (long)a.nx * (y0 + row) + plane * (z0 + pl);
      rx[h] = ok ? a.r[o] : 0.0;
      qx[h] = ok ? pold[o] : 0.0;
    }
#pragma unroll
    for (int h = 0; h < NYH; h++) {
      const int i = t + 256 * h, c = i % TX, row = i / TX % (2 * NF), pl = i / (TX * 2 * NF);
      const int cy = row < NF ? row - NF : ey + row - NF;
      bool ok = pl < ez && c < ex;
      iy[h] = ok ? (pl * WY + cy + NF) * W + c + NF : -1;
      int Y = y0 + cy;
      if (Y < 0 || Y >= a.ny) {
        ok = ok && a.py;
        Y = Y < 0 ? Y + a.ny : Y - a.ny;
      }
      const long o = x0 + c + (long)a.nx * Y + plane * (z0 + pl);
      ry[h] = ok ? a.r[o] : 0.0;
      qy[h] = ok ? pold[o] : 0.0;
    }
    if (!folded) {
      folded = true;
      if (k > 1) {
        // every work-group folds the same partials in the same order, so all of them take the
        // same beta and the same decision (the reference's rule, after iteration k - 1)
        const double r2r = fold256(a.part_r, a.nr, red);
        const int last = k - 1;
        if (last >= a.ncgmin && (last >= a.ncgmax || sqrt(r2r * a.dvo) <= a.eps)) {
          if (blk == 0 && t == 0) {
            a.state[2] = last;
            a.state[0] = 1;
          }
          return;
        }
        beta = last % a.ncgres == 0 ? 0.0 : r2r / a.rr[last & 1];
        if (blk == 0 && t == 0) a.rr[k & 1] = r2r;
      }
    } else {
      __syncthreads();  // the previous tile's values have been read
    }
#pragma unroll
    for (int j = 0; j < NZ; j++) rv[j] = rv[j] + beta * pv[j];
    // (a partial tile's halo columns and rows lie where its idle threads' points would)
    if (act) {
#pragma unroll
      for (int j = 0; j < TZ; j++) box[j][ly + NF][lx + NF] = rv[j + NF];
    }
    double *flat = &box[0][0][0];
#pragma unroll
    for (int h = 0; h < NXH; h++)
      if (ix[h] >= 0) flat[ix[h]] = rx[h] + beta * qx[h];
#pragma unroll
    for (int h = 0; h < NYH; h++)
      if (iy[h] >= 0) flat[iy[h]] = ry[h] + beta * qy[h];
    __syncthreads();
    if (act) {
#pragma unroll
      for (int j = 0; j < TZ; j++) {
        if (j >= ez) break;
        const double *c = &box[j][ly + NF][lx + NF];
        const double p = rv[j + NF];
        double s = a.c0 * p;
#pragma unroll
        for (int m = 1; m <= NF; m++) s += a.cx[m] * (c[-m] + c[m]);
#pragma unroll
        for (int m = 1; m <= NF; m++) s += a.cy[m] * (c[-m * W] + c[m * W]);
#pragma unroll
        for (int m = 1; m <= NF; m++) s += a.cz[m] * (rv[j + NF - m] + rv[j + NF + m]);
        const long o = col + plane * (z0 + j);
        pnew[o] = p;
        a.ap[o] = s;
        dsum += p * s;
      }
    }
  }
  const double tot = sum256(dsum, red);
  if (t == 0) a.part_p[blk] = tot;
}
template <int NF, int TX, int TZ>
__global__ __launch_bounds__(256) void k_hcg_direction(HcgArgs a, int par) {
  hcg_direction<NF, TX, TZ>(a, par, blockIdx.x, gridDim.x);
}
// several solves in one launch: unit[g] = {solve, work-group of the solve}
template <int NF, int TX, int TZ>
__global__ __launch_bounds__(256) void k_hcg_direction_batch(const HcgArgs *tab, const int2 *unit, int par) {
  const int2 u = unit[blockIdx.x];
  const HcgArgs a = tab[u.x];
  hcg_direction<NF, TX, TZ>(a, par, u.y, a.np);
}

// V += alpha p, r -= alpha A p and the <r|r> partials; the first batch of loads is in flight
// while <p|A p> is folded
__device__ inline void hcg_update(const HcgArgs &a, int par, int blk) {
  constexpr int P = 8;
  __shared__ double red[4];
  if (a.state[0]) return;
  const double *p = par ? a.p[0] : a.p[1];
  const long i0 = blk * a.chunk + threadIdx.x, i1 = min(a.n, (blk + 1) * a.chunk);
  double v[P], q[P], r[P], w[P];
  auto load = [&](long i) {
#pragma unroll
    for (int j = 0; j < P; j++) {
      const bool ok = i + 256 * j < i1;
      v[j] = ok ? a.vh[i + 256 * j] : 0.0;
      q[j] = ok ? p[i + 256 * j] : 0.0;
      r[j] = ok ? a.r[i + 256 * j] : 0.0;
      w[j] = ok ? a.ap[i + 256 * j] : 0.0;
    }
  };
  load(i0);
  const double alpha = a.rr[1 - par] / fold256(a.part_p, a.np, red);
  double s = 0.0;
  for (long i = i0; i < i1; i += 256 * P) {
    if (i > i0) load(i);
#pragma unroll
    for (int j = 0; j < P; j++) {
      if (i + 256 * j >= i1) break;
      a.vh[i + 256 * j] = v[j] + alpha * q[j];
      const double ri = r[j] - alpha * w[j];
      a.r[i + 256 * j] = ri;
      s += ri * ri;
    }
  }
  s = sum256(s, red);
  if (threadIdx.x == 0) {
    a.part_r[blk] = s;
    if (blk == 0) a.state[1] += 1;
  }
}
__global__ __launch_bounds__(256) void k_hcg_update(HcgArgs a, int par) { hcg_update(a, par, blockIdx.x); }
__global__ __launch_bounds__(256) void k_hcg_update_batch(const HcgArgs *tab, const int2 *unit, int par) {
  const int2 u = unit[blockIdx.x];
  const HcgArgs a = tab[u.x];
  hcg_update(a, par, u.y);
}

template <int NF>
void direction(const HcgArgs &a, int par, hipStream_t s) {
  const dim3 g(a.np), b(256);
  if (a.tx == 32) {
    if (a.tz == 8) hipLaunchKernelGGL((k_hcg_direction<NF, 32, 8>), g, b, 0, s, a, par);
    else if (a.tz == 4) hipLaunchKernelGGL((k_hcg_direction<NF, 32, 4>), g, b, 0, s, a, par);
    else hipLaunchKernelGGL((k_hcg_direction<NF, 32, 2>), g, b, 0, s, a, par);
  } else {
    if (a.tz == 8) hipLaunchKernelGGL((k_hcg_direction<NF, 16, 8>), g, b, 0, s, a, par);
    else if (a.tz == 4) hipLaunchKernelGGL((k_hcg_direction<NF, 16, 4>), g, b, 0, s, a, par);
    else hipLaunchKernelGGL((k_hcg_direction<NF, 16, 2>), g, b, 0, s, a, par);
  }
}

template <int TX, int TZ>
void direction_batch(const HcgArgs *tab, const int2 *unit, int nblk, int par, hipStream_t s) {
  hipLaunchKernelGGL((k_hcg_direction_batch<4, TX, TZ>), dim3(nblk), dim3(256), 0, s, tab, unit, par);
}

int up(int n, int t) { return (n + t - 1) / t; }
// tiles and work-groups with tx x (256 / tx) x tz tiles, and points per update work-group
void split(HcgArgs &a, int tx, int tz, long chunk) {
  a.tx = tx;
  a.tz = tz;
  a.ntx = up(a.nx, tx);
  a.nty = up(a.ny, 256 / tx);
  a.ntz = up(a.nz, tz);
  a.np = (int)std::min<long>(HCG_PARTS, ((long)a.ntx * a.nty * a.ntz + 7) / 8 * 8);
  a.chunk = std::max(chunk, ((a.n + HCG_PARTS - 1) / HCG_PARTS + 255) / 256 * 256);
  a.nr = (int)((a.n + a.chunk - 1) / a.chunk);
}
int planes(long tiles4) { return tiles4 < 1024 ? 2 : tiles4 <= 8192 ? 4 : 8; }

}  // namespace

void hcg_plan(HcgArgs &a, int nfh) {
  // 32 x 8 columns where 16 x 16 would leave more of the tiles empty; the planes per tile by
  // the number of tiles: few tiles want the shortest launch (2 planes: 40^3 11.7 us per iteration
  // against 12.5 with 4 and 14.3 with 8), 128^3 fewer halo rows (4: 38.4 us, 2: 41.2, 8: 42.0),
  // and far past the chip's capacity the z halo costs most (256^3, 8: 328 us, 4: 351)
  const long c32 = (long)up(a.nx, 32) * up(a.ny, 8), c16 = (long)up(a.nx, 16) * up(a.ny, 16);
  split(a, c32 < c16 ? 32 : 16, planes(std::min(c16, c32) * up(a.nz, 4)), 256);
}

void hcg_plan_batch(HcgArgs *a, int ns) {
  long t16 = 0, t32 = 0, n = 0;  // tiles of four planes, points
  for (int i = 0; i < ns; i++) {
    t16 += (long)up(a[i].nx, 16) * up(a[i].ny, 16) * up(a[i].nz, 4);
    t32 += (long)up(a[i].nx, 32) * up(a[i].ny, 8) * up(a[i].nz, 4);
    n += a[i].n;
  }
  const int tx = t32 < t16 ? 32 : 16, tz = planes(std::min(t16, t32));
  const long chunk = std::min(2048L, std::max(256L, n / 1024 / 256 * 256));  // about 1024 work-groups
  for (int i = 0; i < ns; i++) split(a[i], tx, tz, chunk);
}

void hcg_iteration_batch(const HcgArgs *dev, const int2 *dir_unit, int ndir, const int2 *upd_unit, int nupd, int tx,
                         int tz, int parity, hipStream_t s) {
  if (tx == 32) {
    if (tz == 8) direction_batch<32, 8>(dev, dir_unit, ndir, parity, s);
    else if (tz == 4) direction_batch<32, 4>(dev, dir_unit, ndir, parity, s);
    else direction_batch<32, 2>(dev, dir_unit, ndir, parity, s);
  } else {
    if (tz == 8) direction_batch<16, 8>(dev, dir_unit, ndir, parity, s);
    else if (tz == 4) direction_batch<16, 4>(dev, dir_unit, ndir, parity, s);
    else direction_batch<16, 2>(dev, dir_unit, ndir, parity, s);
  }
  hipLaunchKernelGGL(k_hcg_update_batch, dim3(nupd), dim3(256), 0, s, dev, upd_unit, parity);
  HIPCK(hipGetLastError());
}

void hcg_iteration(const HcgArgs &a, int nfh, int parity, hipStream_t s) {
  switch (nfh) {
    case 4: direction<4>(a, parity, s); break;
    case 5: direction<5>(a, parity, s); break;
    case 6: direction<6>(a, parity, s); break;
    default: throw Error(6, "error in scf_hartree! This subroutine is for nfh ne 4, 5 or 6.");
  }
  hipLaunchKernelGGL(k_hcg_update, dim3(a.nr), dim3(256), 0, s, a, parity);
  HIPCK(hipGetLastError());
}

}  // namespace kukan
