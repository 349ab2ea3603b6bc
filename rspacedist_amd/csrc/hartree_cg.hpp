// hartree_cg.hpp — one iteration of the Hartree CG as two launches (hartree_cg.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "kukan_internal.hpp"

namespace kukan {

constexpr int HCG_PARTS = 1024;  // most partial sums of either kernel

struct HcgArgs {
  int nx, ny, nz, px, py, pz;
  double cx[9], cy[9], cz[9], c0;
  long n;
  double *vh, *r, *p[2], *ap;  // p: the direction alternates between the two buffers
  double *part_p, *part_r;     // <p|A p> and <r|r> partials (HCG_PARTS each)
  double *rr;                  // rr[k & 1]: <r|r> before iteration k; rr[1] is set at the start
  int *state;                  // {done, iteration (1-based), iterations taken}
  int ncgres, ncgmin, ncgmax;
  double dvo, eps;
  // filled by hcg_plan
  int ntx, nty, ntz, np, nr, tx, tz;
  long chunk;
};
void hcg_plan(HcgArgs &a, int nfh);
// the iterations 1 + parity, 3 + parity, ... (parity 0 or 1): p[parity] is read, p[1 - parity]
// written; p[0] must hold finite values before the first
void hcg_iteration(const HcgArgs &a, int nfh, int parity, hipStream_t s);

// Several solves with nfh = 4 in lock step: one tile shape for all of them, the arguments in a
// device table and a table {solve, work-group of the solve} per launch, each solve's np (nr)
// work-groups in order.  A range of solves may be run by itself with its part of the tables.
void hcg_plan_batch(HcgArgs *a, int ns);
void hcg_iteration_batch(const HcgArgs *dev, const int2 *dir_unit, int ndir, const int2 *upd_unit, int nupd, int tx,
                         int tz, int parity, hipStream_t s);

}  // namespace kukan
