// gemm_f64.hip — FP64 subspace products on the matrix cores (v_mfma_f64_16x16x4_f64).
//
// TN: C(M1 x M2) = alpha A^T B + beta C with a grid-length inner dimension K (Gram matrices,
// Rayleigh-Ritz matrices, band projections), split over K-ranges whose partial tiles are added
// in a fixed order.
// NN: Y = alpha X C + beta Y and X <- X C with a small upper triangular C.
#include <algorithm>

#include "gemm_f64.hpp"
#include "kukan_internal.hpp"

namespace kukan {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
// four consecutive values of a column: a column starts at any multiple of 8 bytes
typedef double d4u __attribute__((ext_vector_type(4), aligned(8)));

struct TNArgs {
  const double *A, *B;
  long lda, ldb, K, KC;
  int M1, M2, nt1, npair, nchunk, tri;
  double *part;
};

// tile pair `p` of the triangle kept (0: all nt1 x nt2 pairs, 1: ti >= tj, 2: ti <= tj)
__device__ inline void tn_pair(int p, int nt1, int tri, int &ti, int &tj) {
  if (tri == 0) {
    ti = p % nt1;
    tj = p / nt1;
    return;
  }
  int a = 0, b = 0;  // a >= b, row by row
  while (p > a) p -= ++a;
  b = p;
  ti = tri == 1 ? a : b;
  tj = tri == 1 ? b : a;
}

// One work-group: a tile of 32 WT x 32 WT outputs (4 waves in 2 x 2, WT x WT MFMA tiles each)
// over one K-range.  Lane l holds, of column l % 16 of its fragment, the four consecutive k
// 4 (l / 16) .. + 3 of each 16-deep step, as 32 consecutive bytes: the four lanes of a column
// cover a whole 128-byte line, and MFMA s of the step takes each lane's value s (A and B in the
// same k order, so the sum is over the same products).  Operands go straight from L1 / L2 to
// registers, no LDS and no barriers, with the whole next step's loads in flight while a step is
// multiplied.
template <int WT>
__global__ __launch_bounds__(256) void k_tn_f64(TNArgs a) {
  constexpr int TM = 32 * WT;
  const int id = blockIdx.x, j8 = id >> 3;
  // the tile pairs of one K-range run on one XCD, so A and B come from HBM about once
  const int chunk = (j8 / a.npair) * 8 + (id & 7), pair = j8 % a.npair;
  if (chunk >= a.nchunk) return;
  int ti, tj;
  tn_pair(pair, a.nt1, a.tri, ti, tj);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, q = lane >> 4, c16 = lane & 15;
  const int r0 = ti * TM + (w & 1) * 16 * WT, s0 = tj * TM + (w >> 1) * 16 * WT;
  const long k0 = chunk * a.KC, k1 = min(a.K, k0 + a.KC);
  // byte offsets from the tile's first column (the host checks that they fit 32 bits)
  const char *pa = (const char *)(a.A + a.lda * (ti * TM) + k0), *pb = (const char *)(a.B + a.ldb * (tj * TM) + k0);
  unsigned oa[WT], ob[WT];
#pragma unroll
  for (int f = 0; f < WT; f++) {  // columns past the edge repeat the last one (results unused)
    oa[f] = (unsigned)(8 * (a.lda * (min(r0 + 16 * f + c16, a.M1 - 1) - ti * TM) + 4 * q));
    ob[f] = (unsigned)(8 * (a.ldb * (min(s0 + 16 * f + c16, a.M2 - 1) - tj * TM) + 4 * q));
  }
  d4 acc[WT][WT];
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WT; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  auto mac = [&](const d4u *x, const d4u *y) {
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
      for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i][s], y[j][s], acc[i][j], 0, 0, 0);
  };
  const long nf = (k1 - k0) / 16;  // full 16-deep steps
  d4u x[WT], y[WT];
  if (nf > 0) {
#pragma unroll
    for (int f = 0; f < WT; f++) {
      x[f] = *(const d4u *)(pa + oa[f]);
      y[f] = *(const d4u *)(pb + ob[f]);
    }
    for (long st = 1; st < nf; st++) {
      pa += 128;
      pb += 128;
      d4u xn[WT], yn[WT];
#pragma unroll
      for (int f = 0; f < WT; f++) {
        xn[f] = *(const d4u *)(pa + oa[f]);
        yn[f] = *(const d4u *)(pb + ob[f]);
      }
      mac(x, y);
#pragma unroll
      for (int f = 0; f < WT; f++) {
        x[f] = xn[f];
        y[f] = yn[f];
      }
    }
    mac(x, y);
    pa += 128;
    pb += 128;
  }
  const int rem = (int)(k1 - k0 - 16 * nf);
  if (rem > 0) {  // the last, partial step: values past k1 are zero on both sides
#pragma unroll
    for (int f = 0; f < WT; f++)
#pragma unroll
      for (int s = 0; s < 4; s++) {
        const bool in = 4 * q + s < rem;
        x[f][s] = in ? *(const double *)(pa + oa[f] + 8 * s) : 0.0;
        y[f][s] = in ? *(const double *)(pb + ob[f] + 8 * s) : 0.0;
      }
    mac(x, y);
  }
  // partial tile, wave by wave in register order (64 consecutive doubles per store); the
  // reduction undoes the layout: register r of lane l is row l / 16 + 4 r, column l % 16
  double *o = a.part + ((long)pair * a.nchunk + chunk) * (TM * TM) + w * (256 * WT * WT);
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) o[((i * WT + j) * 4 + r) * 64 + lane] = acc[i][j][r];
}

// The same 128 x 128 tile with both operands staged in LDS by LDS-DMA (buffer_load ... lds, 16
// bytes per lane, nothing through registers): every value is fetched from L2 once per work-group
// instead of once per wave that uses it.  Two 32 KB slots (the next 16-deep step lands while
// the current one is multiplied, one barrier per step), two work-groups per CU.
// LDS layout: column c's 128-byte row holds its 16-byte chunk m at slot m ^ ((c >> 1) & 7).  The
// DMA writes 64 consecutive chunks per wave, so the swizzle is in the source address of each
// lane; the fragment reads (16 columns, one chunk each) then fall on all 64 banks once.
// Columns past the matrix lie outside the buffer's range and read zero.  Needs 16-byte aligned
// columns.
typedef double d2 __attribute__((ext_vector_type(2)));
#define GF_LDS(x) ((__attribute__((address_space(3))) void *)(x))
// Between two steps of a ring of two slots: this wave's loads into the next slot have landed and its
// reads of the other slot have returned (vmcnt 0 and lgkmcnt 0), then every wave's.  The reads have
// to be waited for here: the barrier alone would let another wave's loads overwrite a slot whose
// values the compiler need not have used yet.
__device__ inline void ring_step() {
  __builtin_amdgcn_s_waitcnt(0x0070);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}
__global__ __launch_bounds__(256, 2) void k_tn_f64_lds(TNArgs a) {
  constexpr int WT = 4, TM = 128;
  __shared__ __attribute__((aligned(1024))) char ring[2][2][TM * 128];  // [slot][A, B]
  const int id = blockIdx.x, j8 = id >> 3;
  const int chunk = (j8 / a.npair) * 8 + (id & 7), pair = j8 % a.npair;
  if (chunk >= a.nchunk) return;
  int ti, tj;
  tn_pair(pair, a.nt1, a.tri, ti, tj);
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, q = lane >> 4, c16 = lane & 15;
  const int ws = __builtin_amdgcn_readfirstlane(w);
  const long k0 = chunk * a.KC, k1 = min(a.K, k0 + a.KC);
  const int nf = (int)((k1 - k0) / 16);
  // operand o: base of the tile's first column at k0; this wave stages columns 32 w .. + 31, and
  // span is the bytes from its first column to the end of the last one (none left: 0)
  const char *base[2] = {(const char *)(a.A + a.lda * (ti * TM) + k0), (const char *)(a.B + a.ldb * (tj * TM) + k0)};
  const long ld8[2] = {8 * a.lda, 8 * a.ldb};
  const int left[2] = {a.M1 - ti * TM - 32 * ws, a.M2 - tj * TM - 32 * ws};
  long span[2];
#pragma unroll
  for (int o = 0; o < 2; o++) span[o] = left[o] > 0 ? ld8[o] * (left[o] - 1) + 8 * (a.K - k0) : 0;
  // this lane's source within an 8-column group: column lane / 8, chunk (lane % 8) ^ (lane / 16),
  // the odd groups' chunk ^ 4
  const unsigned ch = 16 * ((lane & 7) ^ (lane >> 4));
  unsigned off[2][4];
#pragma unroll
  for (int o = 0; o < 2; o++)
#pragma unroll
    for (int i = 0; i < 4; i++)
      off[o][i] = (unsigned)(ld8[o] * (8 * i + (lane >> 3))) + (ch ^ (i & 1 ? 64u : 0u));
  auto issue = [&](int st) {
#pragma unroll
    for (int o = 0; o < 2; o++) {
      const long left = min(max(span[o] - 128L * st, 0L), 0xFFFFFFF0L);
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void *)(base[o] + 32 * ld8[o] * ws + 128L * st), (short)0, (int)(unsigned)left, 0x00020000);
      char *d = &ring[st & 1][o][ws * 4096];
#pragma unroll
      for (int i = 0; i < 4; i++)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, GF_LDS(d + 1024 * i), 16, off[o][i], 0, 0, 0);
    }
  };
  d4 acc[WT][WT];
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WT; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  // fragment f of this wave: column 64 wi + 16 f + c16, chunks q and q + 4
  const int la = 128 * (64 * (w & 1) + c16) + 16 * (q ^ (c16 >> 1)), lb = 128 * (64 * (w >> 1) + c16) + 16 * (q ^ (c16 >> 1));
  if (nf > 0) issue(0);
  for (int st = 0; st < nf; st++) {
    ring_step();
    if (st + 1 < nf) issue(st + 1);
    const char *A = ring[st & 1][0], *B = ring[st & 1][1];
    d2 x[2][WT], y[2][WT];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int f = 0; f < WT; f++) {
        x[h][f] = *(const d2 *)(A + ((la + 2048 * f) ^ (64 * h)));
        y[h][f] = *(const d2 *)(B + ((lb + 2048 * f) ^ (64 * h)));
      }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < WT; i++)
#pragma unroll
          for (int j = 0; j < WT; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[h][i][s], y[h][j][s], acc[i][j], 0, 0, 0);
  }
  const int rem = (int)(k1 - k0) - 16 * nf;
  if (rem > 0) {  // the last, partial step, from global memory: values past k1 are zero
    const double *A = (const double *)(base[0]) + 16L * nf, *B = (const double *)(base[1]) + 16L * nf;
#pragma unroll
    for (int s = 0; s < 4; s++) {
      double x[WT], y[WT];
      const bool in = 4 * q + s < rem;
#pragma unroll
      for (int f = 0; f < WT; f++) {
        const int ca = 64 * (w & 1) + 16 * f + c16, cb = 64 * (w >> 1) + 16 * f + c16;
        x[f] = in && ti * TM + ca < a.M1 ? A[a.lda * ca + 4 * q + s] : 0.0;
        y[f] = in && tj * TM + cb < a.M2 ? B[a.ldb * cb + 4 * q + s] : 0.0;
      }
#pragma unroll
      for (int i = 0; i < WT; i++)
#pragma unroll
        for (int j = 0; j < WT; j++) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[i], y[j], acc[i][j], 0, 0, 0);
    }
  }
  double *o = a.part + ((long)pair * a.nchunk + chunk) * (TM * TM) + w * (256 * WT * WT);
#pragma unroll
  for (int i = 0; i < WT; i++)
#pragma unroll
    for (int j = 0; j < WT; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) o[((i * WT + j) * 4 + r) * 64 + lane] = acc[i][j][r];
}

// C = alpha sum over K-ranges + beta C: 64 outputs per work-group, four threads each take a
// quarter of the K-ranges and the four sums are added in order
template <int WT>
__global__ __launch_bounds__(256) void k_tn_f64_reduce(TNArgs a, double alpha, double beta,
                                                       double *C, long ldc) {
  constexpr int TM = 32 * WT;
  __shared__ double red[4][64];
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int pair = blockIdx.y, e0 = blockIdx.x * 64;
  const double *p = a.part + (long)pair * a.nchunk * (TM * TM) + e0 + lane;
  const int per = (a.nchunk + 3) / 4, c0 = g * per, c1 = min(a.nchunk, c0 + per);
  double s = 0.0;
#pragma unroll 8
  for (int c = c0; c < c1; c++) s += p[(long)c * (TM * TM)];
  red[g][lane] = s;
  __syncthreads();
  if (g) return;
  s = ((red[0][lane] + red[1][lane]) + red[2][lane]) + red[3][lane];
  int ti, tj;
  tn_pair(pair, a.nt1, a.tri, ti, tj);
  const int u = e0 / 64, r = u & 3, f = (u >> 2) % (WT * WT), w = (u >> 2) / (WT * WT);
  const int i = ti * TM + (w & 1) * 16 * WT + 16 * (f / WT) + (lane >> 4) + 4 * r;
  const int j = tj * TM + (w >> 1) * 16 * WT + 16 * (f % WT) + (lane & 15);
  if (i >= a.M1 || j >= a.M2) return;
  double *c = C + i + ldc * j;
  *c = beta == 0.0 ? alpha * s : alpha * s + beta * *c;
}

template <int WT>
void tn_launch(TNArgs a, bool lds, double alpha, double beta, double *C, long ldc, hipStream_t s) {
  constexpr int TM = 32 * WT;
  const int nt1 = (a.M1 + TM - 1) / TM, nt2 = (a.M2 + TM - 1) / TM;
  a.nt1 = nt1;
  a.npair = a.tri ? nt1 * (nt1 + 1) / 2 : nt1 * nt2;
  // K-ranges: a multiple of 8 (one XCD each in turn), at least 256 deep, the count whose
  // rounds of resident work-groups (WT 4: 1 per CU, 2: 4, 1: 8) times depth is least; 128
  // stands for a range's own start and end
  const long res = lds ? 64 : WT == 4 ? 32 : WT == 2 ? 128 : 256;  // per XCD
  long best = 0;
  double cost = 1e300;
  for (long nc = 8; nc <= 2048 && (nc == 8 || nc * 256 <= a.K + 2047); nc += 8) {
    const long kc = (a.K + nc - 1) / nc, rounds = (nc / 8 * a.npair + res - 1) / res;
    const double c = (double)rounds * (kc + 128);
    if (c < cost * 0.99) {
      cost = c;
      best = nc;
    }
  }
  a.KC = ((a.K + best - 1) / best + 15) / 16 * 16;
  a.nchunk = (int)std::max(1L, (a.K + a.KC - 1) / a.KC);
  a.part = (double *)scratch("gemm64.part", sizeof(double) * TM * TM * (size_t)a.npair * a.nchunk);
  const unsigned grid = (unsigned)((long)(a.nchunk + 7) / 8 * 8 * a.npair);
  if (lds) hipLaunchKernelGGL(k_tn_f64_lds, dim3(grid), dim3(256), 0, s, a);
  else hipLaunchKernelGGL(k_tn_f64<WT>, dim3(grid), dim3(256), 0, s, a);
  hipLaunchKernelGGL(k_tn_f64_reduce<WT>, dim3(TM * TM / 64, a.npair), dim3(256), 0, s, a, alpha,
                     beta, C, ldc);
  HIPCK(hipGetLastError());
}

// ----------------------------------------------------------------------------- NN
// Y(R x M2) = alpha X(R x K) C(K x M2) + beta Y with C upper triangular: the projection of K r
// on the lower bands and the application of a Cholesky factor's inverse.
struct NNArgs64 {
  const double *X, *C;  // C: prepared (k_nn_f64_prep), column j at C + Kp j
  double *Y;
  long ldx, ldy, R, row_blocks;
  int K, Kp, M2, ct0, nct;
  double beta;
};

// the upper triangle of C, times alpha, padded with zeros to Kp rows (a multiple of 16) and whole
// tiles of 128 columns; what C holds below the diagonal is not read
__global__ void k_nn_f64_prep(int K, int Kp, int M2, double alpha, const double *C, long ldc, double *out) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (k >= Kp) return;
  out[(long)Kp * j + k] = k < K && j < M2 && k <= j ? alpha * C[k + ldc * j] : 0.0;
}

// 128 points x 128 columns per work-group, both operands through LDS as in k_tn_f64_lds: a
// 16-deep step is 16 bands x 128 points of X (1 KB runs) and 128 columns x 16 rows of C (128-byte
// rows, chunks swizzled).  The MFMA's columns are points and its rows bands, so a lane's results
// are two neighbouring points of one band and the loads and stores of Y are 256-byte runs; lane
// values of X are two points each (points 2 (l % 16), + 1 of a 32-point group feed two tiles).
// The steps below a column tile's last row are skipped: their products are exact zeros.
__global__ __launch_bounds__(256, 2) void k_nn_f64(NNArgs64 a) {
  constexpr int TM = 128;
  __shared__ __attribute__((aligned(1024))) char ring[2][2][TM * 128];  // [slot][X, C]
  const int id = blockIdx.x, j8 = id >> 3;
  // the column tiles of one row block run on one XCD, so X comes from HBM about once
  const long rb = (long)(j8 / a.nct) * 8 + (id & 7);
  if (rb >= a.row_blocks) return;
  const int c0 = (a.ct0 + j8 % a.nct) * TM;
  const long r0 = rb * TM;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, q = lane >> 4, c16 = lane & 15;
  const int ws = __builtin_amdgcn_readfirstlane(w), wi = w & 1, wj = w >> 1;
  const int nst = min(a.Kp, c0 + TM) / 16;
  const char *xb = (const char *)(a.X + r0), *cb = (const char *)(a.C + (long)a.Kp * c0);
  const long ldx8 = 8 * a.ldx;
  const unsigned ch = 16 * ((lane & 7) ^ (lane >> 4));
  unsigned offx[4], offc[4];
#pragma unroll
  for (int i = 0; i < 4; i++) {
    offx[i] = (unsigned)(ldx8 * (4 * w + i) + 16 * lane);
    offc[i] = (unsigned)(8 * a.Kp * (8 * (4 * w + i) + (lane >> 3))) + (ch ^ (i & 1 ? 64u : 0u));
  }
  auto issue = [&](int st) {
    // bytes of X from row 16 st to the end of its last column (values past it read zero)
    const long span = ldx8 * (a.K - 1 - 16 * st) + 8 * (a.R - r0);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(xb + 16 * ldx8 * st), (short)0, (int)(unsigned)min(span, 0xFFFFFFF0L), 0x00020000);
    const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(cb + 128L * st), (short)0, (int)(8 * a.Kp * TM - 128 * st), 0x00020000);
    char *dx = &ring[st & 1][0][ws * 4096], *dc = &ring[st & 1][1][ws * 4096];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rx, GF_LDS(dx + 1024 * i), 16, offx[i], 0, 0, 0);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rc, GF_LDS(dc + 1024 * i), 16, offc[i], 0, 0, 0);
    }
  };
  d4 acc[4][4];  // [16 columns][16 points]
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
  const int lc = 128 * (64 * wi + c16) + 16 * (q ^ (c16 >> 1)), lx = 2048 * q + 512 * wj + 16 * c16;
  issue(0);
  for (int st = 0; st < nst; st++) {
    ring_step();
    if (st + 1 < nst) issue(st + 1);
    const char *X = ring[st & 1][0], *C = ring[st & 1][1];
    d2 x[2][2][2], y[2][4];
#pragma unroll
    for (int h = 0; h < 2; h++) {
#pragma unroll
      for (int f = 0; f < 4; f++) y[h][f] = *(const d2 *)(C + ((lc + 2048 * f) ^ (64 * h)));
#pragma unroll
      for (int s = 0; s < 2; s++)  // band 2 (q + 4 h) + s
#pragma unroll
        for (int g = 0; g < 2; g++) x[h][s][g] = *(const d2 *)(X + lx + 8192 * h + 1024 * s + 256 * g);
    }
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
      for (int s = 0; s < 2; s++)
#pragma unroll
        for (int i = 0; i < 4; i++)
#pragma unroll
          for (int j = 0; j < 4; j++)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(y[h][i][s], x[h][s][j >> 1][j & 1], acc[i][j], 0, 0, 0);
  }
  // a wave's 16 columns x 64 points at a time; with beta the Y values of the next 16 columns are
  // loaded while these are written (past the last point or column: the last ones again, unused)
  d2 yo[2][4][2];
  auto fetch = [&](int i) {
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const int j = min(c0 + 64 * wi + 16 * i + q + 4 * r, a.M2 - 1);
        yo[i & 1][r][g] = *(const d2 *)(a.Y + a.ldy * j + min(r0 + 64 * wj + 32 * g + 2 * c16, a.R - 2));
      }
  };
  if (a.beta != 0.0) fetch(0);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    if (a.beta != 0.0 && i < 3) fetch(i + 1);
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int j = c0 + 64 * wi + 16 * i + q + 4 * r;
      if (j >= a.M2) continue;
#pragma unroll
      for (int g = 0; g < 2; g++) {
        const long p = r0 + 64 * wj + 32 * g + 2 * c16;
        d2 v = {acc[i][2 * g][r], acc[i][2 * g + 1][r]};
        if (a.beta != 0.0) v += a.beta * yo[i & 1][r][g];
        if (p < a.R) *(d2 *)(a.Y + a.ldy * j + p) = v;
      }
    }
  }
}

}  // namespace

static bool aligned16(const void *p, long ld) { return (uintptr_t)p % 16 == 0 && ld % 2 == 0; }

// R even: a lane loads and stores points in pairs (the bands' own length, so an odd one has columns
// that are not 16-byte aligned either)
static bool nn_ok(const double *X, long ldx, const double *Y, long ldy, long R, int K, int M2) {
  return param("gemm_f64", 1.0) >= 1.0 && R > 0 && R % 2 == 0 && K > 0 && M2 > 0 && aligned16(X, ldx) &&
         aligned16(Y, ldy) && ldx < (1L << 24) && K <= 16384;
}

static NNArgs64 nn_prepare(long R, int K, int M2, double alpha, const double *X, long ldx, const double *C,
                           long ldc, double *Y, long ldy, hipStream_t s) {
  NNArgs64 a{};
  a.X = X; a.Y = Y; a.ldx = ldx; a.ldy = ldy; a.R = R; a.K = K; a.M2 = M2;
  a.Kp = (K + 15) / 16 * 16;
  a.nct = (M2 + 127) / 128;
  a.row_blocks = (R + 127) / 128;
  double *cp = (double *)scratch("gemm64.C", sizeof(double) * (size_t)a.Kp * 128 * a.nct);
  hipLaunchKernelGGL(k_nn_f64_prep, dim3((a.Kp + 63) / 64, 128 * a.nct), dim3(64), 0, s, K, a.Kp, M2, alpha, C,
                     ldc, cp);
  a.C = cp;
  return a;
}
static unsigned nn_grid(const NNArgs64 &a) { return (unsigned)((a.row_blocks + 7) / 8 * 8 * a.nct); }

// For a full C the kernel and rocBLAS dgemm take the same time (884736 x 512: 6.9 ms both), so
// it is used where C is triangular and a column tile's steps can be skipped; up to 64 columns
// half the tile is padding (884736 x 64, beta 1: 0.39 against 0.36 ms).
bool gemm_f64_nn_upper(long R, int K, int M2, double alpha, const double *X, long ldx, const double *C, long ldc,
                       double beta, double *Y, long ldy, hipStream_t s) {
  if (M2 <= 64 || alpha == 0.0 || !nn_ok(X, ldx, Y, ldy, R, K, M2)) return false;
  const double k = std::min(K, M2);  // column j takes its first j + 1 rows, at most K
  Timed t("gemm_f64", (double)R * (k * (k + 1.0) + 2.0 * K * (M2 - k)));
  NNArgs64 a = nn_prepare(R, K, M2, alpha, X, ldx, C, ldc, Y, ldy, s);
  a.beta = beta;
  hipLaunchKernelGGL(k_nn_f64, dim3(nn_grid(a)), dim3(256), 0, s, a);
  HIPCK(hipGetLastError());
  return true;
}

// Against dtrsm, which needs no inverse of the factor (a whole orthonormalisation with either, own /
// dtrsm): up to 32 bands dtrsm is one pass and the inverse costs more than the rest (262144 points x
// 20: 323 / 244 us, x 48: 429 / 474; 884736 x 32: 505 / 469) except on the longest bands, where the
// passes count (2097152 x 32: 970 / 1036, x 24: 880 / 793); on short bands the inverse is never
// repaid (4096 x 500: 1901 / 1736, 13824 x 800: 3299 / 3099, 32768 x 200: 892 / 935).
bool apply_upper_ok(long R, int M, const double *X, long ldx) {
  return R >= 32768 && M > (R < (1L << 21) ? 32 : 24) && nn_ok(X, ldx, X, ldx, R, M, M);
}

void gemm_f64_apply_upper(long R, int M, double *X, long ldx, const double *C, long ldc, hipStream_t s) {
  NNArgs64 a = nn_prepare(R, M, M, 1.0, X, ldx, C, ldc, X, ldx, s);
  const int tiles = a.nct;
  a.nct = 1;
  for (a.ct0 = tiles - 1; a.ct0 >= 0; a.ct0--) hipLaunchKernelGGL(k_nn_f64, dim3(nn_grid(a)), dim3(256), 0, s, a);
  HIPCK(hipGetLastError());
}

// Which TN kernel, from times at K = 512 .. 8000000 (rocBLAS dgemm beside them; its times jump between
// neighbouring sizes, and many are ten times these):
//  - at most 32 columns on both sides: 32 x 32 tiles (4096000 x 16 0.34 ms, in 64 x 64 tiles, whose
//    padding is multiplied too, 0.56, dgemm 0.37; 64000 x 32 0.028, 0.034 and 10.2);
//  - at most 64 on one side: 64 x 64 tiles.  rocBLAS runs the whole K in one tile's work-group
//    there: 64000 x 64 takes 10.2 ms against 0.036 ms, 884736 x 64 1.70 against 0.26;
//  - 16-byte aligned columns: 128 x 128 tiles through LDS, 73-75 TFLOP/s from 384 columns on
//    (884736 x 512: 6.34 ms against 8.0; its triangle 4.23 against 5.9 in 256-column blocks;
//    2097152 x 1024, the triangle: 33.7 against 44.5).  Past 128 columns a short K does not repay
//    the eight K-ranges' partial tiles and the launch that adds them: 512 x 512 34 us against 25,
//    768 x 768 52 against 41, but 1024 x 1000 67 against 73; with more than 144 tiles K has to be six
//    times the columns (8192 x 2000 1075 against 915, 12000 x 2000 1538 against 1977), and a full
//    square past 3072 is rocBLAS's (16384 x 4096 8.42 ms against 8.05);
//  - otherwise (an odd column length): the direct 128 x 128 kernel where it is at least as fast
//    as rocBLAS, up to 128 columns (253440 x 100: 0.18 against 40.6 ms), for a triangle up to 384
//    (3.1 against 6.0 ms).
enum class TN { none, t32, t64, lds128, t128 };
static TN tn_kind(int M1, int M2, long K, const double *A, long lda, const double *B, long ldb, int tri) {
  const long ld = std::max(lda, ldb);
  if (param("gemm_f64", 1.0) < 1.0 || M1 <= 0 || M2 <= 0 || K <= 0 || ld >= (1L << 24)) return TN::none;
  const int most = std::max(M1, M2);
  // (the direct kernels' 32-bit offsets within a tile bound the column length)
  if (most <= 32) return TN::t32;
  if (std::min(M1, M2) <= 64 && ld < (1L << 23)) return TN::t64;
  const bool half = tri && M1 == M2;
  if (aligned16(A, lda) && aligned16(B, ldb)) {
    const long nt1 = (M1 + 127) / 128, nt2 = (M2 + 127) / 128, tiles = half ? nt1 * (nt1 + 1) / 2 : nt1 * nt2;
    const bool slow = (most > 128 && K < 1024) || (tiles > 144 && K < 6L * most) || (!half && tiles > 576);
    return slow ? TN::none : TN::lds128;
  }
  return ld < (1L << 22) && most <= (half ? 384 : 128) ? TN::t128 : TN::none;
}

bool gemm_f64_tn(int M1, int M2, long K, double alpha, const double *A, long lda, const double *B,
                 long ldb, double beta, double *C, long ldc, int tri, hipStream_t s) {
  const TN kind = alpha == 0.0 ? TN::none : tn_kind(M1, M2, K, A, lda, B, ldb, tri);
  if (kind == TN::none) return false;
  // the flops of the entries asked for: of a triangle M1 (M1 + 1) / 2
  Timed t("gemm_f64", (double)K * M1 * (tri && M1 == M2 ? M1 + 1.0 : 2.0 * M2));
  TNArgs a{};
  a.A = A; a.B = B; a.lda = lda; a.ldb = ldb; a.K = K; a.M1 = M1; a.M2 = M2;
  a.tri = M1 == M2 ? tri : 0;
  if (kind == TN::t32) tn_launch<1>(a, false, alpha, beta, C, ldc, s);
  else if (kind == TN::t64) tn_launch<2>(a, false, alpha, beta, C, ldc, s);
  else tn_launch<4>(a, kind == TN::lds128, alpha, beta, C, ldc, s);
  return true;
}

}  // namespace kukan
