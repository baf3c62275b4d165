// kernels_cg.hip -- the many-launch form of the Jacobi-preconditioned CG that replaces
// Eigen::ConjugateGradient (include/FluidSolver.h:114, src/FluidSolver.cpp:81,362-425):
// three kernels per iteration, for systems of more unknowns than the one-launch form
// (kernels_pcg.hip) holds in registers (about 2^20), and for a plain solve whose
// co-resident launch was refused or gave up a wait.
//
// Unknowns are the LIQUID cells in row-major order (kernels_pcg.hip's set-up).  The operator
// is applied matrix-free: one info byte per unknown holds the four LIQUID-neighbour bits
// and the count of non-SOLID neighbours, so A's row is diag_tab[count] at the centre and
// off = 1/dx^2 at each LIQUID neighbour; x and p are cell grids.
//
// Synchronisation on gfx950 (measured): a contended returning atomic costs ~90 ns
// per block and agent-scope release/acquire fences write back and invalidate L2.
// So no kernel here uses a last-block ticket or an agent-scope fence: every block
// re-sums the previous kernel's per-block partials in a fixed order (kernel boundaries
// order the data).  Every sum is deterministic (fixed per-thread order, fixed wave /
// block tree, fixed block order).
#include <float.h>

#include "fsg_common.h"
#include "fsg_device.h"
#include "fsg_kernels.h"

namespace fsg {

// ------------------------------------------------------------ system setup
// Exclusive scan of the tiles' LIQUID counts in one block of 1024 threads.
__global__ void __launch_bounds__(1024) k_scan_counts(int nb, const int* __restrict__ counts,
                                                      int* __restrict__ offsets,
                                                      int* __restrict__ n_fluid) {
  __shared__ int sm[1024];
  const int per = (nb + 1023) / 1024;
  const int b0 = threadIdx.x * per;
  int s = 0;
  for (int q = 0; q < per; ++q)
    if (b0 + q < nb) s += counts[b0 + q];
  sm[threadIdx.x] = s;
  __syncthreads();
  for (int off = 1; off < 1024; off <<= 1) {
    const int v = threadIdx.x >= off ? sm[threadIdx.x - off] : 0;
    __syncthreads();
    sm[threadIdx.x] += v;
    __syncthreads();
  }
  int run = sm[threadIdx.x] - s;  // exclusive prefix of this thread's first tile
  for (int q = 0; q < per; ++q)
    if (b0 + q < nb) {
      offsets[b0 + q] = run;
      run += counts[b0 + q];
    }
  if (threadIdx.x == 1023) *n_fluid = sm[1023];
}

// ---------------------------------------------------------------- plain form
// Eigen's conjugate_gradient restated (x0 = 0; stop when |r|^2 < max(tol^2 |b|^2,
// min normal) or after max_iter iterations), one iteration = 3 kernels:
//   spmv:    Ap = A p, partial p.Ap
//   update:  alpha = r.z / p.Ap; x += alpha p, r -= alpha Ap; partial |r|^2, r.z
//   pupdate: stop test, beta = r.z_new / r.z; p = z + beta p
// Each kernel's blocks re-sum the previous kernel's partials in block order;
// block 0 records the scalars for the host.  Scalars are formed in float like
// Eigen's RealScalar; sums are reduced in FP64.

constexpr int kPlainThreads = 256;

template <int NV>
__device__ __forceinline__ void sum_partials(const double* part, int nb, double (&v)[NV],
                                             double* sm) {
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = 0.0;
  for (int b = threadIdx.x; b < nb; b += kPlainThreads)
#pragma unroll
    for (int q = 0; q < NV; ++q) v[q] += part[b * NV + q];
  block_sum<NV, kPlainThreads>(v, sm);
}

template <int NV>
__device__ __forceinline__ void write_partials(double (&v)[NV], double* part, double* sm) {
  block_sum<NV, kPlainThreads>(v, sm);
  if (threadIdx.x == 0)
#pragma unroll
    for (int q = 0; q < NV; ++q) part[blockIdx.x * NV + q] = v[q];
}

__global__ void __launch_bounds__(256) k_cg_sum_b(int F, const float* __restrict__ b,
                                                  double* __restrict__ part) {
  __shared__ double sm[4];
  double v[1] = {0.0};
  for (int k = blockIdx.x * 256 + threadIdx.x; k < F; k += gridDim.x * 256) v[0] += b[k];
  write_partials<1>(v, part, sm);
}

__global__ void __launch_bounds__(256) k_cg_init(int F, CgParams cp, const int* __restrict__ cell_of,
                                                 const uint8_t* __restrict__ info,
                                                 const float* __restrict__ b, float* __restrict__ r,
                                                 float* __restrict__ pg, float* __restrict__ xg,
                                                 const double* __restrict__ mean_part,
                                                 double* __restrict__ part, CgScalars* sc) {
  __shared__ double sm[2 * 4];
  float mean = 0.f;
  if (cp.project_mean) {
    double m[1];
    sum_partials<1>(mean_part, gridDim.x, m, sm);
    mean = (float)m[0] / (float)F;
  }
  double v[2] = {0.0, 0.0};
  for (int k = blockIdx.x * 256 + threadIdx.x; k < F; k += gridDim.x * 256) {
    const int c = cell_of[k];
    const float rk = cp.project_mean ? b[k] - mean : b[k];
    const float z = sel5((info[k] >> 4) & 7, cp.invd_tab) * rk;
    r[k] = rk;
    pg[c] = z;
    xg[c] = 0.f;
    v[0] += (double)(rk * rk);
    v[1] += (double)(rk * z);
  }
  write_partials<2>(v, part, sm);
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->done = 0;
    sc->iter = 0;
    sc->spmv = 0;
    sc->err = 0.0;
  }
}

// part0: (|r|^2, r.z) of the previous update (or init, it == 0); part1: p.Ap out
__global__ void __launch_bounds__(256) k_cg_spmv(int F, int nx, int it, CgParams cp,
                                                 const int* __restrict__ cell_of,
                                                 const uint8_t* __restrict__ info,
                                                 const float* __restrict__ pg, float* __restrict__ ap,
                                                 const double* __restrict__ part_rz,
                                                 double* __restrict__ part_pap, CgScalars* sc) {
  __shared__ double sm[2 * 4];
  if (it == 0) {
    // Eigen's entry checks: |b|^2 == 0 -> x = 0; |r0|^2 < threshold -> done
    double v[2];
    sum_partials<2>(part_rz, gridDim.x, v, sm);
    const float rhs = (float)v[0];
    float thr = cp.tol * cp.tol * rhs;
    if (thr < FLT_MIN) thr = FLT_MIN;
    const bool stop = rhs == 0.f || rhs < thr;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
      sc->rhs_norm2 = rhs;
      sc->threshold = thr;
      sc->rz[0] = (float)v[1];
      sc->rr = rhs;
      sc->err = rhs == 0.f ? 0.0 : (stop ? 1.0 : 0.0);
      if (stop) sc->done = 1;
    }
    if (stop) return;
  } else if (sc->done) {
    return;
  }
  double v[1] = {0.0};
  for (int k = blockIdx.x * 256 + threadIdx.x; k < F; k += gridDim.x * 256) {
    const int c = cell_of[k];
    const uint8_t inf = info[k];
    const float pc = pg[c];
    float acc = sel5((inf >> 4) & 7, cp.diag_tab) * pc;
    if (inf & 1) acc += cp.off * pg[c - 1];
    if (inf & 2) acc += cp.off * pg[c + 1];
    if (inf & 4) acc += cp.off * pg[c - nx];
    if (inf & 8) acc += cp.off * pg[c + nx];
    ap[k] = acc;
    v[0] += (double)(pc * acc);
  }
  write_partials<1>(v, part_pap, sm);
}

__global__ void __launch_bounds__(256) k_cg_update(int F, int it, CgParams cp,
                                                   const int* __restrict__ cell_of,
                                                   const uint8_t* __restrict__ info,
                                                   float* __restrict__ r, const float* __restrict__ ap,
                                                   const float* __restrict__ pg, float* __restrict__ xg,
                                                   const double* __restrict__ part_pap,
                                                   double* __restrict__ part_rz, CgScalars* sc) {
  __shared__ double sm[2 * 4];
  if (sc->done) return;
  double pap[1];
  sum_partials<1>(part_pap, gridDim.x, pap, sm);
  const float alpha = sc->rz[it & 1] / (float)pap[0];
  double v[2] = {0.0, 0.0};
  for (int k = blockIdx.x * 256 + threadIdx.x; k < F; k += gridDim.x * 256) {
    const int c = cell_of[k];
    xg[c] = xg[c] + alpha * pg[c];
    const float rk = r[k] - alpha * ap[k];
    r[k] = rk;
    const float z = sel5((info[k] >> 4) & 7, cp.invd_tab) * rk;
    v[0] += (double)(rk * rk);
    v[1] += (double)(rk * z);
  }
  write_partials<2>(v, part_rz, sm);
}

__global__ void __launch_bounds__(256) k_cg_pupdate(int F, int it, CgParams cp,
                                                    const int* __restrict__ cell_of,
                                                    const uint8_t* __restrict__ info,
                                                    const float* __restrict__ r, float* __restrict__ pg,
                                                    const double* __restrict__ part_rz, CgScalars* sc) {
  __shared__ double sm[2 * 4];
  if (sc->done) return;
  double v[2];
  sum_partials<2>(part_rz, gridDim.x, v, sm);
  const float rr = (float)v[0];
  const bool conv = rr < (float)sc->threshold;
  const float abs_old = sc->rz[it & 1];
  const float abs_new = (float)v[1];
  const float beta = abs_new / abs_old;
  const bool last = !conv && it + 1 >= cp.max_iter;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->rr = rr;
    sc->err = sqrt((double)rr / sc->rhs_norm2);
    sc->spmv = it + 1;
    if (conv) {
      sc->iter = it;
      sc->done = 1;
    } else {
      sc->iter = it + 1;
      sc->rz[(it + 1) & 1] = abs_new;
      sc->beta = beta;
      if (last) sc->done = 1;
    }
  }
  if (conv || last) return;
  for (int k = blockIdx.x * 256 + threadIdx.x; k < F; k += gridDim.x * 256) {
    const int c = cell_of[k];
    const float z = sel5((info[k] >> 4) & 7, cp.invd_tab) * r[k];
    pg[c] = z + beta * pg[c];
  }
}

static inline int cg_blocks(int F) {
  int nb = (F + 1023) / 1024;  // ~4 unknowns per thread
  if (nb < 1) nb = 1;
  if (nb > 1024) nb = 1024;
  return nb;
}

void launch_scan_counts(hipStream_t s, int nb, const int* counts, int* offsets, int* n_fluid) {
  k_scan_counts<<<1, 1024, 0, s>>>(nb, counts, offsets, n_fluid);
}
void launch_cg_init(hipStream_t s, int F, const CgParams& cp, const int* cell_of,
                    const uint8_t* info, const float* b, float* r, float* pg, float* xg,
                    double* partials, CgScalars* sc) {
  const int nb = cg_blocks(F);
  // partials layout: [0, 4096) mean, [4096, 8192) r.z sets (2 x 2 values), [12288,...) p.Ap
  double* mean_part = partials;
  if (cp.project_mean) k_cg_sum_b<<<nb, 256, 0, s>>>(F, b, mean_part);
  k_cg_init<<<nb, 256, 0, s>>>(F, cp, cell_of, info, b, r, pg, xg, mean_part, partials + 4096, sc);
}
void launch_cg_iteration(hipStream_t s, int F, int nx, int it, const CgParams& cp,
                         const int* cell_of, const uint8_t* info, float* r, float* ap, float* pg,
                         float* xg, double* partials, CgScalars* sc) {
  const int nb = cg_blocks(F);
  double* rz_prev = partials + 4096 + (it & 1) * 2048;
  double* rz_next = partials + 4096 + ((it + 1) & 1) * 2048;
  double* pap = partials + 8192;
  k_cg_spmv<<<nb, 256, 0, s>>>(F, nx, it, cp, cell_of, info, pg, ap, rz_prev, pap, sc);
  k_cg_update<<<nb, 256, 0, s>>>(F, it, cp, cell_of, info, r, ap, pg, xg, pap, rz_next, sc);
  k_cg_pupdate<<<nb, 256, 0, s>>>(F, it, cp, cell_of, info, r, pg, rz_next, sc);
}

}  // namespace fsg
