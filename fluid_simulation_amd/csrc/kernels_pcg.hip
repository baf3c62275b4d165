// kernels_pcg.hip -- Jacobi-preconditioned CG with every iteration of a solve in one
// launch, optionally inside FP64 iterative refinement, and the set-up of the systems.
// Replaces Eigen::ConjugateGradient (include/FluidSolver.h:114, src/FluidSolver.cpp:81,
// 424-425).
//
// G blocks of 512 threads; block b owns the range [b*per, (b+1)*per) of the unknowns (the
// LIQUID cells in tile order, k_pcg_fill), a thread up to KPT of them (k = k0 + tid +
// j*512) whose x, r, z, p and Ap stay in its registers.  The search direction p of the
// block's unknowns and of their neighbours in other blocks (its halo) is in LDS.
//
// Iteration (Eigen's PCG, the same float operations per unknown as the kernels of
// kernels_cg.hip, sums in FP64):
//   A: p = z + beta p (own unknowns and halo alike); Ap; sum p.Ap
//      -- alpha = r.z / p.Ap
//   B: x += alpha p, r -= alpha Ap, z = M^-1 r; sums |r|^2, r.z
//      -- stop test, beta
// Only z crosses blocks: a block keeps p on its halo itself, from the halo's z.
//
// What bounds an iteration is the chain of device-coherent round trips between blocks
// (0.6 us between two blocks, 1.2-1.3 us for all of 23-123 blocks to have read a word of
// each), not arithmetic or bytes: 250,000 unknowns are 1 MB per vector, held in
// registers.  So nothing is ordered by waiting for stores, counting arrivals in a memory
// location and reading the data afterwards (three to four round trips per sum): every
// 32-bit value that crosses blocks travels in a 64-bit word together with a tag (the
// number of the sum it belongs to), and its readers poll the word itself until the tag
// is the one they wait for.  A sum then costs one store and one successful poll; the
// halo's z is polled by other waves of the block while the sums of phase B are, so it
// costs no trip of its own.  Refined form at 250,000 unknowns (1024^2): 15.0 -> 4.9 us
// per iteration against a counting grid barrier on 123 blocks of 1024 threads.
//
// A single block (k_pcg_one) exchanges nothing: its sums go through LDS with one
// workgroup barrier each.  1.0 us per iteration at 530 unknowns, 1.6 us at 3,800 (bound
// by VALU issue: 8 unknowns per thread), where three launches per iteration take 15-17.
//
// Ordering: words are cleared before the launch (k_pcg_clear) and tags grow, so a tag
// is never met before its value.  Sum e uses slot set e & 1: a block publishes sum e + 2
// only after it has read every block's sum e + 1, which each publishes after it has read
// all of sum e.  A block's z words of iteration k are rewritten in phase B of the next
// iteration, after the sum of phase A, which every block joins only after it has read
// its halo.  Waits are bounded: a wave that polls for too long raises an abort flag,
// every block leaves at its next sum, and the host reports it (or, for the plain form,
// solves again with the kernels of kernels_cg.hip).
//
// Refined form: FP64 iterative refinement around the FP32 solve -- r64 = b - A x64
// with the SpMV and its reduction in FP64, inner solve of A e = r64 to a relative
// tolerance, x64 += e -- until |b - A x64| < tol |b| in FP64.
#include <float.h>

#include <algorithm>

#include "fsg_common.h"
#include "fsg_device.h"
#include "fsg_kernels.h"

namespace fsg {

namespace {

constexpr int kPcgThreads = 512;
constexpr int kSlotWords = 4;              // 64-bit words per block and sum: 2 doubles

// Sum over the first 8 lanes of each 16-lane row, in lane 7 of the row.
__device__ __forceinline__ double row_sum8(double v) {
  v += dpp_f64<0x111, 0xF>(v);  // row_shr:1, 2, 4
  v += dpp_f64<0x112, 0xF>(v);
  v += dpp_f64<0x114, 0xF>(v);
  return v;
}
// Lane `from`'s value, in every lane.
__device__ __forceinline__ double lane_value(double v, int from) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), from),
                          __builtin_amdgcn_readlane(__double2loint(v), from));
}

// Halo entries of a block of `per` unknowns in tile order, at most: an unknown on the rim
// of its 32 x 32 tile has at most two neighbours in other tiles, and the first and the
// last tile of the range may be shared with another block (33 links each).
__host__ __device__ constexpr int pcg_halo_cap(int per) { return 2 * per + 66; }

__device__ __forceinline__ uint64_t tagged(uint32_t bits, uint32_t tag) {
  return ((uint64_t)tag << 32) | bits;
}
__device__ __forceinline__ uint32_t tag_of(uint64_t w) { return (uint32_t)(w >> 32); }

struct PcgNet {
  uint64_t* slots;  // [2][G][kSlotWords]
  uint64_t* z;      // one word per unknown: z of the unknowns in some block's halo
  unsigned* abort;
  unsigned spin_max;  // polls of a wait, at most
  uint32_t epoch;     // sums so far; the tag of the last one
};

struct PcgShared {
  double part[2][2][8];  // the block's wave sums, by epoch parity and value
  double tot[2][2][8];   // the grid's totals per polling wave; 0 past those
  int ok;
  int n_halo;
};

// Polls a thread's N words until each carries the tag (at(q): word q, null for none);
// false when the wait was abandoned.  All loads of a round are in flight together.
template <int N, typename At>
__device__ __forceinline__ bool poll(At&& at, uint32_t tag, uint64_t (&w)[N], const PcgNet& net) {
  for (unsigned spins = 0;; ++spins) {
    bool good = true;
#pragma unroll
    for (int q = 0; q < N; ++q) {
      const uint64_t* p = at(q);
      w[q] = p ? ld_dev(p) : tagged(0u, tag);
    }
#pragma unroll
    for (int q = 0; q < N; ++q) good &= tag_of(w[q]) == tag;
    if (good) return true;
    if (spins >= net.spin_max) {
      st_dev(net.abort, 1u);
      return false;
    }
    if ((spins & 255u) == 255u && ld_dev(net.abort)) return false;
  }
}

// The sums of NV values over the grid, in every thread (the same fixed order in every
// block); false when a wait was abandoned: the caller leaves the kernel without
// another sum.  `side` runs in the waves that do not poll the sums, while those do.
// DRAIN: the block's device-coherent stores are complete before its sum is published
// (a reader that has the sum may then read what they wrote).
// One slot per block, not one per wave (which would save the first barrier): beyond the
// two trips a sum costs what the blocks poll of each other (62 blocks: 5.5 us per
// iteration with a slot per block, 6.9 with one per wave; 245 blocks: 8.6 and 17).
template <int NV, bool ONE, bool DRAIN, typename Side>
__device__ __forceinline__ bool grid_sum(PcgNet& net, double (&v)[NV], PcgShared& sh,
                                         Side&& side) {
  static_assert(NV <= 2, "grid_sum: at most 2 values");
  constexpr int NW = kPcgThreads / 64;
  static_assert(NW == 8, "grid_sum: eight waves");
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint32_t e = ++net.epoch;
  const int par = e & 1;
  wave_sums(v);
  if (lane == 63)
#pragma unroll
    for (int q = 0; q < NV; ++q) sh.part[par][q][wave] = v[q];
  if (DRAIN && !ONE) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
  }
  __syncthreads();
  // value q's total over the waves in lane 16 q + 7
  auto total = [&](const double (&t)[2][8]) {
    return row_sum8(t[(lane >> 4) & (NV - 1)][lane & 7]);
  };
  if (!ONE) {
    const int G = gridDim.x, npoll = (G + 63) >> 6;
    uint64_t* set = net.slots + (size_t)par * G * kSlotWords;
    bool good = true;
    if (wave < npoll) {
      if (wave == 0) {
        const double s = total(sh.part[par]);
        if ((lane & 15) == 7 && (lane >> 4) < NV) {
          uint64_t* dst = set + (size_t)blockIdx.x * kSlotWords + 2 * (lane >> 4);
          st_dev(dst, tagged((uint32_t)__double2loint(s), e));
          st_dev(dst + 1, tagged((uint32_t)__double2hiint(s), e));
        }
      }
      const int b = wave * 64 + lane;
      uint64_t w[2 * NV];
      good = poll([&](int q) { return b < G ? set + (size_t)b * kSlotWords + q : nullptr; }, e, w,
                  net);
      double t[NV];
#pragma unroll
      for (int q = 0; q < NV; ++q)
        t[q] = __hiloint2double((int)(uint32_t)w[2 * q + 1], (int)(uint32_t)w[2 * q]);
      wave_sums(t);
      if (lane == 63)
#pragma unroll
        for (int q = 0; q < NV; ++q) sh.tot[par][q][wave] = t[q];
    } else {
      good = side(wave - npoll, NW - npoll);
    }
    if (!good) sh.ok = 0;
    __syncthreads();
    if (!sh.ok) return false;
  }
  // each wave adds the parts itself
  const double s = total(ONE ? sh.part[par] : sh.tot[par]);
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] = lane_value(s, 16 * q + 7);
  return true;
}

// ---------------------------------------------------------------- set-up
// The unknowns (LIQUID cells) in tile order: 32 x 32-cell tiles row by row, a tile's
// cells row by row.  A block's range of them is then a compact patch: its halo is the
// patch's rim (320 links for 4 full tiles), where a range of the row-major order has a
// full row of the grid above and below it (2044 at 1024 columns); the halo is read
// through device-coherent loads in every iteration (62 blocks: 5.5 -> 5.0 us each).
// ROWS: row-major order, a "tile" being 1024 cells in a row: the many-launch form's, whose
// kernels walk the unknowns through the cell grids and are bound by the lines that a wave
// touches (2048^2 box, 4.2 million unknowns: 67.9 us per iteration in rows, 74.1 in tiles;
// 3000^2, 4.6 million in no simple shape: 76.9 and 88.9).
template <bool ROWS>
__device__ __forceinline__ bool tile_cell(const Geom& g, int tile, int t, int& i, int& j) {
  if (ROWS) {
    const int c = tile * 1024 + t;
    j = c / g.nx;
    i = c - j * g.nx;
    return j < g.ny;
  }
  const int tiles_x = (g.nx + 31) >> 5;
  i = (tile % tiles_x) * 32 + (t & 31);
  j = (tile / tiles_x) * 32 + (t >> 5);
  return i < g.nx && j < g.ny;
}

// LIQUID cells per tile (thread t: the four cells 4 t .. 4 t + 3 of the tile).
template <bool ROWS>
__global__ void __launch_bounds__(256) k_pcg_count(Geom g, const uint8_t* __restrict__ label,
                                                   int* __restrict__ counts) {
  __shared__ int s_w[4];
  int n = 0;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    int i, j;
    if (tile_cell<ROWS>(g, blockIdx.x, 4 * threadIdx.x + e, i, j)) n += label[i + j * g.nx] == kLiquid;
  }
  for (int off = 32; off > 0; off >>= 1) n += __shfl_down(n, off, 64);
  if ((threadIdx.x & 63) == 0) s_w[threadIdx.x >> 6] = n;
  __syncthreads();
  if (threadIdx.x == 0) counts[blockIdx.x] = s_w[0] + s_w[1] + s_w[2] + s_w[3];
}

// Per unknown: its cell, neighbour info (src/FluidSolver.cpp:379-410) and right-hand side
// b = divVelX + divVelY (:413, MacGrid.h:98-111); per cell: its unknown's index (-1), and
// b (0) as fsg_get_rhs returns it.
// A block needs the number of unknowns in the tiles before its own.  With SCAN it sums
// their counts itself and the last block writes the total; else k_scan_counts has formed
// the offsets.  Up to kPcgScanTiles tiles (four loads per thread) that costs the kernel
// less than the scan's launch (3.5 us): with the splat's buckets likewise, four steps of
// 60 x 40 cells 663 -> 635 us.  More tiles: more passes, for a launch that a solve of that
// size does not notice.
constexpr int kPcgScanTiles = 1024;
template <bool SCAN, bool ROWS>
__global__ void __launch_bounds__(256) k_pcg_fill(Geom g, const uint8_t* __restrict__ label,
                                                  const int* __restrict__ offsets,
                                                  int* __restrict__ n_fluid,
                                                  int* __restrict__ index_of,
                                                  int* __restrict__ cell_of,
                                                  const float* __restrict__ uf,
                                                  const float* __restrict__ vf,
                                                  float* __restrict__ b, float* __restrict__ rhs,
                                                  uint8_t* __restrict__ info) {
  __shared__ int s_w[4], s_before[4];
  const int nx = g.nx, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int c[4], n = 0;
  bool in[4], liq[4];
  int ci[4], cj[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    in[e] = tile_cell<ROWS>(g, blockIdx.x, 4 * threadIdx.x + e, ci[e], cj[e]);
    c[e] = in[e] ? ci[e] + cj[e] * nx : 0;
    liq[e] = in[e] && label[c[e]] == kLiquid;
    n += liq[e];
  }
  int x = n;  // inclusive scan over the wave
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(x, o, 64);
    if (lane >= o) x += y;
  }
  if (lane == 63) s_w[wave] = x;
  if (SCAN) {
    int before = 0;
    for (int q = threadIdx.x; q < (int)blockIdx.x; q += 256) before += offsets[q];
    for (int o = 32; o > 0; o >>= 1) before += __shfl_down(before, o, 64);
    if (lane == 0) s_before[wave] = before;
  }
  __syncthreads();
  int k = SCAN ? s_before[0] + s_before[1] + s_before[2] + s_before[3] : offsets[blockIdx.x];
  if (SCAN && threadIdx.x == 0 && blockIdx.x == gridDim.x - 1)
    *n_fluid = k + s_w[0] + s_w[1] + s_w[2] + s_w[3];
  k += x - n;
  for (int w = 0; w < wave; ++w) k += s_w[w];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (!in[e]) continue;
    float bf = 0.f;
    int idx = -1;
    if (liq[e]) {
      const int i = ci[e], j = cj[e], q = c[e];
      // out-of-range neighbours count as SOLID (a SOLID border makes this moot)
      const uint8_t lxm = i > 0 ? label[q - 1] : kSolid;
      const uint8_t lxp = i < nx - 1 ? label[q + 1] : kSolid;
      const uint8_t lym = j > 0 ? label[q - nx] : kSolid;
      const uint8_t lyp = j < g.ny - 1 ? label[q + nx] : kSolid;
      const int bits = (lxm == kLiquid) | ((lxp == kLiquid) << 1) | ((lym == kLiquid) << 2) |
                       ((lyp == kLiquid) << 3);
      const int nns = (lxm != kSolid) + (lxp != kSolid) + (lym != kSolid) + (lyp != kSolid);
      const float uxp = i < nx - 1 ? uf[q + 1] : 0.f;
      const float vyp = j < g.ny - 1 ? vf[q + nx] : 0.f;
      const float dvx = div_x(uxp - uf[q], g);
      const float dvy = div_y(vyp - vf[q], g);
      bf = dvx + dvy;
      idx = k++;
      info[idx] = (uint8_t)(bits | (nns << 4));
      cell_of[idx] = q;
      b[idx] = bf;
    }
    index_of[c[e]] = idx;
    rhs[c[e]] = bf;
  }
}

__global__ void __launch_bounds__(256) k_pcg_clear(uint64_t* __restrict__ z, int64_t n,
                                                   uint64_t* __restrict__ slots, int n_slots,
                                                   unsigned* __restrict__ abort) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (t < n) z[t] = 0;
  if (t < n_slots) slots[t] = 0;
  if (t == 0) *abort = 0;
}

}  // namespace

namespace {

// The solve of F > 0 unknowns (F <= KPT NT gridDim.x).
template <int KPT, bool REFINED, bool ONE>
__device__ __forceinline__ void pcg_solve(const PersistentArgs& a, int F, float* lds,
                                          PcgShared& sh) {
  constexpr int NT = kPcgThreads;
  CgScalars* sc = a.sc;
  const int tid = threadIdx.x;
  const int G = ONE ? 1 : (int)gridDim.x;
  const int per = (F + G - 1) / G;
  const int k0 = ONE ? 0 : min(F, (int)blockIdx.x * per);
  const int k1 = min(F, k0 + per);
  // LDS: lds[0] = 0, p of the block's unknowns (room for KPT per thread) and of its halo
  // (pcg_halo_cap), then the halo's z and unknown indices
  constexpr int cap = KPT * NT;
  const int hcap = ONE ? 0 : pcg_halo_cap(per);
  float* lp = lds + 1;
  float* lph = lp + cap;
  float* lzh = lph + hcap;
  int* lhq = reinterpret_cast<int*>(lzh + hcap);
  const CgParams& cp = a.cp;
  if (tid < 32) {
    (&sh.part[0][0][0])[tid] = 0.0;
    (&sh.tot[0][0][0])[tid] = 0.0;
  }
  if (tid == 0) {
    sh.ok = 1;
    sh.n_halo = 0;
    lds[0] = 0.f;
  }
  __syncthreads();

  // unknown j of this thread: k = k0 + tid + j*NT, LDS slot k - k0.  nb: byte offsets in
  // LDS of its left, right, down and up neighbours' p.  A neighbour that is not an
  // unknown reads lds[0], so its term is + 0; a thread's j past the block's unknowns hold
  // zeros and read lds[0]: the iterations run without branches and selects, every LDS
  // read of a phase in flight at once.  A neighbour in another block gets a halo entry of
  // its own (a cell may have two), and the unknown itself is in that neighbour's block's
  // halo.
  int nb[KPT][4];
  float diag[KPT], invd[KPT];
  unsigned exported = 0;
  int nv = 0;  // valid unknowns: j = 0 .. nv - 1
#define FSG_VALID(j) ((j) < nv)
#define FSG_K(j) (k0 + tid + (j) * NT)
  char* const ldsb = reinterpret_cast<char*>(lds);
  auto ld_p = [&](int off) { return *reinterpret_cast<const float*>(ldsb + off); };
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    const int k = FSG_K(j);
    nb[j][0] = nb[j][1] = nb[j][2] = nb[j][3] = 0;
    diag[j] = invd[j] = 0.f;
    if (k >= k1) continue;
    nv = j + 1;
    const unsigned f = a.info[k];
    const int c = a.cell_of[k];
    diag[j] = sel5((int)(f >> 4) & 7, cp.diag_tab);
    invd[j] = sel5((int)(f >> 4) & 7, cp.invd_tab);
    const int d[4] = {-1, 1, -a.nx, a.nx};
    int q[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) q[t] = (f & (1u << t)) ? a.index_of[c + d[t]] : -1;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (q[t] < 0) continue;
      int slot = q[t] - k0;
      if (!ONE && (q[t] < k0 || q[t] >= k1)) {
        const int h = atomicAdd(&sh.n_halo, 1);  // < hcap (pcg_halo_cap)
        lhq[h] = q[t];
        slot = cap + h;
        exported |= 1u << j;
      }
      nb[j][t] = 4 * (slot + 1);
    }
  }
  __syncthreads();
  const int nh = ONE ? 0 : sh.n_halo;
  PcgNet net{a.slots, a.zx, a.abort, a.spin_max, 0u};
  auto idle = [](int, int) { return true; };
  // z of the halo, published for sum e: four words of a thread in flight at once
  auto stage_halo = [&](int w, int nw) {
    constexpr int U = 4;
    bool good = true;
    const int n = nw * 64;
    for (int t0 = w * 64 + (tid & 63); t0 < nh; t0 += U * n) {
      auto at = [&](int u) -> const uint64_t* {
        const int t = t0 + u * n;
        return t < nh ? net.z + lhq[t] : nullptr;
      };
      uint64_t v[U];
      good &= poll(at, net.epoch, v, net);
#pragma unroll
      for (int u = 0; u < U; ++u)
        if (t0 + u * n < nh) lzh[t0 + u * n] = __uint_as_float((uint32_t)v[u]);
    }
    return good;
  };

  // optional mean removal of b (fully Neumann systems)
  float mean = 0.f;
  if (cp.project_mean) {
    double v[1] = {0.0};
#pragma unroll
    for (int j = 0; j < KPT; ++j)
      if (FSG_VALID(j)) v[0] += (double)a.b[FSG_K(j)];
    if (!grid_sum<1, ONE, false>(net, v, sh, idle)) return;
    mean = (float)v[0] / (float)F;
  }

  float x[KPT], r[KPT], z[KPT], p[KPT], ap[KPT];
  int total_it = 0, total_spmv = 0, sweeps = 0;
  double err = 0.0, b2 = 0.0, res2 = 0.0, thr2 = 0.0;
  // Start: x0 = 0 (Eigen's solve()), or with warm_start the previous solution kept
  // in xg (zero at cells that were not LIQUID).  r0 = b - A x0 is formed in FP64
  // from xg, which nothing writes during the solve.
  {
    const double off = (double)cp.off;
    double v[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      r[j] = 0.f;
      if (!FSG_VALID(j)) continue;
      const int k = FSG_K(j);
      const double bk = (double)(cp.project_mean ? a.b[k] - mean : a.b[k]);
      double rk = bk;
      double x0 = 0.0;
      if (a.warm_start) {
        const int c = a.cell_of[k];
        x0 = (double)a.xg[c];
        double ax = (double)diag[j] * x0;
        if (nb[j][0]) ax += off * (double)a.xg[c - 1];
        if (nb[j][1]) ax += off * (double)a.xg[c + 1];
        if (nb[j][2]) ax += off * (double)a.xg[c - a.nx];
        if (nb[j][3]) ax += off * (double)a.xg[c + a.nx];
        rk = bk - ax;
      }
      if (REFINED) st_dev(a.x64 + k, x0);
      r[j] = (float)rk;
      v[0] += bk * bk;
      v[1] += rk * rk;
    }
    if (!grid_sum<2, ONE, REFINED>(net, v, sh, idle)) return;
    b2 = v[0];
    res2 = v[1];
    thr2 = a.outer_tol * a.outer_tol * b2;
  }

  const float tol = REFINED ? a.inner_tol : cp.tol;
  while (true) {
    if (REFINED && !(b2 > 0.0 && res2 >= thr2 && sweeps < a.max_outer)) break;
    // ------------- one FP32 Jacobi-PCG solve of A e = r (x0 = 0) -------------
    // z for the halo of the neighbouring blocks, tagged with the sum that follows
    auto publish_z = [&](int j) {
      if (!ONE && (exported & (1u << j)))
        st_dev(net.z + FSG_K(j), tagged(__float_as_uint(z[j]), net.epoch + 1));
    };
    double v2[2] = {0.0, 0.0};
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      x[j] = p[j] = 0.f;
      z[j] = invd[j] * r[j];
      publish_z(j);
      v2[0] += (double)(r[j] * r[j]);
      v2[1] += (double)(r[j] * z[j]);
    }
    for (int t = tid; t < nh; t += NT) lph[t] = 0.f;
    if (!grid_sum<2, ONE, false>(net, v2, sh, stage_halo)) return;
    const float rhs = (float)v2[0];
    int it = 0, spmv = 0;
    float rr = rhs;
    // Eigen's test |r| < tol |b|; the refined form's inner solves are relative to
    // their own right-hand side (the current residual)
    const float ref = REFINED ? rhs : (float)b2;
    float thr = tol * tol * ref;
    if (thr < FLT_MIN) thr = FLT_MIN;
    if (ref != 0.f && rhs != 0.f && !(rr < thr) && cp.max_iter >= a.min_iter) {
      float abs_new = (float)v2[1];
      float beta = 0.f;
      while (true) {
        // phase A: p on the window (beta = 0 and p = 0 at first), its halo from the halo's z
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
          p[j] = z[j] + beta * p[j];
          lp[tid + j * NT] = p[j];
        }
        for (int t = tid; t < nh; t += NT) lph[t] = lzh[t] + beta * lph[t];
        __syncthreads();
        double v1[1] = {0.0};
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
          const float nl = ld_p(nb[j][0]), nr = ld_p(nb[j][1]);
          const float nd = ld_p(nb[j][2]), nu = ld_p(nb[j][3]);
          float acc = diag[j] * p[j];
          acc += cp.off * nl;
          acc += cp.off * nr;
          acc += cp.off * nd;
          acc += cp.off * nu;
          ap[j] = acc;
          v1[0] += (double)(p[j] * acc);
        }
        if (!grid_sum<1, ONE, false>(net, v1, sh, idle)) return;
        ++spmv;
        const float alpha = abs_new / (float)v1[0];
        // phase B
        v2[0] = 0.0;
        v2[1] = 0.0;
#pragma unroll
        for (int j = 0; j < KPT; ++j) {
          r[j] = r[j] - alpha * ap[j];
          z[j] = invd[j] * r[j];
          publish_z(j);
          x[j] = x[j] + alpha * p[j];
          v2[0] += (double)(r[j] * r[j]);
          v2[1] += (double)(r[j] * z[j]);
        }
        if (!grid_sum<2, ONE, false>(net, v2, sh, stage_halo)) return;
        rr = (float)v2[0];
        if (rr < thr) break;
        const float abs_old = abs_new;
        abs_new = (float)v2[1];
        beta = abs_new / abs_old;
        ++it;
        if (it >= cp.max_iter) break;
      }
    }
    total_it += it;
    total_spmv += spmv;
    err = ref != 0.f ? sqrt((double)rr / (double)ref) : 0.0;
    if (!REFINED) break;
    // ------------- FP64 refinement: x64 += e; r = b - A x64 -------------
    ++sweeps;
#pragma unroll
    for (int j = 0; j < KPT; ++j)
      if (FSG_VALID(j)) {
        const int k = FSG_K(j);
        st_dev(a.x64 + k, ld_dev(a.x64 + k) + (double)x[j]);
      }
    double w[1] = {0.0};
    if (!grid_sum<1, ONE, true>(net, w, sh, idle)) return;
    const double off = (double)cp.off;
    w[0] = 0.0;
#pragma unroll
    for (int j = 0; j < KPT; ++j) {
      if (!FSG_VALID(j)) {
        r[j] = 0.f;
        continue;
      }
      __builtin_amdgcn_sched_barrier(0);  // one unknown's loads at a time: no spills
      const int k = FSG_K(j);
      double ax = (double)diag[j] * ld_dev(a.x64 + k);
#pragma unroll
      for (int t = 0; t < 4; ++t)
        if (nb[j][t]) {
          const int slot = nb[j][t] / 4 - 1;
          ax += off * ld_dev(a.x64 + (slot < cap ? k0 + slot : lhq[slot - cap]));
        }
      const double bk = (double)(cp.project_mean ? a.b[k] - mean : a.b[k]);
      const double rk = bk - ax;
      r[j] = (float)rk;
      w[0] += rk * rk;
    }
    if (!grid_sum<1, ONE, false>(net, w, sh, idle)) return;
    res2 = w[0];
    total_spmv += 1;
  }
  // solution into grid layout for the gradient update
#pragma unroll
  for (int j = 0; j < KPT; ++j) {
    if (!FSG_VALID(j)) continue;
    const int k = FSG_K(j);
    const int c = a.cell_of[k];
    float xk;
    if (b2 == 0.0) xk = 0.f;  // Eigen: |b| = 0 gives x = 0
    else if (REFINED) xk = (float)ld_dev(a.x64 + k);
    else xk = a.warm_start ? a.xg[c] + x[j] : x[j];
    a.xg[c] = xk;
  }
#undef FSG_VALID
#undef FSG_K
  if (REFINED) err = b2 > 0.0 ? sqrt(res2 / b2) : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    sc->iter = total_it;
    sc->spmv = total_spmv;
    sc->err = cp.max_iter >= a.min_iter ? err : 0.0;
    sc->b64_norm2 = b2;
    sc->res64_norm2 = res2;
    sc->refine_sweeps = sweeps;
    sc->total_unknown_iters += (unsigned long long)F * (unsigned long long)total_spmv;
    sc->total_solves += 1;
  }
}

// Many blocks, KPT unknowns per thread (F > 0).
template <int KPT, bool REFINED>
__global__ void __launch_bounds__(kPcgThreads) k_pcg(PersistentArgs a) {
  extern __shared__ float lds[];
  __shared__ PcgShared sh;
  pcg_solve<KPT, REFINED, false>(a, *a.n_fluid, lds, sh);
}

// One block.  The launch may be sized by a bound of F, so the unknowns per thread (up to
// KMAX) are chosen here: an iteration costs instructions for each of them, used or not.
// 512 threads: 256 take 1.95 us per iteration at 3,800 unknowns against 1.59, and the
// same at 530.
template <int KMAX, bool REFINED>
__global__ void __launch_bounds__(kPcgThreads) k_pcg_one(PersistentArgs a) {
  constexpr int NT = kPcgThreads;
  extern __shared__ float lds[];
  __shared__ PcgShared sh;
  const int F = *a.n_fluid;
  if (threadIdx.x == 0) {
    *a.abort = 0;  // (more blocks: k_pcg_clear)
    if (F == 0) {
      a.sc->iter = a.sc->spmv = a.sc->refine_sweeps = 0;
      a.sc->err = 0.0;
    }
  }
  if (F == 0) return;
  if (F <= NT) pcg_solve<1, REFINED, true>(a, F, lds, sh);
  else if (F <= 2 * NT) pcg_solve<2, REFINED, true>(a, F, lds, sh);
  else if (F <= 4 * NT) pcg_solve<4, REFINED, true>(a, F, lds, sh);
  else if (F <= 8 * NT) pcg_solve<8, REFINED, true>(a, F, lds, sh);
  else if constexpr (KMAX >= 16) pcg_solve<16, REFINED, true>(a, F, lds, sh);
}

}  // namespace

int pcg_tiles(const Geom& g) { return ((g.nx + 31) / 32) * ((g.ny + 31) / 32); }
void launch_pcg_count(hipStream_t s, const Geom& g, const uint8_t* label, int* counts) {
  k_pcg_count<false><<<pcg_tiles(g), 256, 0, s>>>(g, label, counts);
}
void launch_pcg_fill(hipStream_t s, const Geom& g, const uint8_t* label, const int* counts,
                     int* offsets, int* n_fluid, int* index_of, int* cell_of, const float* uf,
                     const float* vf, float* b, float* rhs, uint8_t* info, bool scanned) {
  const int nb = pcg_tiles(g);
  if (nb <= kPcgScanTiles && !scanned) {
    k_pcg_fill<true, false><<<nb, 256, 0, s>>>(g, label, counts, n_fluid, index_of, cell_of, uf,
                                               vf, b, rhs, info);
    return;
  }
  if (!scanned) launch_scan_counts(s, nb, counts, offsets, n_fluid);
  k_pcg_fill<false, false><<<nb, 256, 0, s>>>(g, label, offsets, n_fluid, index_of, cell_of, uf,
                                              vf, b, rhs, info);
}
void launch_pcg_rows(hipStream_t s, const Geom& g, const uint8_t* label, int* counts, int* offsets,
                     int* n_fluid, int* index_of, int* cell_of, const float* uf, const float* vf,
                     float* b, float* rhs, uint8_t* info) {
  const int nb = (g.nx * g.ny + 1023) / 1024;  // at most pcg_tiles(g)
  k_pcg_count<true><<<nb, 256, 0, s>>>(g, label, counts);
  launch_scan_counts(s, nb, counts, offsets, n_fluid);
  k_pcg_fill<false, true><<<nb, 256, 0, s>>>(g, label, offsets, n_fluid, index_of, cell_of, uf, vf,
                                             b, rhs, info);
}

size_t pcg_row_window(int F, int grid, int nx) {
  const int per = (F + grid - 1) / grid;
  return (size_t)3 * (per + 2 * nx) * sizeof(float);
}
size_t pcg_lds_bytes(int F, int grid, int kpt) {
  if (grid == 1) {
    int cap = kPcgThreads;  // the kernel's unknowns per thread x threads for any number up to F
    while (cap < F) cap *= 2;
    return (size_t)(cap + 1) * sizeof(float);
  }
  return (size_t)(1 + 1024 * kpt + 3 * pcg_halo_cap((F + grid - 1) / grid)) * sizeof(float);
}
size_t pcg_slot_words(int grid) { return (size_t)2 * grid * kSlotWords; }

namespace {
template <int KPT>
const void* pcg_kernel(bool refined) {
  return refined ? (const void*)k_pcg<KPT, true> : (const void*)k_pcg<KPT, false>;
}
}  // namespace

hipError_t launch_pcg(hipStream_t s, const PersistentArgs& a, int grid, int kpt) {
  void* args[] = {(void*)&a};
  const bool ref = a.refined != 0;
  const void* f = nullptr;
  const size_t lds = pcg_lds_bytes(a.F_actual, grid, kpt);
  if (grid == 1) {
    if (a.F_actual > (ref ? kPcgOneRefined : kPcgOneUnknowns)) return hipErrorInvalidValue;
    f = ref ? (const void*)k_pcg_one<8, true> : (const void*)k_pcg_one<16, false>;
    return hipLaunchKernel(f, dim3(1), dim3(kPcgThreads), args, lds, s);
  }
  const int per = (a.F_actual + grid - 1) / grid;
  if (per > 1024 * kpt) return hipErrorInvalidValue;
  const int n_slots = (int)pcg_slot_words(grid);
  const int64_t n = std::max<int64_t>(a.F_actual, n_slots);
  k_pcg_clear<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(a.zx, a.F_actual, a.slots, n_slots,
                                                          a.abort);
  switch (kpt) {
    case 1: f = pcg_kernel<2>(ref); break;
    case 2: f = pcg_kernel<4>(ref); break;
    case 4: f = pcg_kernel<8>(ref); break;
    default: return hipErrorInvalidValue;
  }
  return hipLaunchCooperativeKernel(f, dim3(grid), dim3(kPcgThreads), args, lds, s);
}

hipError_t pcg_set_lds_limit(size_t max_bytes) {
  for (bool ref : {false, true})
    for (const void* f : {pcg_kernel<2>(ref), pcg_kernel<4>(ref), pcg_kernel<8>(ref)}) {
      hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize,
                                         (int)max_bytes);
      if (e != hipSuccess) return e;
    }
  return hipSuccess;
}

}  // namespace fsg
