// fsg_common.h -- reduction and device-coherent memory helpers shared by the
// pressure-solver kernels.
#pragma once
#include <hip/hip_runtime.h>

namespace fsg {

// DPP move of a double; lanes without a source take 0.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, ROWS, 0xF, false);
  return __hiloint2double(hi, lo);
}
// Sums over the wave, in lane 63, the values' steps interleaved (register moves only: a
// shuffle tree of doubles costs 12 LDS-latency exchanges).
template <int CTRL, int ROWS, int NV>
__device__ __forceinline__ void dpp_step(double (&v)[NV]) {
  double t[NV];
#pragma unroll
  for (int q = 0; q < NV; ++q) t[q] = dpp_f64<CTRL, ROWS>(v[q]);
#pragma unroll
  for (int q = 0; q < NV; ++q) v[q] += t[q];
}
template <int NV>
__device__ __forceinline__ void wave_sums(double (&v)[NV]) {
  dpp_step<0x111, 0xF>(v);
  dpp_step<0x112, 0xF>(v);
  dpp_step<0x114, 0xF>(v);
  dpp_step<0x118, 0xF>(v);
  dpp_step<0x142, 0xA>(v);  // row_bcast:15 into rows 1 and 3
  dpp_step<0x143, 0xC>(v);  // row_bcast:31 into rows 2 and 3
}
// Sum NV doubles over a block of NT threads; the result is returned in every
// thread.  The order is fixed (the lanes' register moves, then waves in order), so equal
// inputs give bit-identical sums in every block and every launch.  A tree of shuffles in
// place of the moves keeps the LDS pipe of a CU with 32 waves busy for 1.3 us.
// sm: NV * (NT / 64) doubles of LDS.
template <int NV, int NT>
__device__ __forceinline__ void block_sum(double (&v)[NV], double* sm) {
  constexpr int NW = NT / 64;
  wave_sums(v);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 63)
#pragma unroll
    for (int q = 0; q < NV; ++q) sm[q * NW + wave] = v[q];
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; ++q) {
    double s = 0.0;
#pragma unroll
    for (int w = 0; w < NW; ++w) s += sm[q * NW + w];
    v[q] = s;
  }
}

// t[n] for n in 0..4 without dynamic indexing (keeps the table in registers).
__device__ __forceinline__ float sel5(int n, const float (&t)[5]) {
  float r = t[0];
  r = n == 1 ? t[1] : r;
  r = n == 2 ? t[2] : r;
  r = n == 3 ? t[3] : r;
  r = n == 4 ? t[4] : r;
  return r;
}

// Agent-scope relaxed atomic load / store: served at the device coherence point,
// so values written by blocks on other XCDs are seen without cache maintenance.
template <typename T>
__device__ __forceinline__ T ld_dev(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <typename T>
__device__ __forceinline__ void st_dev(T* p, T v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace fsg
