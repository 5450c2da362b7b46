// Conversion between the callers' k vectors one after another (element
// c*dim + j) and the state-major block (element j*k + c), shared by the TPQ and
// LOBPCG drivers (included by their kernel files).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

// Bound by memory: a tile of BL_TILE amplitudes (BL_TILE / K states) passes
// through LDS, so both sides are read and written in runs of at least 1 KB
// (K <= 16); one element per thread with a 64-bit division each ran at
// 0.9 TB/s (2.50 ms to load and 1.89 ms to store 16 vectors of 2^22 states; now
// 0.41 and 0.40 ms, 5.3 TB/s).
#define BL_TPB 256
#define BL_TILE 1024

// scale of column c: sp[c] where sp is given, else sv.f[c]
struct BlScale {
  double f[16];
};

// TO_BLOCK: block[j*K + c] = vecs[c*dim + j]; else vecs[c*dim + j] = scale_c block[j*K + c]
template <int K, bool TO_BLOCK>
__global__ __launch_bounds__(BL_TPB) void k_block_layout(const double2 *__restrict__ from, double2 *__restrict__ to,
                                                         uint64_t dim, const double *sp, BlScale sv) {
  constexpr int S = BL_TILE / K;  // states per tile
  __shared__ double2 t[K * (S + 1)];
  for (uint64_t j0 = (uint64_t)blockIdx.x * S; j0 < dim; j0 += (uint64_t)gridDim.x * S) {
#pragma unroll
    for (int i = threadIdx.x; i < BL_TILE; i += BL_TPB) {
      const int c = TO_BLOCK ? i / S : i % K, j = TO_BLOCK ? i % S : i / K;
      if (j0 + j < dim) t[c * (S + 1) + j] = TO_BLOCK ? from[(uint64_t)c * dim + j0 + j] : from[j0 * K + i];
    }
    __syncthreads();
#pragma unroll
    for (int i = threadIdx.x; i < BL_TILE; i += BL_TPB) {
      const int c = TO_BLOCK ? i % K : i / S, j = TO_BLOCK ? i / K : i % S;
      if (j0 + j < dim) {
        const double2 a = t[c * (S + 1) + j];
        if (TO_BLOCK) {
          to[j0 * K + i] = a;
        } else {
          const double f = sp ? sp[c] : sv.f[c];
          to[(uint64_t)c * dim + j0 + j] = make_double2(f * a.x, f * a.y);
        }
      }
    }
    __syncthreads();
  }
}

// sp (device, may be null) or sv scales the columns on the way to vectors; the caller checks the launch
template <bool TO_BLOCK>
static inline void block_layout(const double2 *from, double2 *to, uint64_t dim, int k, const double *sp, BlScale sv,
                                hipStream_t st) {
  const uint64_t tiles = (dim * (uint64_t)k + BL_TILE - 1) / BL_TILE;
  const dim3 g((unsigned)(tiles < 8192 ? (tiles ? tiles : 1) : 8192));
  switch (k) {
    case 1: hipLaunchKernelGGL((k_block_layout<1, TO_BLOCK>), g, dim3(BL_TPB), 0, st, from, to, dim, sp, sv); break;
    case 2: hipLaunchKernelGGL((k_block_layout<2, TO_BLOCK>), g, dim3(BL_TPB), 0, st, from, to, dim, sp, sv); break;
    case 4: hipLaunchKernelGGL((k_block_layout<4, TO_BLOCK>), g, dim3(BL_TPB), 0, st, from, to, dim, sp, sv); break;
    case 8: hipLaunchKernelGGL((k_block_layout<8, TO_BLOCK>), g, dim3(BL_TPB), 0, st, from, to, dim, sp, sv); break;
    case 16: hipLaunchKernelGGL((k_block_layout<16, TO_BLOCK>), g, dim3(BL_TPB), 0, st, from, to, dim, sp, sv); break;
  }
}
