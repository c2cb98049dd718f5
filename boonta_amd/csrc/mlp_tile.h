// One Dense layer's contraction over a tile of 16 rows, shared by the launches
// that run several layers on the rows they own (mlp_chain.hip, step_towers.hip).
#pragma once
#include "common.h"

namespace {

template <int NB> struct VecOf;
template <> struct VecOf<1> { typedef float type; };
template <> struct VecOf<2> { typedef float type __attribute__((ext_vector_type(2))); };

template <int NB>
__device__ __forceinline__ void load_nb(const float* p, float (&v)[NB]) {
  const typename VecOf<NB>::type x = *reinterpret_cast<const typename VecOf<NB>::type*>(p);
  if constexpr (NB == 1) v[0] = x;
  else
#pragma unroll
    for (int j = 0; j < NB; ++j) v[j] = x[j];
}

template <int NB>
__device__ __forceinline__ void store_nb(float* p, const float (&v)[NB]) {
  typename VecOf<NB>::type x;
  if constexpr (NB == 1) x = v[0];
  else
#pragma unroll
    for (int j = 0; j < NB; ++j) x[j] = v[j];
  *reinterpret_cast<typename VecOf<NB>::type*>(p) = x;
}

// acc += A[16 rows][K] W[K][columns c ..]: chunk q of 16 reduction elements as
// four dependent MFMAs per block, lane group kq taking k = 16 q + 4 kq + s.
// LDSA: A from the tile row (K = 64 NB), else from global rows.  CH chunks are
// loaded at a time, the next ones ahead of this set's MFMAs.
// The kernels' row pitch is F, so a lane's loads take one 32-bit offset from a
// uniform base each.
template <int F, int NB, bool LDSA, bool VA, int CH>
__device__ __forceinline__ void act_contract(floatx4 (&acc)[NB], const float* arow, bool a_live, const float* W, int K,
                                             int kq, int c) {
  float a[2][CH][4], w[2][CH][4][NB];
  auto load = [&](int set, int k0) {
#pragma unroll
    for (int q = 0; q < CH; ++q) {
      const int kb = k0 + 16 * q + 4 * kq;
      if (LDSA || VA) {
        // (global rows: a pitch of at least K rounded up to 4)
        const floatx4 x = *reinterpret_cast<const floatx4*>(arow + (LDSA || (a_live && kb < K) ? kb : 0));
#pragma unroll
        for (int s = 0; s < 4; ++s) a[set][q][s] = LDSA || (a_live && kb + s < K) ? x[s] : 0.f;
      } else {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const bool in = a_live && kb + s < K;
          const float x = arow[in ? kb + s : 0];
          a[set][q][s] = in ? x : 0.f;
        }
      }
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if (LDSA) {
          load_nb<NB>(W + (k0 + 16 * q + s) * F + (uint32_t)(4 * kq * F + c), w[set][q][s]);
        } else {
          const bool in = kb + s < K;
          load_nb<NB>(W + (uint32_t)(min(kb + s, K - 1) * F + c), w[set][q][s]);
#pragma unroll
          for (int j = 0; j < NB; ++j) w[set][q][s][j] = in ? w[set][q][s][j] : 0.f;
        }
      }
    }
  };
  auto mma = [&](int set) {
#pragma unroll
    for (int q = 0; q < CH; ++q)
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int j = 0; j < NB; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[set][q][s], w[set][q][s][j], acc[j], 0, 0, 0);
  };
  load(0, 0);
#pragma unroll 1
  for (int k0 = 0; k0 < K; k0 += 32 * CH) {
    const bool second = k0 + 16 * CH < K;
    if (second) load(1, k0 + 16 * CH);
    __builtin_amdgcn_sched_barrier(0);
    mma(0);
    __builtin_amdgcn_sched_barrier(0);
    if (!second) break;
    if (k0 + 32 * CH < K) load(0, k0 + 32 * CH);
    __builtin_amdgcn_sched_barrier(0);
    mma(1);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// Brings this workgroup's share of n floats at p into the L2 of its XCD with
// copies into the wave's 1 KB of scratch LDS (256-float pieces; a remainder is
// left out): workgroups go to the 8 XCDs in turn, so blocks x, x + 8, .. of a
// tower share one L2.  Wait for the copies before the LDS is used or freed.
template <int NW>
__device__ __forceinline__ void warm_l2(const float* p, int n, float* scratch) {
  const int wave = threadIdx.x >> 6;
  const int share = blockIdx.x >> 3, shares = (gridDim.x + 7) >> 3;
  for (int c = share * NW + wave; c < n / 256; c += shares * NW)
    ppo::lds_copy16(p + 256 * c + 4 * (threadIdx.x & 63), scratch + 256 * wave);
}

}  // namespace
