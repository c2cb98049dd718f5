// Linear-recurrence scan h_t = a_t * h_{t-1} + b_t over [batch, steps, features]
// and its vector-Jacobian product, the kernels behind boonta's SSM / MinGRU
// torsos (boonta/networks/kernels/scan.py:13-88: `scan` with its custom VJP;
// the SSM block calls it at networks/blocks/ssm.py:31-55).
//
// Forward:  h_t = a_t h_{t-1} + b_t, h_{-1} = init, accumulated in float32 and
//           stored in the operands' type (float32 or bf16 storage).
// Backward (cotangent g of h):
//           db_t = g_t + a_{t+1} db_{t+1}   (db_{steps-1} = g_{steps-1})
//           da_t = db_t h_{t-1}             (h_{-1} = init)
//           dinit = db_0 a_0
//           with db accumulated in float32 and stored in the operands' type;
//           for bf16 storage da and dinit multiply the stored (rounded) db and
//           are rounded again, as the reference's bf16 array arithmetic does.
//
// The SSM block's episode resets (networks/blocks/ssm.py:45-48) can be folded
// into the same launches (ppo_ssm_scan_*): where done[n, t], the step's decay
// becomes 0 and its input b + a r (r the carry a reset restarts from, zeros
// by default), and the backward carries the reset's own chain rule (da = r db
// there, and no decay into the step).
//
// Layout and parallelism: element (n, t, f) at (n * steps + t) * features + f.
// Each lane owns VW = 4 consecutive features of one sequence where the rows
// allow (one 16-byte float32 or 8-byte bf16 access), so every step reads one
// coalesced row.  The time axis is cut into chunks of a few steps, one wave
// each: a wave loads its chunk into registers, folds it into the affine map
// (A, B) of h_end = A h_start + B, the waves exchange the maps through LDS, and
// each composes the maps before it (in time order for the forward, in reverse
// for the backward) to write its chunk's outputs from the exact carry.
// Sequences of up to 128 steps are one such tile of 16 chunks, longer ones run
// tile after tile.  A chunk's decay is the product of its steps' and can leave
// float32's range where no state does: a tile of a long sequence whose composed
// state is not finite is stepped through instead; one tile alone (9 to 128
// steps) is not.  Below the range the product rounds to the subnormals' grid, at
// most 2^-149 of the state entering the chunk.
#include "split_f32.h"

#include <algorithm>

namespace {

constexpr int MAX_CHUNKS = 16;

enum ScanDtype { SCAN_F32 = 0, SCAN_BF16 = 1 };

__device__ __forceinline__ void load_vec(const float* p, int64_t i, float (&v)[1]) { v[0] = p[i]; }
__device__ __forceinline__ void load_vec(const float* p, int64_t i, float (&v)[4]) {
  const floatx4 x = *reinterpret_cast<const floatx4*>(p + i);
  v[0] = x[0]; v[1] = x[1]; v[2] = x[2]; v[3] = x[3];
}
__device__ __forceinline__ float bf16_to_f32(uint16_t u) { return __uint_as_float((uint32_t)u << 16); }
__device__ __forceinline__ void load_vec(const uint16_t* p, int64_t i, float (&v)[1]) { v[0] = bf16_to_f32(p[i]); }
__device__ __forceinline__ void load_vec(const uint16_t* p, int64_t i, float (&v)[4]) {
  const uint2 x = *reinterpret_cast<const uint2*>(p + i);
  v[0] = __uint_as_float(x.x << 16); v[1] = __uint_as_float(x.x & 0xffff0000u);
  v[2] = __uint_as_float(x.y << 16); v[3] = __uint_as_float(x.y & 0xffff0000u);
}

__device__ __forceinline__ void store_vec(float* p, int64_t i, const float (&v)[1]) { p[i] = v[0]; }
__device__ __forceinline__ void store_vec(float* p, int64_t i, const float (&v)[4]) {
  floatx4 x;
  x[0] = v[0]; x[1] = v[1]; x[2] = v[2]; x[3] = v[3];
  *reinterpret_cast<floatx4*>(p + i) = x;
}
// (rounded by v_cvt_pk_bf16_f32, two values an instruction: to nearest even,
// as ppo::bf16_bits rounds in nine)
__device__ __forceinline__ void store_vec(uint16_t* p, int64_t i, const float (&v)[1]) {
  p[i] = (uint16_t)ppo::pack_bf16(v[0], v[0]);
}
__device__ __forceinline__ void store_vec(uint16_t* p, int64_t i, const float (&v)[4]) {
  uint2 x;
  x.x = ppo::pack_bf16(v[0], v[1]);
  x.y = ppo::pack_bf16(v[2], v[3]);
  *reinterpret_cast<uint2*>(p + i) = x;
}
// The value a stored element of type S holds (identity for float32).
__device__ __forceinline__ float stored(float x, const float*) { return x; }
__device__ __forceinline__ float stored(float x, const uint16_t*) {
  return __uint_as_float(ppo::pack_bf16(x, x) << 16);
}

struct ScanArgs {
  const void* a;
  const void* b;     // forward: b; backward: the cotangent of h
  const void* h;     // backward: the forward's output
  const void* init;
  void* out;         // forward: h; backward: db
  void* da;
  void* dinit;
  int steps, F;
  const uint8_t* done;  // [batch, steps] episode starts of the SSM block, or null
  const void* reset;    // [batch, features] carry a done step restarts from, or null (zeros)
};

// The SSM block's reset (networks/blocks/ssm.py:45-48) applied to step t's
// operands: where done, b' = b + a * r and a' = 0, in the storage type's
// arithmetic (each product and sum rounded for bf16).
__device__ __forceinline__ bool is_done(const ScanArgs& p, int64_t n, int t) {
  return p.done && p.done[n * p.steps + t];
}

template <typename S, int VW>
__device__ __forceinline__ void load_reset(const ScanArgs& p, int64_t n, int f0, float (&rv)[VW]) {
  if (p.reset) {
    load_vec(static_cast<const S*>(p.reset), n * (int64_t)p.F + f0, rv);
  } else {
#pragma unroll
    for (int k = 0; k < VW; ++k) rv[k] = 0.f;
  }
}

template <typename S, int VW>
__device__ __forceinline__ void load_ab(const ScanArgs& p, const S* a, const S* b, int64_t base, int64_t n, int t,
                                        int f0, float (&av)[VW], float (&bv)[VW]) {
  load_vec(a, base + (int64_t)t * p.F, av);
  load_vec(b, base + (int64_t)t * p.F, bv);
  if (is_done(p, n, t)) {
    float rv[VW];
    load_reset<S, VW>(p, n, f0, rv);
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      bv[k] = stored(bv[k] + stored(av[k] * rv[k], a), a);
      av[k] = 0.f;
    }
  }
}

// alpha_t = a'_{t+1}, the (reset) decay of the next step; 0 past the last step
template <typename S, int VW>
__device__ __forceinline__ void load_alpha(const ScanArgs& p, const S* a, int64_t base, int64_t n, int t,
                                           float (&al)[VW]) {
  if (t + 1 < p.steps && !is_done(p, n, t + 1)) {
    load_vec(a, base + (int64_t)(t + 1) * p.F, al);
  } else {
#pragma unroll
    for (int k = 0; k < VW; ++k) al[k] = 0.f;
  }
}

// da_t: db'_t h_{t-1} where step t was not reset; r db'_t where it was (the
// cotangent of a through b' = b + a r; a' = 0 passes none)
template <typename S, int VW>
__device__ __forceinline__ void reset_da(const ScanArgs& p, const S* a, int64_t n, int t, int f0,
                                         const float (&dv)[VW], float (&dav)[VW]) {
  if (is_done(p, n, t)) {
    float rv[VW];
    load_reset<S, VW>(p, n, f0, rv);
#pragma unroll
    for (int k = 0; k < VW; ++k) dav[k] = stored(rv[k] * dv[k], a);
  }
}

// Register-resident chunks: each wave loads its chunk of at most RL steps once
// (all loads issued before the first multiply-add), folds it into its affine
// map, exchanges the maps through LDS, and writes its outputs from the same
// registers, so chunking costs no second read of the operands.  Steps past
// the chunk's end hold the identity map (a = 1, b = 0 forward; alpha = 1,
// g = 0 backward).
constexpr int RL = 8;

template <typename S, int VW>
__global__ void __launch_bounds__(64 * MAX_CHUNKS) scan_fwd_reg_kernel(ScanArgs p) {
  extern __shared__ float smem[];
  float* sA = smem;
  float* sB = smem + (blockDim.x >> 6) * 64 * VW;
  const S* a = static_cast<const S*>(p.a);
  const S* b = static_cast<const S*>(p.b);
  const S* init = static_cast<const S*>(p.init);
  S* out = static_cast<S*>(p.out);
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6, C = blockDim.x >> 6;
  const int f0 = (blockIdx.x * 64 + lane) * VW;
  const bool ok = f0 < p.F;
  const int64_t n = blockIdx.y;
  const int t0 = c * RL, t1 = min(p.steps, t0 + RL);
  const int64_t base = n * (int64_t)p.steps * p.F + f0;
  float av[RL][VW], bv[RL][VW], h[VW];
#pragma unroll
  for (int i = 0; i < RL; ++i) {
    if (ok && t0 + i < t1) {
      load_ab<S, VW>(p, a, b, base, n, t0 + i, f0, av[i], bv[i]);
    } else {
#pragma unroll
      for (int k = 0; k < VW; ++k) { av[i][k] = 1.f; bv[i][k] = 0.f; }
    }
  }
  if (ok) {
    load_vec(init, n * (int64_t)p.F + f0, h);
  } else {
#pragma unroll
    for (int k = 0; k < VW; ++k) h[k] = 0.f;
  }
  if (C > 1) {
    float A[VW], B[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) { A[k] = 1.f; B[k] = 0.f; }
#pragma unroll
    for (int i = 0; i < RL; ++i) {
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        A[k] = av[i][k] * A[k];
        B[k] = av[i][k] * B[k] + bv[i][k];
      }
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      sA[(c * 64 + lane) * VW + k] = A[k];
      sB[(c * 64 + lane) * VW + k] = B[k];
    }
    __syncthreads();
    for (int cc = 0; cc < c; ++cc) {
#pragma unroll
      for (int k = 0; k < VW; ++k) h[k] = sA[(cc * 64 + lane) * VW + k] * h[k] + sB[(cc * 64 + lane) * VW + k];
    }
  }
  if (!ok) return;
#pragma unroll
  for (int i = 0; i < RL; ++i) {
#pragma unroll
    for (int k = 0; k < VW; ++k) h[k] = av[i][k] * h[k] + bv[i][k];
    if (t0 + i < t1) store_vec(out, base + (int64_t)(t0 + i) * p.F, h);
  }
}

template <typename S, int VW>
__global__ void __launch_bounds__(64 * MAX_CHUNKS) scan_bwd_reg_kernel(ScanArgs p) {
  extern __shared__ float smem[];
  float* sA = smem;
  float* sB = smem + (blockDim.x >> 6) * 64 * VW;
  const S* a = static_cast<const S*>(p.a);
  const S* g = static_cast<const S*>(p.b);
  const S* hs = static_cast<const S*>(p.h);
  const S* init = static_cast<const S*>(p.init);
  S* db = static_cast<S*>(p.out);
  S* da = static_cast<S*>(p.da);
  S* dinit = static_cast<S*>(p.dinit);
  const int lane = threadIdx.x & 63, c = threadIdx.x >> 6, C = blockDim.x >> 6;
  const int f0 = (blockIdx.x * 64 + lane) * VW;
  const bool ok = f0 < p.F;
  const int64_t n = blockIdx.y;
  const int t0 = c * RL, t1 = min(p.steps, t0 + RL);
  const int64_t base = n * (int64_t)p.steps * p.F + f0;
  // al[i] = a_{t+1} (0 past the last step), gv[i] = g_t, hp[i] = h_{t-1} (init at t = 0)
  float al[RL][VW], gv[RL][VW], hp[RL][VW];
#pragma unroll
  for (int i = 0; i < RL; ++i) {
    const int t = t0 + i;
    if (ok && t < t1) {
      load_alpha<S, VW>(p, a, base, n, t, al[i]);
      load_vec(g, base + (int64_t)t * p.F, gv[i]);
      if (t > 0) {
        load_vec(hs, base + (int64_t)(t - 1) * p.F, hp[i]);
      } else {
        load_vec(init, n * (int64_t)p.F + f0, hp[i]);
      }
    } else {
#pragma unroll
      for (int k = 0; k < VW; ++k) { al[i][k] = 1.f; gv[i][k] = 0.f; hp[i][k] = 0.f; }
    }
  }
  float d[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) d[k] = 0.f;
  if (C > 1) {
    float P[VW], Q[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) { P[k] = 1.f; Q[k] = 0.f; }
#pragma unroll
    for (int i = RL - 1; i >= 0; --i) {
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        P[k] = al[i][k] * P[k];
        Q[k] = al[i][k] * Q[k] + gv[i][k];
      }
    }
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      sA[(c * 64 + lane) * VW + k] = P[k];
      sB[(c * 64 + lane) * VW + k] = Q[k];
    }
    __syncthreads();
    for (int cc = C - 1; cc > c; --cc) {
#pragma unroll
      for (int k = 0; k < VW; ++k) d[k] = sA[(cc * 64 + lane) * VW + k] * d[k] + sB[(cc * 64 + lane) * VW + k];
    }
  }
  if (!ok) return;
#pragma unroll
  for (int i = RL - 1; i >= 0; --i) {
    const int t = t0 + i;
    float dv[VW], dav[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      d[k] = al[i][k] * d[k] + gv[i][k];
      dv[k] = stored(d[k], db);
      dav[k] = dv[k] * hp[i][k];
    }
    if (t < t1) {
      reset_da<S, VW>(p, a, n, t, f0, dv, dav);
      store_vec(db, base + (int64_t)t * p.F, d);
      store_vec(da, base + (int64_t)t * p.F, dav);
      if (t == 0) {
        float a0[VW], di[VW];
        load_vec(a, base, a0);
        if (is_done(p, n, 0)) {
#pragma unroll
          for (int k = 0; k < VW; ++k) a0[k] = 0.f;
        }
#pragma unroll
        for (int k = 0; k < VW; ++k) di[k] = dv[k] * a0[k];
        store_vec(dinit, n * (int64_t)p.F + f0, di);
      }
    }
  }
}

// Long sequences: the workgroup's waves take the register-resident chunks of
// one tile of steps after another, the state entering a tile carried in
// registers from the tile before it, and the next tile's loads issued before
// this tile's maps are exchanged.  Every operand is read once.  What bounds it
// is HBM: [128, 1000, 512] bf16 with resets, forward 153 -> 78 us, backward 296
// -> 130 us, 5.0 TB/s (chunks that re-read their operands before).  A
// chunk holds 8 steps of operands and the next 8 in storage type, so a
// workgroup has 8 waves (16 of them spilled registers).
constexpr int TILE_WAVES = 8;

template <typename S, int VW> struct Raw;
template <> struct Raw<float, 4> { floatx4 v; };
template <> struct Raw<float, 1> { float v; };
template <> struct Raw<uint16_t, 4> { uint2 v; };
template <> struct Raw<uint16_t, 1> { uint16_t v; };

template <typename S, int VW>
__device__ __forceinline__ Raw<S, VW> load_raw(const S* p, int64_t i) {
  return Raw<S, VW>{*reinterpret_cast<const decltype(Raw<S, VW>::v)*>(p + i)};
}
__device__ __forceinline__ void expand(const Raw<float, 4>& r, float (&v)[4]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) v[k] = r.v[k];
}
__device__ __forceinline__ void expand(const Raw<float, 1>& r, float (&v)[1]) { v[0] = r.v; }
__device__ __forceinline__ void expand(const Raw<uint16_t, 4>& r, float (&v)[4]) {
  v[0] = __uint_as_float(r.v.x << 16); v[1] = __uint_as_float(r.v.x & 0xffff0000u);
  v[2] = __uint_as_float(r.v.y << 16); v[3] = __uint_as_float(r.v.y & 0xffff0000u);
}
__device__ __forceinline__ void expand(const Raw<uint16_t, 1>& r, float (&v)[1]) { v[0] = bf16_to_f32(r.v); }

// Every wave's LDS writes so far are visible to the workgroup; loads from
// global memory stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Bit i: step t0 + i (below steps) of sequence n restarts.
__device__ __forceinline__ uint32_t done_bits(uint8_t flag, bool live) { return (uint32_t)__ballot(live && flag); }

// Whether a lane's state after a tile is not finite.  Every wave composes the
// same maps, so all take the same way.
template <int VW>
__device__ __forceinline__ bool any_nonfinite(const float (&x)[VW]) {
  float z = 0.f;
#pragma unroll
  for (int k = 0; k < VW; ++k) z = __fmaf_rn(x[k], 0.f, z);
  return __any(z != 0.f);
}

// The states entering (mine) and leaving (x) a tile from the one entering it
// (x), chunk after chunk, each by its own wave a step at a time: the cold path
// of a tile whose composed state is not finite.  A map's decay can overflow (or
// its sum) where no step does: eight decays of 1e5 from a zero state are
// inf * 0.  pa, pb: LDS that every wave has read past.
template <int C, int TL, int VW, bool REVERSE>
__device__ __forceinline__ void step_by_step(const float (&a)[TL][VW], const float (&b)[TL][VW], float (&x)[VW],
                                             float (&mine)[VW], float* pa, float* pb, int c, int lane) {
  lds_barrier();
#pragma unroll 1
  for (int i = 0; i < C; ++i) {
    float* slot = (i & 1 ? pb : pa) + lane * VW;
    if (c == (REVERSE ? C - 1 - i : i)) {
#pragma unroll
      for (int k = 0; k < VW; ++k) mine[k] = x[k];
#pragma unroll
      for (int j = 0; j < TL; ++j)
#pragma unroll
        for (int k = 0; k < VW; ++k)
          x[k] = a[REVERSE ? TL - 1 - j : j][k] * x[k] + b[REVERSE ? TL - 1 - j : j][k];
#pragma unroll
      for (int k = 0; k < VW; ++k) slot[k] = x[k];
    }
    lds_barrier();
#pragma unroll
    for (int k = 0; k < VW; ++k) x[k] = slot[k];
  }
}

template <typename S, int VW>
__global__ void __launch_bounds__(64 * TILE_WAVES) scan_fwd_tile_kernel(ScanArgs p) {
  __shared__ float sA[2][TILE_WAVES * 64 * VW], sB[2][TILE_WAVES * 64 * VW];
  const S* a = static_cast<const S*>(p.a);
  const S* b = static_cast<const S*>(p.b);
  S* out = static_cast<S*>(p.out);
  const int lane = threadIdx.x & 63;
  constexpr int C = TILE_WAVES, TL = RL;
  const int c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int f0 = (blockIdx.x * 64 + lane) * VW;
  const bool ok = f0 < p.F;
  const int64_t n = blockIdx.y;
  const int fc = ok ? f0 : 0;  // lanes past the row read its start and store nothing
  const int64_t base = n * (int64_t)p.steps * p.F + fc;
  float h[VW], rv[VW];
  load_vec(static_cast<const S*>(p.init), n * (int64_t)p.F + fc, h);
  load_reset<S, VW>(p, n, fc, rv);
  Raw<S, VW> ra[2][TL], rb[2][TL];
  uint8_t rd[2] = {0, 0};
  auto fetch = [&](int set, int t0) {
#pragma unroll
    for (int i = 0; i < TL; ++i) {
      const int64_t o = base + (int64_t)min(t0 + i, p.steps - 1) * p.F;
      ra[set][i] = load_raw<S, VW>(a, o);
      rb[set][i] = load_raw<S, VW>(b, o);
    }
    if (p.done) rd[set] = p.done[n * p.steps + min(t0 + min(lane, TL - 1), p.steps - 1)];
  };
  const int tile = C * TL;
  auto step_tile = [&](int set, int t0) {
    // the chunk's operands (the identity map past the last step)
    const uint32_t done = p.done ? done_bits(rd[set], lane < TL) : 0u;
    float av[TL][VW], bv[TL][VW], A[VW], B[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) { A[k] = 1.f; B[k] = 0.f; }
#pragma unroll
    for (int i = 0; i < TL; ++i) {
      expand(ra[set][i], av[i]);
      expand(rb[set][i], bv[i]);
      const bool live = t0 + i < p.steps;
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        bv[i][k] = live ? bv[i][k] : 0.f;
        av[i][k] = live ? av[i][k] : 1.f;
      }
    }
    if (done) {  // a restart in this chunk
#pragma unroll
      for (int i = 0; i < TL; ++i) {
        if (!((done >> i) & 1) || t0 + i >= p.steps) continue;
#pragma unroll
        for (int k = 0; k < VW; ++k) {
          bv[i][k] = stored(bv[i][k] + stored(av[i][k] * rv[k], a), a);
          av[i][k] = 0.f;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < TL; ++i) {
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        A[k] = av[i][k] * A[k];
        B[k] = av[i][k] * B[k] + bv[i][k];
      }
    }
    float* pa = sA[set];
    float* pb = sB[set];
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      pa[(c * 64 + lane) * VW + k] = A[k];
      pb[(c * 64 + lane) * VW + k] = B[k];
    }
    if (t0 - c * TL + tile < p.steps) fetch(set ^ 1, t0 + tile);
    lds_barrier();
    float hc[VW], hs[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) hs[k] = h[k];
#pragma unroll
    for (int cc = 0; cc < C; ++cc) {
      if (cc == c) {
#pragma unroll
        for (int k = 0; k < VW; ++k) hc[k] = h[k];
      }
#pragma unroll
      for (int k = 0; k < VW; ++k) h[k] = pa[(cc * 64 + lane) * VW + k] * h[k] + pb[(cc * 64 + lane) * VW + k];
    }
    if (__builtin_expect(any_nonfinite(h), 0)) {
#pragma unroll
      for (int k = 0; k < VW; ++k) h[k] = hs[k];
      step_by_step<C, TL, VW, false>(av, bv, h, hc, pa, pb, c, lane);
    }
#pragma unroll
    for (int i = 0; i < TL; ++i) {
#pragma unroll
      for (int k = 0; k < VW; ++k) hc[k] = av[i][k] * hc[k] + bv[i][k];
      if (ok && t0 + i < p.steps) store_vec(out, base + (int64_t)(t0 + i) * p.F, hc);
    }
  };
  fetch(0, c * TL);
  // (the register sets alternate by unrolling, so that each is indexed by a constant)
  for (int t0 = c * TL, done_steps = 0; done_steps < p.steps; done_steps += 2 * tile, t0 += 2 * tile) {
    step_tile(0, t0);
    if (done_steps + tile < p.steps) step_tile(1, t0 + tile);
  }
}

template <typename S, int VW>
__global__ void __launch_bounds__(64 * TILE_WAVES) scan_bwd_tile_kernel(ScanArgs p) {
  __shared__ float sA[2][TILE_WAVES * 64 * VW], sB[2][TILE_WAVES * 64 * VW];
  const S* a = static_cast<const S*>(p.a);
  const S* g = static_cast<const S*>(p.b);
  const S* hs = static_cast<const S*>(p.h);
  const S* init = static_cast<const S*>(p.init);
  S* db = static_cast<S*>(p.out);
  S* da = static_cast<S*>(p.da);
  S* dinit = static_cast<S*>(p.dinit);
  const int lane = threadIdx.x & 63;
  constexpr int C = TILE_WAVES, TL = sizeof(S) * VW > 8 ? 4 : RL;  // 8 float4 steps spill
  const int c = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int f0 = (blockIdx.x * 64 + lane) * VW;
  const bool ok = f0 < p.F;
  const int64_t n = blockIdx.y;
  const int fc = ok ? f0 : 0;
  const int64_t base = n * (int64_t)p.steps * p.F + fc;
  float d[VW], rv[VW];
#pragma unroll
  for (int k = 0; k < VW; ++k) d[k] = 0.f;
  load_reset<S, VW>(p, n, fc, rv);
  // of step t: a_{t+1}, g_t, h_{t-1} (init at t = 0); the flags of steps t0 .. t0 + TL
  Raw<S, VW> ra[2][TL], rg[2][TL], rh[2][TL];
  uint8_t rd[2] = {0, 0};
  auto fetch = [&](int set, int t0) {
#pragma unroll
    for (int i = 0; i < TL; ++i) {
      const int t = min(t0 + i, p.steps - 1);
      ra[set][i] = load_raw<S, VW>(a, base + (int64_t)min(t + 1, p.steps - 1) * p.F);
      rg[set][i] = load_raw<S, VW>(g, base + (int64_t)t * p.F);
      rh[set][i] = load_raw<S, VW>(t > 0 ? hs : init, t > 0 ? base + (int64_t)(t - 1) * p.F : n * (int64_t)p.F + fc);
    }
    if (p.done) rd[set] = p.done[n * p.steps + min(t0 + min(lane, TL), p.steps - 1)];
  };
  const int tile = C * TL;
  const int ntiles = (p.steps + tile - 1) / tile;
  auto step_tile = [&](int set, int it) {
    const int t0 = it * tile + c * TL;
    const uint32_t done = p.done ? done_bits(rd[set], lane <= TL) : 0u;
    float al[TL][VW], gv[TL][VW], hp[TL][VW], P[VW], Q[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) { P[k] = 1.f; Q[k] = 0.f; }
#pragma unroll
    for (int i = TL - 1; i >= 0; --i) {
      expand(ra[set][i], al[i]);
      expand(rg[set][i], gv[i]);
      expand(rh[set][i], hp[i]);
      // no decay into a restarted step or past the last one; the identity past the end
      const bool live = t0 + i < p.steps, cut = t0 + i + 1 >= p.steps || ((done >> (i + 1)) & 1);
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        al[i][k] = live ? (cut ? 0.f : al[i][k]) : 1.f;
        gv[i][k] = live ? gv[i][k] : 0.f;
        P[k] = al[i][k] * P[k];
        Q[k] = al[i][k] * Q[k] + gv[i][k];
      }
    }
    float* pa = sA[set];
    float* pb = sB[set];
#pragma unroll
    for (int k = 0; k < VW; ++k) {
      pa[(c * 64 + lane) * VW + k] = P[k];
      pb[(c * 64 + lane) * VW + k] = Q[k];
    }
    if (it > 0) fetch(set ^ 1, t0 - tile);
    lds_barrier();
    float dc[VW], ds[VW];
#pragma unroll
    for (int k = 0; k < VW; ++k) ds[k] = d[k];
#pragma unroll
    for (int cc = C - 1; cc >= 0; --cc) {
      if (cc == c) {
#pragma unroll
        for (int k = 0; k < VW; ++k) dc[k] = d[k];
      }
#pragma unroll
      for (int k = 0; k < VW; ++k) d[k] = pa[(cc * 64 + lane) * VW + k] * d[k] + pb[(cc * 64 + lane) * VW + k];
    }
    if (__builtin_expect(any_nonfinite(d), 0)) {
#pragma unroll
      for (int k = 0; k < VW; ++k) d[k] = ds[k];
      step_by_step<C, TL, VW, true>(al, gv, d, dc, pa, pb, c, lane);
    }
#pragma unroll
    for (int i = TL - 1; i >= 0; --i) {
      const int t = t0 + i;
      float dv[VW], dav[VW];
#pragma unroll
      for (int k = 0; k < VW; ++k) {
        dc[k] = al[i][k] * dc[k] + gv[i][k];
        dv[k] = stored(dc[k], db);
        dav[k] = dv[k] * hp[i][k];
      }
      if ((done >> i) & 1) {
#pragma unroll
        for (int k = 0; k < VW; ++k) dav[k] = stored(rv[k] * dv[k], a);
      }
      if (ok && t < p.steps) {
        store_vec(db, base + (int64_t)t * p.F, dc);
        store_vec(da, base + (int64_t)t * p.F, dav);
        if (t == 0) {
          float a0[VW], di[VW];
          load_vec(a, base, a0);
#pragma unroll
          for (int k = 0; k < VW; ++k) di[k] = dv[k] * ((done & 1) ? 0.f : a0[k]);
          store_vec(dinit, n * (int64_t)p.F + f0, di);
        }
      }
    }
  };
  int it = ntiles - 1;
  fetch(0, it * tile + c * TL);
  for (; it >= 0; it -= 2) {
    step_tile(0, it);
    if (it > 0) step_tile(1, it - 1);
  }
}

bool aligned(const void* ptr, int bytes) { return (reinterpret_cast<uintptr_t>(ptr) % bytes) == 0; }

template <typename S, int VW, bool BWD>
int launch_tile(hipStream_t st, const ScanArgs& p, int batch) {
  const int groups = ppo::ceil_div(ppo::ceil_div(p.F, VW), 64);
  dim3 grid(groups, batch), block(64 * TILE_WAVES);
  if constexpr (BWD) {
    hipLaunchKernelGGL((scan_bwd_tile_kernel<S, VW>), grid, block, 0, st, p);
  } else {
    hipLaunchKernelGGL((scan_fwd_tile_kernel<S, VW>), grid, block, 0, st, p);
  }
  return PPO_OK;
}

template <typename S, int VW, bool BWD>
int launch_reg(hipStream_t st, const ScanArgs& p, int batch) {
  const int groups = ppo::ceil_div(ppo::ceil_div(p.F, VW), 64);
  const int C = ppo::ceil_div(p.steps, RL);
  dim3 grid(groups, batch), block(64 * C);
  const size_t lds = C > 1 ? 2 * sizeof(float) * (size_t)C * 64 * VW : 0;
  if (BWD) {
    hipLaunchKernelGGL((scan_bwd_reg_kernel<S, VW>), grid, block, lds, st, p);
  } else {
    hipLaunchKernelGGL((scan_fwd_reg_kernel<S, VW>), grid, block, lds, st, p);
  }
  return PPO_OK;
}

template <bool BWD>
int dispatch(hipStream_t st, int dtype, ScanArgs p, int batch, const char* what) {
  // 4 features per lane where the rows allow (16-byte float32 or 8-byte bf16
  // accesses; for bf16, 8 per lane would halve the waves in flight).
  const int esize = dtype == SCAN_F32 ? 4 : 2;
  const void* ptrs[8] = {p.a, p.b, p.h, p.init, p.out, p.da, p.dinit, p.reset};
  bool vec = p.F % 4 == 0;
  for (const void* q : ptrs)
    if (q && !aligned(q, 4 * esize)) vec = false;
  // up to 128 steps one register-resident tile (every load of the sequence in
  // flight at once), longer sequences tile after tile
  const bool one = p.steps <= RL * MAX_CHUNKS;
  if (dtype == SCAN_F32) {
    if (vec) one ? launch_reg<float, 4, BWD>(st, p, batch) : launch_tile<float, 4, BWD>(st, p, batch);
    else one ? launch_reg<float, 1, BWD>(st, p, batch) : launch_tile<float, 1, BWD>(st, p, batch);
  } else {
    if (vec) one ? launch_reg<uint16_t, 4, BWD>(st, p, batch) : launch_tile<uint16_t, 4, BWD>(st, p, batch);
    else one ? launch_reg<uint16_t, 1, BWD>(st, p, batch) : launch_tile<uint16_t, 1, BWD>(st, p, batch);
  }
  return ppo::check_launch(what);
}

}  // namespace

PPO_EXPORT int ppo_linear_scan_fwd(void* stream, int dtype, const void* a, const void* b, const void* init, void* out,
                                   int batch, int steps, int features) {
  if (batch < 0 || steps < 0 || features < 0 || (dtype != SCAN_F32 && dtype != SCAN_BF16))
    return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_fwd: bad argument (batch %d steps %d features %d dtype %d)",
                          batch, steps, features, dtype);
  if (batch == 0 || steps == 0 || features == 0) return PPO_OK;
  if (!a || !b || !init || !out) return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_fwd: null buffer");
  if (batch > 65535) return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_fwd: batch above 65535");
  ScanArgs p{a, b, nullptr, init, out, nullptr, nullptr, steps, features, nullptr, nullptr};
  return dispatch<false>(ppo::as_stream(stream), dtype, p, batch, "ppo_linear_scan_fwd");
}

PPO_EXPORT int ppo_ssm_scan_fwd(void* stream, int dtype, const void* a, const void* b, const uint8_t* done,
                                const void* reset, const void* carry, void* out, int batch, int steps, int features) {
  if (batch < 0 || steps < 0 || features < 0 || (dtype != SCAN_F32 && dtype != SCAN_BF16))
    return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_fwd: bad argument (batch %d steps %d features %d dtype %d)",
                          batch, steps, features, dtype);
  if (batch == 0 || steps == 0 || features == 0) return PPO_OK;
  if (!a || !b || !done || !carry || !out) return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_fwd: null buffer");
  if (batch > 65535) return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_fwd: batch above 65535");
  ScanArgs p{a, b, nullptr, carry, out, nullptr, nullptr, steps, features, done, reset};
  return dispatch<false>(ppo::as_stream(stream), dtype, p, batch, "ppo_ssm_scan_fwd");
}

PPO_EXPORT int ppo_linear_scan_bwd(void* stream, int dtype, const void* a, const void* h, const void* init,
                                   const void* cot, void* da, void* db, void* dinit, int batch, int steps,
                                   int features) {
  if (batch < 0 || steps < 0 || features < 0 || (dtype != SCAN_F32 && dtype != SCAN_BF16))
    return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_bwd: bad argument (batch %d steps %d features %d dtype %d)",
                          batch, steps, features, dtype);
  if (batch == 0 || steps == 0 || features == 0) return PPO_OK;
  if (!a || !h || !init || !cot || !da || !db || !dinit)
    return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_bwd: null buffer");
  if (batch > 65535) return ppo::set_error(PPO_ERR_ARG, "ppo_linear_scan_bwd: batch above 65535");
  ScanArgs p{a, cot, h, init, db, da, dinit, steps, features, nullptr, nullptr};
  return dispatch<true>(ppo::as_stream(stream), dtype, p, batch, "ppo_linear_scan_bwd");
}

PPO_EXPORT int ppo_ssm_scan_bwd(void* stream, int dtype, const void* a, const void* h, const uint8_t* done,
                                const void* reset, const void* carry, const void* cot, void* da, void* db,
                                void* dcarry, int batch, int steps, int features) {
  if (batch < 0 || steps < 0 || features < 0 || (dtype != SCAN_F32 && dtype != SCAN_BF16))
    return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_bwd: bad argument (batch %d steps %d features %d dtype %d)",
                          batch, steps, features, dtype);
  if (batch == 0 || steps == 0 || features == 0) return PPO_OK;
  if (!a || !h || !done || !carry || !cot || !da || !db || !dcarry)
    return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_bwd: null buffer");
  if (batch > 65535) return ppo::set_error(PPO_ERR_ARG, "ppo_ssm_scan_bwd: batch above 65535");
  ScanArgs p{a, cot, h, carry, db, da, dcarry, steps, features, done, reset};
  return dispatch<true>(ppo::as_stream(stream), dtype, p, batch, "ppo_ssm_scan_bwd");
}
