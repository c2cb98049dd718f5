// The whole rollout-side PPO.step (boonta/algorithms/ppo.py:57-74) of an MLP
// actor-critic with separate torsos of one shape (flax's ActorCritic, e.g. the
// Gaussian workload's 4 x 256 LayerNorm + SiLU towers) in one launch: both
// towers' Dense [+ LayerNorm] + activation layers, the policy and value heads
// and dist.sample_and_log_prob(seed=key) (categorical.h, gaussian.h).
//
// A workgroup owns 16 env rows of one tower: the draw needs only the actor's
// outputs and the value only the critic's, so the towers never meet.  Each
// layer is 16 x F outputs with the features split over the workgroup's waves
// (v_mfma_f32_16x16x4f32; wave w's lane li holds features 16 NB w + NB li ..),
// its input the observation rows or the previous layer's outputs in LDS; no
// layer's output goes to memory.  The head (<= 16 outputs) splits its
// contraction over the waves; then one 16-lane group per row draws.
//
// What bounds it: a serial chain of L contractions, each reading its kernel from
// L2 beside fp32 MFMA (24 us of them at 4096 rows of 4 x 256 towers on 87
// inputs).  There (two workgroups per CU) the step with its host side takes 64
// us, eleven launches 125; with 64-deep sets of loads in flight (214 registers,
// one workgroup per CU) instead of 32-deep ones 87.
#include "categorical.h"
#include "common.h"
#include "gaussian.h"
#include "mlp_tile.h"

namespace {

constexpr int ST_ROWS = 16;
constexpr int ST_MAX_LAYERS = 8;
constexpr int ST_HEAD = 16;  // head outputs

struct StepTowersArgs {
  const float* obs;
  int64_t ldo;
  int rows, K0, L;
  float eps;
  const float* W[2][ST_MAX_LAYERS];  // [tower][layer]: [K_l, F]
  const float* bias[2][ST_MAX_LAYERS];
  const float* gamma[2][ST_MAX_LAYERS];
  const float* beta[2][ST_MAX_LAYERS];
  const float* Wh[2];  // heads [F, ldwh]
  const float* bh[2];
  int64_t ldwh[2];
  int A;               // actor outputs
  const float* scale;  // Gaussian: raw scale [A]; categorical: null
  const uint32_t* key;
  float temperature;
  int32_t* action_i;
  float* action_f;
  float* log_prob;
  float* value;
};

template <int F, int NW, int ACT, bool LN, bool VA>
__global__ void __launch_bounds__(64 * NW, F == 256 ? 4 : 1) step_towers_kernel(StepTowersArgs p) {
  constexpr int NB = F / (16 * NW);  // a wave's 16-feature blocks
  static_assert(NB * 16 * NW == F && NW >= 4, "four waves draw");
  constexpr int CH = F == 256 ? 2 : 4;  // 16-deep chunks of loads ahead of the MFMAs (256 wide: two workgroups per CU)
  __shared__ __attribute__((aligned(16))) float sX[ST_ROWS][F + 4];
  __shared__ float s_sum[LN ? NW : 1][ST_ROWS];
  __shared__ float s_sq[LN ? NW : 1][ST_ROWS];
  __shared__ float s_head[NW][ST_ROWS][ST_HEAD + 1];
  __shared__ float s_out[ST_ROWS][ST_HEAD + 1];
  const int t = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
  const int li = lane & 15;
  const int kq = lane >> 4;
  const int r0 = blockIdx.x * ST_ROWS;
  const int c = 16 * NB * wave + NB * li;
  const bool a_live = r0 + li < p.rows;
  const float* xrow = p.obs + (a_live ? (int64_t)(r0 + li) * p.ldo : 0);

  // this lane's head weights: features 16 (NB wave + q) + 4 kq + s, output li
  const float* Wh = p.Wh[t];
  const int64_t ldwh = p.ldwh[t];
  const bool out_live = li < (t == 0 ? p.A : 1);
  float wh[NB][4];
#pragma unroll
  for (int q = 0; q < NB; ++q)
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const float x = Wh[(16 * (NB * wave + q) + 4 * kq + s) * ldwh + (out_live ? li : 0)];
      wh[q][s] = out_live ? x : 0.f;
    }

  for (int l = 0; l < p.L; ++l) {
    const float* W = p.W[t][l];
    float bias[NB], g[NB], be[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) bias[j] = 0.f;
    if (p.bias[t][l]) load_nb<NB>(p.bias[t][l] + c, bias);
    if constexpr (LN) {
      load_nb<NB>(p.gamma[t][l] + c, g);
      load_nb<NB>(p.beta[t][l] + c, be);
    }
    floatx4 acc[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (l == 0)
      act_contract<F, NB, false, VA, CH>(acc, xrow, a_live, W, p.K0, kq, c);
    else
      act_contract<F, NB, true, true, CH>(acc, &sX[li][0], true, W, F, kq, c);
    if constexpr (LN) {
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        float ps = 0.f, pq = 0.f;
#pragma unroll
        for (int j = 0; j < NB; ++j) ppo::ln_accum(acc[j][v] + bias[j], ps, pq);
        ps = ppo::sum16(ps);
        pq = ppo::sum16(pq);
        if (li == 0) {
          s_sum[wave][4 * kq + v] = ps;
          s_sq[wave][4 * kq + v] = pq;
        }
      }
    }
    __syncthreads();  // every wave is past its reads of the tile
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int rr = 4 * kq + v;
      float y[NB];
      if constexpr (LN) {
        float s = 0.f, s2 = 0.f, mean, rstd;
#pragma unroll
        for (int w = 0; w < NW; w += 2) {
          s += s_sum[w][rr] + s_sum[w + 1][rr];
          s2 += s_sq[w][rr] + s_sq[w + 1][rr];
        }
        static_assert(!LN || F == 256, "row statistics over 256 features");
        ppo::ln_stats256(s, s2, p.eps, mean, rstd);
#pragma unroll
        for (int j = 0; j < NB; ++j)
          y[j] = ppo::act_fwd(ACT, ppo::ln_apply(acc[j][v] + bias[j], mean, rstd, g[j], be[j]));
      } else {
#pragma unroll
        for (int j = 0; j < NB; ++j) y[j] = ppo::act_fwd(ACT, acc[j][v] + bias[j]);
      }
      store_nb<NB>(&sX[rr][c], y);
    }
    __syncthreads();
  }

  // head: wave w contracts its 16 NB features for all outputs
  {
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      const floatx4 x = *reinterpret_cast<const floatx4*>(&sX[li][16 * (NB * wave + q) + 4 * kq]);
#pragma unroll
      for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[s], wh[q][s], acc, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) s_head[wave][4 * kq + v][li] = acc[v];
  }
  __syncthreads();
  const int row = threadIdx.x / 16;
  const int j0 = threadIdx.x % 16;
  const int r = r0 + row;
  const int n = t == 0 ? p.A : 1;
  if (wave < 4) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < NW; w += 2) o += s_head[w][row][j0] + s_head[w + 1][row][j0];
    s_out[row][j0] = o + (j0 < n && p.bh[t] ? p.bh[t][j0] : 0.f);
  }
  __syncthreads();
  if (wave >= 4) return;
  const bool row_ok = r < p.rows;
  if (t == 1) {
    if (row_ok && j0 == 0) p.value[r] = s_out[row][0];
    return;
  }
  const uint32_t k0 = p.key[0], k1 = p.key[1];
  if (p.scale) {
    float lpx = 0.f, logdet = 0.f;
    if (row_ok && j0 < p.A) {
      const uint64_t i = (uint64_t)r * (uint64_t)p.A + (uint64_t)j0;
      p.action_f[i] = ppo::gauss::draw(s_out[row][j0], p.scale[j0], k0, k1, i, p.temperature, lpx, logdet);
    }
    lpx = ppo::cat::group_sum(lpx);
    logdet = ppo::cat::group_sum(logdet);
    if (row_ok && j0 == 0) p.log_prob[r] = lpx - logdet;
  } else {
    int act_i;
    float lp;
    ppo::cat::draw(&s_out[row][0], p.A, row_ok, r, k0, k1, p.temperature, j0, act_i, lp);
    if (row_ok && j0 == 0) {
      p.action_i[r] = act_i;
      p.log_prob[r] = lp;
    }
  }
}

// A shared head of at most 16 outputs and its categorical draw: 16 rows per
// workgroup, the contraction over the F features split over eight waves (alternate
// 16-deep chunks), then a 16-lane group per row.  Bound by latency; instead of
// the head GEMM, whose 64-column tiles are three quarters padding, and the
// sampling launch.
constexpr int HS_WAVES = 8;

struct HeadSampleArgs {
  const float* X;  // [rows, F]
  int64_t ldx;
  int rows, F;
  const float* Wh;  // [F, ldwh]: A logits, then the value
  int64_t ldwh;
  const float* bh;
  int A;
  const uint32_t* key;
  float temperature;
  int32_t* action;
  float* log_prob;
  float* value;
};

__global__ void __launch_bounds__(64 * HS_WAVES) head_sample_kernel(HeadSampleArgs p) {
  __shared__ float s_head[HS_WAVES][ST_ROWS][ST_HEAD + 1];
  __shared__ float s_out[ST_ROWS][ST_HEAD + 1];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int li = lane & 15;
  const int kq = lane >> 4;
  const int r0 = blockIdx.x * ST_ROWS;
  const bool a_live = r0 + li < p.rows;
  const float* xrow = p.X + (int64_t)(a_live ? r0 + li : r0) * p.ldx;
  const bool out_live = li <= p.A;
  const float* wcol = p.Wh + (out_live ? li : 0);
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
  for (int k0 = 16 * wave; k0 < p.F; k0 += 16 * HS_WAVES) {
    const int k = k0 + 4 * kq;
    const floatx4 x = *reinterpret_cast<const floatx4*>(xrow + k);
    float w[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) w[s] = wcol[(k + s) * p.ldwh];
#pragma unroll
    for (int s = 0; s < 4; ++s)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a_live ? x[s] : 0.f, out_live ? w[s] : 0.f, acc, 0, 0, 0);
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) s_head[wave][4 * kq + v][li] = acc[v];
  __syncthreads();
  const int row = threadIdx.x / 16;
  const int j0 = threadIdx.x % 16;
  const int r = r0 + row;
  if (wave < 4) {
    float o = 0.f;
#pragma unroll
    for (int w = 0; w < HS_WAVES; w += 2) o += s_head[w][row][j0] + s_head[w + 1][row][j0];
    s_out[row][j0] = o + (j0 <= p.A && p.bh ? p.bh[j0] : 0.f);
  }
  __syncthreads();
  if (wave >= 4) return;
  const bool row_ok = r < p.rows;
  int act_i;
  float lp;
  ppo::cat::draw(&s_out[row][0], p.A, row_ok, r, p.key[0], p.key[1], p.temperature, j0, act_i, lp);
  if (row_ok && j0 == 0) {
    p.action[r] = act_i;
    p.log_prob[r] = lp;
    p.value[r] = s_out[row][p.A];
  }
}

bool aligned16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; }

}  // namespace

PPO_EXPORT int ppo_step_towers_max_layers() { return ST_MAX_LAYERS; }
PPO_EXPORT int ppo_step_towers_max_outputs() { return ST_HEAD; }

PPO_EXPORT int ppo_step_towers_f32(void* stream, const float* obs, int64_t ldo, int rows, int obs_dim, int layers,
                                   int features, const float* const* weights, const float* const* biases,
                                   const float* const* gammas, const float* const* betas, float eps, int act,
                                   const float* const* head_w, const int64_t* ldwh, const float* const* head_b, int A,
                                   const float* scale, const uint32_t* key, float temperature, void* action,
                                   float* log_prob, float* value) {
  const char* name = "ppo_step_towers_f32";
  const bool ln = gammas != nullptr;
  const int F = features;
  if (rows < 0 || obs_dim < 1 || ldo < obs_dim || layers < 1 || layers > ST_MAX_LAYERS || act < 0 || act > 3 ||
      (F != 64 && F != 128 && F != 256) || (ln && (F != 256 || !betas)) || (!ln && act == ACT_SILU) ||
      (int64_t)obs_dim * F > INT32_MAX || A < 1 || A > ST_HEAD || !weights || !biases || !head_w || !ldwh || !head_b)
    return ppo::set_error(PPO_ERR_ARG, "%s: bad argument (rows %d obs %d layers %d features %d act %d A %d)", name,
                          rows, obs_dim, layers, F, act, A);
  if (rows == 0) return PPO_OK;
  if (!obs || !key || !action || !log_prob || !value) return ppo::set_error(PPO_ERR_ARG, "%s: null buffer", name);
  StepTowersArgs a{};
  a.obs = obs; a.ldo = ldo; a.rows = rows; a.K0 = obs_dim; a.L = layers; a.eps = eps;
  for (int t = 0; t < 2; ++t) {
    for (int l = 0; l < layers; ++l) {
      const int i = t * layers + l;
      if (!weights[i] || !aligned16(weights[i]) || (biases[i] && !aligned16(biases[i])) ||
          (ln && (!gammas[i] || !betas[i] || !aligned16(gammas[i]) || !aligned16(betas[i]))))
        return ppo::set_error(PPO_ERR_ARG, "%s: tower %d layer %d needs 16-byte aligned parameters", name, t, l);
      a.W[t][l] = weights[i]; a.bias[t][l] = biases[i];
      if (ln) { a.gamma[t][l] = gammas[i]; a.beta[t][l] = betas[i]; }
    }
    if (!head_w[t] || ldwh[t] < (t == 0 ? A : 1))
      return ppo::set_error(PPO_ERR_ARG, "%s: bad head of tower %d", name, t);
    a.Wh[t] = head_w[t]; a.ldwh[t] = ldwh[t]; a.bh[t] = head_b[t];
  }
  a.A = A; a.scale = scale; a.key = key; a.temperature = temperature; a.log_prob = log_prob; a.value = value;
  if (scale) a.action_f = static_cast<float*>(action);
  else a.action_i = static_cast<int32_t*>(action);
  const bool va = aligned16(obs) && ldo % 4 == 0;  // ldo >= obs_dim, so >= obs_dim rounded up to 4
  const dim3 grid(ppo::ceil_div(rows, ST_ROWS), 2);
  hipStream_t st = ppo::as_stream(stream);
#define PPO_STEP_TOWERS(FV, NWV, ACTV, LNV)                                                                     \
  if (va) hipLaunchKernelGGL((step_towers_kernel<FV, NWV, ACTV, LNV, true>), grid, dim3(64 * NWV), 0, st, a);  \
  else hipLaunchKernelGGL((step_towers_kernel<FV, NWV, ACTV, LNV, false>), grid, dim3(64 * NWV), 0, st, a);
#define PPO_STEP_TOWERS_W(ACTV)                                \
  if (F == 64) { PPO_STEP_TOWERS(64, 4, ACTV, false) }         \
  else if (F == 128) { PPO_STEP_TOWERS(128, 8, ACTV, false) }  \
  else if (!ln) { PPO_STEP_TOWERS(256, 8, ACTV, false) }       \
  else { PPO_STEP_TOWERS(256, 8, ACTV, true) }
  switch (act) {
    case ACT_RELU: PPO_STEP_TOWERS_W(ACT_RELU) break;
    case ACT_TANH: PPO_STEP_TOWERS_W(ACT_TANH) break;
    case ACT_SILU: PPO_STEP_TOWERS(256, 8, ACT_SILU, true) break;
    default: PPO_STEP_TOWERS_W(ACT_NONE) break;
  }
#undef PPO_STEP_TOWERS_W
#undef PPO_STEP_TOWERS
  return ppo::check_launch(name);
}

PPO_EXPORT int ppo_head_sample_categorical_f32(void* stream, const float* x, int64_t ldx, int rows, int F,
                                               const float* head_w, int64_t ldwh, const float* head_b, int A,
                                               const uint32_t* key, float temperature, int32_t* action,
                                               float* log_prob, float* value) {
  const char* name = "ppo_head_sample_categorical_f32";
  if (rows < 0 || F < 16 || F % 16 || ldx < F || ldx % 4 || A < 1 || A + 1 > ST_HEAD || ldwh < A + 1)
    return ppo::set_error(PPO_ERR_ARG, "%s: bad argument (rows %d features %d A %d)", name, rows, F, A);
  if (rows == 0) return PPO_OK;
  if (!x || !head_w || !key || !action || !log_prob || !value || !aligned16(x))
    return ppo::set_error(PPO_ERR_ARG, "%s: null or misaligned buffer", name);
  HeadSampleArgs a{x, ldx, rows, F, head_w, ldwh, head_b, A, key, temperature, action, log_prob, value};
  hipLaunchKernelGGL(head_sample_kernel, dim3(ppo::ceil_div(rows, ST_ROWS)), dim3(64 * HS_WAVES), 0,
                     ppo::as_stream(stream), a);
  return ppo::check_launch(name);
}
