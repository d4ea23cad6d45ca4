// A whole MLP forward in one launch, for the rollout side (rsl_rl/models/mlp_model.py:82-118): concatenate the
// observation groups, normalise them (rsl_rl/modules/normalization.py:46-48), and run every linear layer with its
// activation (rsl_rl/modules/mlp.py:91-95).
//
// What bounds it is latency: a policy step of a few thousand rows is 0.1 to 3 GFLOP, and as one launch per layer it spent
// its time on launches, on the host calls before them and on GEMM tiles that filled a fraction of the chip (4,096 rows x
// [512, 256, 128], actor: normaliser and four GEMMs 80 us of kernel time and 94 us of host time).  Here a block takes 16
// rows through all layers: the rows' activations stay in LDS (two buffers), the weights come from the caches straight
// into the MFMA operand registers, 64 k ahead, and nothing is written but the output: one launch of 33 us for 16 to
// 2,048 rows, 34 for 4,096 (the layers one by one 64 us).  16 rows give 4,096 rows 256 blocks, one per
// compute unit.  v_mfma_f32_16x16x4f32 with the weights as the first operand leaves each lane 4 consecutive outputs of one
// row: one 16-byte LDS store each.  Past some thousands of rows, and for networks of more weights than those launches' time
// (every block reads all of them; _Route in models.py), the layers' own GEMMs (weights read once per 128 rows, bf16 matrix
// cores) are faster: the caller's choice.
#include "gemm_core.hpp"

namespace ppo {
namespace {

constexpr int kMlpRows = 16, kMlpWaves = 8, kMlpThreads = 64 * kMlpWaves;
constexpr int kMlpMaxWidth = 1024;

struct MlpArgs {
  ppo_mlp_problem p;
  int32_t blocks;  // of 16 rows
  int32_t ldx;     // floats per LDS row
  int64_t rows;
};
static_assert(sizeof(MlpArgs) <= 4096, "kernel arguments");

// One launch of ppo_mlp_fwd_pairs: layers l0 and, where there is one, l0 + 1.
struct MlpPairs {
  MlpArgs g;
  const float* in;  // [rows, ld] (NULL: the problem's input blocks)
  float* to;        // [rows, ld]
  int64_t ld;
  int32_t slices;  // blocks per 16 rows, kSliceTiles tiles of the second layer each
  int32_t l0;
};
static_assert(sizeof(MlpPairs) <= 4096, "kernel arguments");
constexpr int kSliceTiles = 4;  // one per SIMD

// Where a layer's outputs go: LDS y, or global rows (`out`).
struct MlpOut {
  float* y;  // [16][ldx], used where out is NULL
  float* out;
  int64_t ldo, row0, rows;
};

// Output tiles [t_begin, t_end) of one layer for the block's 16 rows: x [16][ldx] (columns past K up to the next multiple
// of 16 zero) -> D, after the activation `act` (PPO_ACT_NONE: none).  TILES 16-wide output tiles per wave and AH k-groups
// of 16 loaded ahead at a time.  (For the one launch of all layers, deeper prefetch, eight k-groups and the next tiles'
// first chunk at two waves per SIMD, measured 44 us against 34 for 16 rows of 48 -> [512, 256, 128] -> 12.)
template <int TILES, int AH, bool VEC>
__device__ __forceinline__ void mlp_layer(const ppo_mlp_layer& L, int act, const float* x, int ldx, const MlpOut& D,
                                          int t_begin, int t_end, int wave, int lane) {
  const int K = L.in_features, N = L.out_features;
  const int m = lane & 15, q = lane >> 4;
  const int groups = (K + 15) >> 4;
  for (int t0 = t_begin + wave * TILES; t0 < t_end; t0 += kMlpWaves * TILES) {
    const float* wrow[TILES];
#pragma unroll
    for (int j = 0; j < TILES; ++j) wrow[j] = L.w + static_cast<int64_t>(min(16 * (t0 + j) + m, N - 1)) * K;
    auto load_w = [&](int g, f32x4 (&v)[TILES]) __attribute__((always_inline)) {
      const int k = 16 * g + 4 * q;
#pragma unroll
      for (int j = 0; j < TILES; ++j) {
        if constexpr (VEC) {  // K % 4 == 0: a piece is in the row or past it
          v[j] = *reinterpret_cast<const f32x4*>(wrow[j] + min(k, K - 4));
          if (k >= K) v[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float w = wrow[j][min(k + e, K - 1)];
            v[j][e] = k + e < K ? w : 0.0f;
          }
        }
      }
    };
    f32x4 acc[TILES][2];
#pragma unroll
    for (int j = 0; j < TILES; ++j) acc[j][0] = acc[j][1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    f32x4 w[2][AH][TILES];
#pragma unroll
    for (int i = 0; i < AH; ++i) load_w(min(i, groups - 1), w[0][i]);
    float bias[TILES][4];
    auto load_bias = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < TILES; ++j)
#pragma unroll
        for (int e = 0; e < 4; ++e) bias[j][e] = L.b[min(16 * (t0 + j) + 4 * q + e, N - 1)];
    };
    if constexpr (TILES == 1) load_bias();  // (two tiles' weights fill the registers)
    for (int g0 = 0; g0 < groups; g0 += 2 * AH) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int gb = g0 + b * AH;
        if (gb < groups) {
#pragma unroll
          for (int i = 0; i < AH; ++i) load_w(min(gb + AH + i, groups - 1), w[b ^ 1][i]);
#pragma unroll
          for (int i = 0; i < AH; ++i) {
            if (gb + i < groups) {
              const f32x4 xv = *reinterpret_cast<const f32x4*>(x + m * ldx + 16 * (gb + i) + 4 * q);
#pragma unroll
              for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int j = 0; j < TILES; ++j)
                  acc[j][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(w[b][i][j][s], xv[s], acc[j][i & 1], 0, 0, 0);
            }
          }
        }
      }
    }
    if constexpr (TILES > 1) load_bias();
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int n = 16 * (t0 + j) + 4 * q;
      if (t0 + j >= t_end) continue;
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = acc[j][0][e] + acc[j][1][e] + bias[j][e];
        o[e] = n + e >= N ? 0.0f : act == PPO_ACT_NONE ? z : act == PPO_ACT_ELU ? elu_fast(z) : act_fwd(act, z);
      }
      if (D.out == nullptr) {
        *reinterpret_cast<f32x4*>(D.y + m * ldx + n) = o;
      } else if (D.row0 + m < D.rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) D.out[(D.row0 + m) * D.ldo + n + e] = o[e];
      }
    }
  }
}

// DEEP: one tile per wave at a time with eight k-groups ahead (a block has a few tiles, each wave's loads are its time).
template <bool DEEP>
__device__ __forceinline__ void mlp_run_layer(const ppo_mlp_layer& L, int act, const float* x, int ldx, const MlpOut& D,
                                              int t_begin, int t_end, int wave, int lane) {
  const bool vec = L.in_features % 4 == 0 && reinterpret_cast<uintptr_t>(L.w) % 16 == 0;
  if (!vec)
    mlp_layer<1, 4, false>(L, act, x, ldx, D, t_begin, t_end, wave, lane);
  else if (t_end - t_begin > kMlpWaves)
    mlp_layer<2, 4, true>(L, act, x, ldx, D, t_begin, t_end, wave, lane);
  else
    mlp_layer<1, DEEP ? 8 : 4, true>(L, act, x, ldx, D, t_begin, t_end, wave, lane);
}

__device__ __forceinline__ int mlp_tiles(const ppo_mlp_layer& L) { return (L.out_features + 15) >> 4; }

// The problem's 16 input rows -> x: 32 threads per row, the blocks side by side, normalised as ppo_obs_normalize does.
__device__ __forceinline__ void mlp_input(const ppo_mlp_problem& P, float* x, int ldx, int64_t row0, int64_t rows, int tid) {
  const int r = tid >> 5, c0 = tid & 31;
  const int64_t row = min(row0 + r, rows - 1);
  const bool in = row0 + r < rows;
  int col = 0;
  for (int s = 0; s < P.num_blocks; ++s) {
    const ppo_column_block& B = P.x[s];
    const float* const src = B.src + row * B.stride;
    for (int c = c0; c < B.width; c += 128) {  // four columns' loads in flight (past the width the last one, dropped)
      float v[4], mean[4], sd[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int cc = min(c + 32 * u, B.width - 1);
        v[u] = src[cc];
        if (P.norm_mean != nullptr) {
          mean[u] = P.norm_mean[col + cc];
          sd[u] = P.norm_std[col + cc];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        float q = in ? v[u] : 0.0f;
        if (P.norm_mean != nullptr) q = (q - mean[u]) / (sd[u] + P.norm_eps);
        if (c + 32 * u < B.width) x[r * ldx + col + c + 32 * u] = q;
      }
    }
    col += B.width;
  }
  for (int c = col + c0; c < (col + 15) / 16 * 16; c += 32) x[r * ldx + c] = 0.0f;
}

__global__ __launch_bounds__(kMlpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void mlp_fwd_kernel(const MlpArgs g) {
  extern __shared__ __align__(16) float lds[];
  const ppo_mlp_problem& P = g.p;
  const int64_t row0 = static_cast<int64_t>(blockIdx.x) * kMlpRows;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int ldx = g.ldx;
  float* x = lds;
  float* y = lds + kMlpRows * ldx;
  mlp_input(P, x, ldx, row0, g.rows, tid);
  __syncthreads();
  for (int l = 0; l < P.num_layers; ++l) {
    const ppo_mlp_layer& L = P.layers[l];
    const bool last = l == P.num_layers - 1;
    mlp_run_layer<false>(L, last ? PPO_ACT_NONE : P.activation, x, ldx, {y, last ? P.out : nullptr, P.ldo, row0, g.rows}, 0,
                         mlp_tiles(L), wave, lane);
    __syncthreads();
    float* const t = x;
    x = y;
    y = t;
  }
}

// A launch of few rows leaves all but a few compute units idle and takes the time of one block's products and load
// latencies (16 rows of 48 -> [512, 256, 128] -> 12: 33 us in one launch, 10 of them fp32 MFMA).  Here each 16 rows have
// as many blocks as the pair's second layer has groups of four tiles, each computing the first layer for itself: two
// launches of 13.4 us for the four layers, no waits between blocks.
// Layers l0 (all of it, in LDS) and l0 + 1 (the block's slice of tiles, to global memory), or a slice of l0 alone.
__global__ __launch_bounds__(kMlpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void mlp_pairs_kernel(const MlpPairs a) {
  extern __shared__ __align__(16) float lds[];
  const ppo_mlp_problem& P = a.g.p;
  const int b = static_cast<int>(blockIdx.x), rb = b / a.slices, slice = b - rb * a.slices;
  const int64_t row0 = static_cast<int64_t>(rb) * kMlpRows, rows = a.g.rows;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int ldx = a.g.ldx;
  float* x = lds;
  float* y = lds + kMlpRows * ldx;
  if (a.in == nullptr) {
    mlp_input(P, x, ldx, row0, rows, tid);
  } else {  // a previous launch's rows, whole 16-byte pieces
    const int K = P.layers[a.l0].in_features, pieces = (K + 15) / 16 * 4;
    const int64_t ld = a.ld;
    for (int i = tid; i < kMlpRows * pieces; i += kMlpThreads) {
      const int r = i / pieces, c = 4 * (i - r * pieces);
      const f32x4 v = *reinterpret_cast<const f32x4*>(a.in + min(row0 + r, rows - 1) * ld + min(c, static_cast<int>(ld) - 4));
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = c + e < K ? v[e] : 0.0f;
      *reinterpret_cast<f32x4*>(x + r * ldx + c) = o;
    }
  }
  __syncthreads();
  int l = a.l0;
  if (l + 1 < P.num_layers) {
    mlp_run_layer<true>(P.layers[l], P.activation, x, ldx, {y, nullptr, 0, row0, rows}, 0, mlp_tiles(P.layers[l]), wave, lane);
    __syncthreads();
    x = y;
    ++l;
  }
  const bool last = l == P.num_layers - 1;
  const int t0 = slice * kSliceTiles, t1 = min(t0 + kSliceTiles, mlp_tiles(P.layers[l]));
  mlp_run_layer<true>(P.layers[l], last ? PPO_ACT_NONE : P.activation, x, ldx,
                      {nullptr, last ? P.out : a.to, last ? P.ldo : a.ld, row0, rows}, t0, t1, wave, lane);
}

int64_t round16(int64_t n) { return (n + 15) / 16 * 16; }

// The checked problem as kernel arguments.
int mlp_args(const ppo_mlp_problem* problem, int64_t rows, const char* who, MlpArgs& g) {
  int64_t widest = 0, width = 0;
  PPO_REQUIRE(problem != nullptr, "%s: no problem", who);
  PPO_REQUIRE(rows > 0 && rows <= INT32_MAX / 4, "%s: rows=%lld", who, (long long)rows);
  const ppo_mlp_problem& q = *problem;
  PPO_REQUIRE(q.num_blocks >= 1 && q.num_blocks <= PPO_MAX_MLP_BLOCKS && q.num_layers >= 1 &&
                  q.num_layers <= PPO_MAX_MLP_LAYERS,
              "%s: %d input blocks (at most %d), %d layers (at most %d)", who, q.num_blocks, PPO_MAX_MLP_BLOCKS,
              q.num_layers, PPO_MAX_MLP_LAYERS);
  PPO_REQUIRE(q.activation >= PPO_ACT_NONE && q.activation < PPO_ACT_COUNT, "%s: activation=%d", who, q.activation);
  PPO_REQUIRE((q.norm_mean == nullptr) == (q.norm_std == nullptr), "%s: one of mean / std", who);
  for (int s = 0; s < q.num_blocks; ++s) {
    PPO_REQUIRE(q.x[s].src && q.x[s].width > 0 && q.x[s].stride >= q.x[s].width, "%s: input block %d", who, s);
    width += q.x[s].width;
  }
  for (int l = 0; l < q.num_layers; ++l) {
    const ppo_mlp_layer& L = q.layers[l];
    PPO_REQUIRE(L.w && L.b && L.in_features == width && L.out_features > 0,
                "%s: layer %d: %d -> %d features after %lld", who, l, L.in_features, L.out_features, (long long)width);
    if (width > kMlpMaxWidth) return fail(PPO_EUNSUPPORTED, "%s: layers of at most %d features", who, kMlpMaxWidth);
    widest = std::max(widest, width);
    width = L.out_features;
  }
  PPO_REQUIRE(q.out && q.ldo >= width, "%s: output", who);
  g.p = q;
  g.rows = rows;
  g.blocks = static_cast<int>(ceil_div(rows, static_cast<int64_t>(kMlpRows)));
  // rows of whole 64 floats plus 4: a 16-byte read of the same columns of 16 rows falls on all 64 banks
  g.ldx = static_cast<int>((round16(widest) + 63) / 64 * 64 + 4);
  return PPO_OK;
}

template <typename K, typename A>
int launch_mlp(K kernel, int64_t blocks, const MlpArgs& g, const A& args, hipStream_t s, const char* name) {
  const size_t lds = 2 * static_cast<size_t>(kMlpRows) * g.ldx * sizeof(float);
  if (lds > 64 * 1024)
    PPO_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                      2 * kMlpRows * (kMlpMaxWidth + 4) * 4));
  PPO_REQUIRE(blocks <= INT32_MAX, "%s: too many rows", name);
  hipLaunchKernelGGL(kernel, dim3(static_cast<unsigned>(blocks)), dim3(kMlpThreads), lds, s, args);
  return check_launch(name);
}

// Floats per row of one of the two intermediate buffers: the widest layer of odd index but the last (0: none).
int64_t pairs_width(const ppo_mlp_problem& q) {
  int64_t w = 0;
  for (int l = 1; l + 1 < q.num_layers && l < PPO_MAX_MLP_LAYERS; l += 2)
    w = std::max<int64_t>(w, (q.layers[l].out_features + 3) / 4 * 4);
  return w;
}

}  // namespace
}  // namespace ppo

using namespace ppo;

extern "C" int ppo_mlp_fwd(const ppo_mlp_problem* problem, int64_t rows, ppo_stream_t stream) {
  MlpArgs g{};
  if (int rc = mlp_args(problem, rows, "ppo_mlp_fwd", g)) return rc;
  return launch_mlp(mlp_fwd_kernel, g.blocks, g, g, static_cast<hipStream_t>(stream), "mlp_fwd_kernel");
}

extern "C" size_t ppo_mlp_fwd_pairs_workspace_bytes(const ppo_mlp_problem* problem, int64_t rows) {
  if (problem == nullptr || rows <= 0) return 0;
  return 2 * static_cast<size_t>(pairs_width(*problem)) * static_cast<size_t>(rows) * sizeof(float);
}

extern "C" int ppo_mlp_fwd_pairs(const ppo_mlp_problem* problem, int64_t rows, void* workspace, size_t workspace_bytes,
                                 ppo_stream_t stream) {
  MlpPairs a{};
  if (int rc = mlp_args(problem, rows, "ppo_mlp_fwd_pairs", a.g)) return rc;
  const ppo_mlp_problem& q = *problem;
  const size_t need = ppo_mlp_fwd_pairs_workspace_bytes(problem, rows);
  PPO_REQUIRE(need == 0 || (workspace != nullptr && workspace_bytes >= need && reinterpret_cast<uintptr_t>(workspace) % 16 == 0),
              "ppo_mlp_fwd_pairs: workspace of %zu bytes (%zu, 16-byte aligned, needed)", workspace_bytes, need);
  a.ld = pairs_width(q);
  float* const ws = static_cast<float*>(workspace);
  float* const buf[2] = {ws, ws == nullptr ? nullptr : ws + rows * a.ld};
  for (int l0 = 0, p = 0; l0 < q.num_layers; l0 += 2, ++p) {
    const int l = std::min(l0 + 1, q.num_layers - 1);  // the sliced layer
    a.in = p == 0 ? nullptr : buf[(p - 1) & 1];
    a.to = buf[p & 1];
    a.slices = static_cast<int>(ceil_div(ceil_div(q.layers[l].out_features, 16), kSliceTiles));
    a.l0 = l0;
    const int64_t blocks = static_cast<int64_t>(a.g.blocks) * a.slices;
    if (int rc = launch_mlp(mlp_pairs_kernel, blocks, a.g, a, static_cast<hipStream_t>(stream), "mlp_pairs_kernel")) return rc;
  }
  return PPO_OK;
}
