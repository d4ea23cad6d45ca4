// A whole MLP forward in one launch, for the rollout side (rsl_rl/models/mlp_model.py:82-118): concatenate the
// observation groups, normalise them (rsl_rl/modules/normalization.py:46-48), and run every linear layer with its
// activation (rsl_rl/modules/mlp.py:91-95).
//
// What bounds it is latency: a policy step of a few thousand rows is 0.1 to 3 GFLOP, and as one launch per layer it spent
// its time on launches, on the host calls before them and on GEMM tiles that filled a fraction of the chip (4,096 rows x
// [512, 256, 128], actor: normaliser and four GEMMs 80 us of kernel time and 94 us of host time).  Here a block takes 16
// rows through all layers: the rows' activations stay in LDS (two buffers), the weights come from the caches straight
// into the MFMA operand registers, 64 k ahead, and nothing is written but the output: one launch of 34 us for 16 to
// 1,024 rows, 37 for 4,096 (37 / 44 us with 96 normalised inputs and 29 actions; the layers one by one 64 / 77 us).  16 rows give 4,096 rows 256 blocks, one per
// compute unit.  v_mfma_f32_16x16x4f32 with the weights as the first operand leaves each lane 4 consecutive outputs of one
// row: one 16-byte LDS store each.  Past some thousands of rows the layers' own GEMMs (weights read once per 128 rows, bf16
// matrix cores) are faster: the caller's choice.
#include "gemm_core.hpp"

namespace ppo {
namespace {

constexpr int kMlpRows = 16, kMlpWaves = 8, kMlpThreads = 64 * kMlpWaves;
constexpr int kMlpMaxWidth = 1024;

struct MlpGroup {
  ppo_mlp_problem p[PPO_MAX_MLP_PROBLEMS];
  int32_t count, blocks;  // blocks per problem
  int32_t ldx;            // floats per LDS row
  int64_t rows;
};
static_assert(sizeof(MlpGroup) <= 4096, "kernel arguments");

// One layer for the block's 16 rows: x [16][ldx] (columns past K up to the next multiple of 16 zero) -> y, or the
// output.  TILES 16-wide output tiles per wave at a time.  (Deeper prefetch, eight k-groups and the next tiles' first
// chunk at two waves per SIMD, measured 44 us against 34 for 16 rows of 48 -> [512, 256, 128] -> 12.)
template <int TILES, bool VEC>
__device__ __forceinline__ void mlp_layer(const ppo_mlp_layer& L, bool last, int act, const float* x, float* y, int ldx,
                                          float* out, int64_t ldo, int64_t row0, int64_t rows, int wave, int lane) {
  const int K = L.in_features, N = L.out_features;
  const int m = lane & 15, q = lane >> 4;
  const int groups = (K + 15) >> 4, tiles = (N + 15) >> 4;
  constexpr int AH = 4;  // k-groups of 16 loaded ahead
  for (int t0 = wave * TILES; t0 < tiles; t0 += kMlpWaves * TILES) {
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
#pragma unroll
    for (int j = 0; j < TILES; ++j) {
      const int n = 16 * (t0 + j) + 4 * q;
      if (16 * (t0 + j) >= N) continue;
      f32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float z = acc[j][0][e] + acc[j][1][e] + L.b[min(n + e, N - 1)];
        o[e] = n + e >= N ? 0.0f : last ? z : act == PPO_ACT_ELU ? elu_fast(z) : act_fwd(act, z);
      }
      if (!last) {
        *reinterpret_cast<f32x4*>(y + m * ldx + n) = o;
      } else if (row0 + m < rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < N) out[(row0 + m) * ldo + n + e] = o[e];
      }
    }
  }
}

__global__ __launch_bounds__(kMlpThreads) __attribute__((amdgpu_waves_per_eu(4, 4))) void mlp_fwd_kernel(const MlpGroup g) {
  extern __shared__ __align__(16) float lds[];
  const int pi = static_cast<int>(blockIdx.x) >= g.blocks ? 1 : 0;
  const ppo_mlp_problem& P = g.p[pi];
  const int64_t row0 = static_cast<int64_t>(static_cast<int>(blockIdx.x) - pi * g.blocks) * kMlpRows;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int ldx = g.ldx;
  float* x = lds;
  float* y = lds + kMlpRows * ldx;
  // the input rows: 32 threads per row, the blocks side by side, normalised as ppo_obs_normalize does
  {
    const int r = tid >> 5, c0 = tid & 31;
    const int64_t row = row0 + r;
    int col = 0;
    for (int s = 0; s < P.num_blocks; ++s) {
      const ppo_column_block& B = P.x[s];
      for (int c = c0; c < B.width; c += 32) {
        float v = row < g.rows ? B.src[row * B.stride + c] : 0.0f;
        if (P.norm_mean != nullptr) v = (v - P.norm_mean[col + c]) / (P.norm_std[col + c] + P.norm_eps);
        x[r * ldx + col + c] = v;
      }
      col += B.width;
    }
    for (int c = col + c0; c < (col + 15) / 16 * 16; c += 32) x[r * ldx + c] = 0.0f;
  }
  __syncthreads();
  for (int l = 0; l < P.num_layers; ++l) {
    const ppo_mlp_layer& L = P.layers[l];
    const bool last = l == P.num_layers - 1;
    const bool vec = L.in_features % 4 == 0 && reinterpret_cast<uintptr_t>(L.w) % 16 == 0;
    const bool wide = L.out_features > 16 * kMlpWaves;
    auto run = [&](auto tiles_c, auto vec_c) __attribute__((always_inline)) {
      mlp_layer<decltype(tiles_c)::value, decltype(vec_c)::value>(L, last, P.activation, x, y, ldx, P.out, P.ldo, row0,
                                                                  g.rows, wave, lane);
    };
    if (vec) {
      if (wide) run(IntC<2>{}, BoolC<true>{});
      else run(IntC<1>{}, BoolC<true>{});
    } else {
      run(IntC<1>{}, BoolC<false>{});
    }
    __syncthreads();
    float* const t = x;
    x = y;
    y = t;
  }
}

int64_t round16(int64_t n) { return (n + 15) / 16 * 16; }

}  // namespace
}  // namespace ppo

using namespace ppo;

extern "C" int ppo_mlp_fwd(const ppo_mlp_problem* problems, int32_t count, int64_t rows, ppo_stream_t stream) {
  PPO_REQUIRE(problems != nullptr && count >= 1 && count <= PPO_MAX_MLP_PROBLEMS, "ppo_mlp_fwd: count=%d outside [1, %d]",
              count, PPO_MAX_MLP_PROBLEMS);
  PPO_REQUIRE(rows > 0 && rows <= INT32_MAX / 4, "ppo_mlp_fwd: rows=%lld", (long long)rows);
  MlpGroup g{};
  int64_t widest = 0;
  for (int i = 0; i < count; ++i) {
    const ppo_mlp_problem& q = problems[i];
    PPO_REQUIRE(q.num_blocks >= 1 && q.num_blocks <= PPO_MAX_MLP_BLOCKS && q.num_layers >= 1 &&
                    q.num_layers <= PPO_MAX_MLP_LAYERS,
                "ppo_mlp_fwd: problem %d: %d input blocks (at most %d), %d layers (at most %d)", i, q.num_blocks,
                PPO_MAX_MLP_BLOCKS, q.num_layers, PPO_MAX_MLP_LAYERS);
    PPO_REQUIRE(q.activation >= PPO_ACT_NONE && q.activation < PPO_ACT_COUNT, "ppo_mlp_fwd: activation=%d", q.activation);
    PPO_REQUIRE((q.norm_mean == nullptr) == (q.norm_std == nullptr), "ppo_mlp_fwd: problem %d: one of mean / std", i);
    int64_t width = 0;
    for (int s = 0; s < q.num_blocks; ++s) {
      PPO_REQUIRE(q.x[s].src && q.x[s].width > 0 && q.x[s].stride >= q.x[s].width, "ppo_mlp_fwd: problem %d: input block %d",
                  i, s);
      width += q.x[s].width;
    }
    for (int l = 0; l < q.num_layers; ++l) {
      const ppo_mlp_layer& L = q.layers[l];
      PPO_REQUIRE(L.w && L.b && L.in_features == width && L.out_features > 0,
                  "ppo_mlp_fwd: problem %d layer %d: %d -> %d features after %lld", i, l, L.in_features, L.out_features,
                  (long long)width);
      if (width > kMlpMaxWidth) return fail(PPO_EUNSUPPORTED, "ppo_mlp_fwd: layers of at most %d features", kMlpMaxWidth);
      widest = std::max(widest, width);
      width = L.out_features;
    }
    PPO_REQUIRE(q.out && q.ldo >= width, "ppo_mlp_fwd: problem %d output", i);
    g.p[i] = q;
  }
  g.count = count;
  g.rows = rows;
  g.blocks = static_cast<int>(ceil_div(rows, static_cast<int64_t>(kMlpRows)));
  // rows of whole 64 floats plus 4: a 16-byte read of the same columns of 16 rows falls on all 64 banks
  g.ldx = static_cast<int>((round16(widest) + 63) / 64 * 64 + 4);
  const size_t lds = 2 * static_cast<size_t>(kMlpRows) * g.ldx * sizeof(float);
  if (lds > 64 * 1024)
    PPO_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(mlp_fwd_kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, 2 * kMlpRows * (kMlpMaxWidth + 4) * 4));
  hipLaunchKernelGGL(mlp_fwd_kernel, dim3(count * g.blocks), dim3(kMlpThreads), lds, static_cast<hipStream_t>(stream), g);
  return check_launch("mlp_fwd_kernel");
}
