// Rollout-side Gaussian head (rsl_rl/algorithms/ppo.py:124-135 act(); rsl_rl/modules/distribution.py:183-232):
// std = clamp/exp of the std parameter, actions = noise * std + mean (torch.normal(mean, std) draws a standard
// normal and scales it), log_prob of the actions summed over the action dimension, and the per-row std copy the
// rollout storage keeps as distribution_params[1].  The standard-normal noise is drawn by the caller.
// And the rollout storage's writes of one env step (rsl_rl/storage/rollout_storage.py:173-205) as one launch.
#include "common.hpp"

#pragma clang fp contract(off)

namespace ppo {
namespace {

constexpr double kLogSqrt2Pi = 0.91893853320467274178;

struct SampleArgs {
  const float* mean; int64_t ld_mean;
  const float* std_param; int32_t std_type; float std_lo, std_hi;
  const float* noise; int64_t ld_noise;     // NULL: actions are given in `actions` (log-prob only)
  float* actions; int64_t ld_actions;
  float* logp;                              // [rows] or NULL
  float* std_out; int64_t ld_std;           // [rows, A] or NULL
  int64_t rows; int32_t A;
};

// A block takes kSampleRows rows: the elements are spread over the threads in memory order (a thread per row, used
// before, read and wrote 64 rows' lines per instruction and ran 16 blocks for 4,096 rows: 16.6 us at 29 actions, this
// one 8.1 us), their log-density terms pass through LDS, and one thread per row adds them in fp64 in the actions'
// order.
constexpr int kSampleRows = 32;

__global__ __launch_bounds__(256) void gauss_sample_kernel(const SampleArgs a) {
  __shared__ float s_std[PPO_MAX_ACTIONS], s_var[PPO_MAX_ACTIONS], s_log[PPO_MAX_ACTIONS];
  __shared__ float s_t[kSampleRows * (PPO_MAX_ACTIONS + 1)];
  for (int j = threadIdx.x; j < a.A; j += blockDim.x) {
    float sd, lg;
    std_from_param(a.std_param[j], a.std_type, a.std_lo, a.std_hi, sd, lg);
    s_std[j] = sd;
    s_var[j] = sd * sd;
    s_log[j] = lg;
  }
  __syncthreads();
  const int64_t r0 = static_cast<int64_t>(blockIdx.x) * kSampleRows;
  const int rows = static_cast<int>(min(static_cast<int64_t>(kSampleRows), a.rows - r0));
  const int pitch = a.A | 1;  // odd: the row sums' reads fall on different banks
  const float c_lp = static_cast<float>(kLogSqrt2Pi);
  for (int e = threadIdx.x; e < rows * a.A; e += blockDim.x) {
    const int i = e / a.A, j = e - i * a.A;
    const int64_t r = r0 + i;
    const float mu = a.mean[r * a.ld_mean + j];
    float x;
    if (a.noise != nullptr) {
      x = a.noise[r * a.ld_noise + j] * s_std[j] + mu;
      a.actions[r * a.ld_actions + j] = x;
    } else {
      x = a.actions[r * a.ld_actions + j];
    }
    const float d = x - mu;
    float t = -(d * d) / (2.0f * s_var[j]);
    t = t - s_log[j];
    s_t[i * pitch + j] = t - c_lp;
    if (a.std_out != nullptr) a.std_out[r * a.ld_std + j] = s_std[j];
  }
  if (a.logp == nullptr) return;
  __syncthreads();
  if (static_cast<int>(threadIdx.x) < rows) {
    double lp = 0.0;
    for (int j = 0; j < a.A; ++j) lp += static_cast<double>(s_t[threadIdx.x * pitch + j]);
    a.logp[r0 + threadIdx.x] = static_cast<float>(lp);
  }
}

// The writes of one transition, each a [rows, width] block (ppo_store_item): block b of an item takes kStorePer
// elements of it, or of its 16-byte pieces where both sides are whole 16-byte pieces without gaps.  A few MB: what
// bounds it is the launch, so all of a step's writes share one (as a torch copy each they were 11 to 13 launches of 2 to 5 us
// and 5 us of host time; 24 env steps of 4,096 humanoid envs, with act()'s distribution in one launch instead of three:
// 9.98 -> 8.60 ms, of which the noise's draw on the CPU is 5.6; this kernel 5.9 us a step).
constexpr int kStoreThreads = 256, kStorePer = 4 * kStoreThreads;

struct StoreGroup {
  ppo_store_item it[PPO_MAX_STORE_ITEMS];
  int32_t block_begin[PPO_MAX_STORE_ITEMS];
  int32_t vec;  // bit i: item i moves as 16-byte pieces
  int32_t count;
};
static_assert(sizeof(StoreGroup) <= 4096, "kernel arguments");

// torch's conversion to uint8 goes through int64
__device__ __forceinline__ uint8_t to_u8(float x) { return static_cast<uint8_t>(static_cast<int64_t>(x)); }

__device__ __forceinline__ float flag_value(const void* p, int type, int64_t i) {
  return type == PPO_STORE_T_F32  ? static_cast<const float*>(p)[i]
         : type == PPO_STORE_T_U8 ? static_cast<float>(static_cast<const uint8_t*>(p)[i])
                                  : static_cast<float>(static_cast<const int64_t*>(p)[i]);
}

__global__ __launch_bounds__(kStoreThreads) void store_rows_kernel(const StoreGroup g) {
  int i = 0;
  for (int k = 1; k < g.count; ++k)
    if (static_cast<int>(blockIdx.x) >= g.block_begin[k]) i = k;
  const ppo_store_item& it = g.it[i];
  const bool vec = (g.vec >> i) & 1;
  const uint32_t w = static_cast<uint32_t>(it.width);
  const uint32_t n = static_cast<uint32_t>(it.rows) * w >> (vec ? 2 : 0);
  const uint32_t first = static_cast<uint32_t>(static_cast<int>(blockIdx.x) - g.block_begin[i]) * kStorePer + threadIdx.x;
#pragma unroll
  for (int u = 0; u < kStorePer / kStoreThreads; ++u) {
    const uint32_t e = first + u * kStoreThreads;
    if (e >= n) return;
    if (vec) {
      static_cast<float4*>(it.dst)[e] = static_cast<const float4*>(it.src)[e];
      continue;
    }
    const uint32_t r = e / w, c = e - r * w;
    const int64_t si = static_cast<int64_t>(r) * it.src_stride + c, di = static_cast<int64_t>(r) * it.dst_stride + c;
    switch (it.kind) {
      case PPO_STORE_F32:
        static_cast<float*>(it.dst)[di] = static_cast<const float*>(it.src)[si];
        break;
      case PPO_STORE_U8: {
        uint8_t v;
        if (it.type == PPO_STORE_T_F32) v = to_u8(static_cast<const float*>(it.src)[si]);
        else if (it.type == PPO_STORE_T_U8) v = static_cast<const uint8_t*>(it.src)[si];
        else v = static_cast<uint8_t>(static_cast<const int64_t*>(it.src)[si]);
        static_cast<uint8_t*>(it.dst)[di] = v;
        break;
      }
      default: {  // PPO_STORE_BOOTSTRAP (width 1)
        const float boot = it.gamma * (it.value[r] * flag_value(it.flag, it.type, r));
        static_cast<float*>(it.dst)[di] = static_cast<const float*>(it.src)[si] + boot;
      }
    }
  }
}

}  // namespace
}  // namespace ppo

using namespace ppo;

extern "C" int ppo_gauss_sample(const float* mean, int64_t ld_mean, const float* std_param, int32_t std_type,
                                double std_lo, double std_hi, const float* noise, int64_t ld_noise, float* actions,
                                int64_t ld_actions, float* logp, float* std_out, int64_t ld_std, int64_t rows,
                                int32_t num_actions, ppo_stream_t stream) {
  PPO_REQUIRE(mean && std_param && actions, "ppo_gauss_sample: null pointer");
  PPO_REQUIRE(rows > 0 && num_actions > 0 && num_actions <= PPO_MAX_ACTIONS, "ppo_gauss_sample: rows=%lld A=%d",
              (long long)rows, num_actions);
  PPO_REQUIRE(std_type == PPO_STD_LOG || std_type == PPO_STD_SCALAR, "ppo_gauss_sample: std_type=%d", std_type);
  PPO_REQUIRE(ld_mean >= num_actions && ld_actions >= num_actions && (noise == nullptr || ld_noise >= num_actions) &&
                  (std_out == nullptr || ld_std >= num_actions),
              "ppo_gauss_sample: bad leading dimension");
  SampleArgs a{mean, ld_mean, std_param, std_type, static_cast<float>(std_lo), static_cast<float>(std_hi), noise,
               ld_noise, actions, ld_actions, logp, std_out, ld_std, rows, num_actions};
  const int64_t blocks = ceil_div(rows, static_cast<int64_t>(kSampleRows));
  PPO_REQUIRE(blocks <= INT32_MAX, "ppo_gauss_sample: too many rows");
  hipLaunchKernelGGL(gauss_sample_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  return check_launch("gauss_sample_kernel");
}

extern "C" int ppo_store_rows(const ppo_store_item* items, int32_t count, ppo_stream_t stream) {
  PPO_REQUIRE(items != nullptr && count >= 1 && count <= PPO_MAX_STORE_ITEMS, "ppo_store_rows: count=%d outside [1, %d]",
              count, PPO_MAX_STORE_ITEMS);
  StoreGroup g{};
  int64_t blocks = 0;
  for (int i = 0; i < count; ++i) {
    const ppo_store_item& q = items[i];
    PPO_REQUIRE(q.src && q.dst && q.rows > 0 && q.width > 0, "ppo_store_rows: item %d: null pointer or empty", i);
    PPO_REQUIRE(q.src_stride >= q.width && q.dst_stride >= q.width, "ppo_store_rows: item %d: bad stride", i);
    PPO_REQUIRE(q.rows <= INT32_MAX / q.width, "ppo_store_rows: item %d: %lld x %d elements (at most 2^31 - 1)", i,
                (long long)q.rows, q.width);
    PPO_REQUIRE(q.kind >= PPO_STORE_F32 && q.kind <= PPO_STORE_BOOTSTRAP && q.type >= PPO_STORE_T_F32 &&
                    q.type <= PPO_STORE_T_I64,
                "ppo_store_rows: item %d: kind=%d type=%d", i, q.kind, q.type);
    PPO_REQUIRE(q.kind != PPO_STORE_BOOTSTRAP || (q.value && q.flag && q.width == 1),
                "ppo_store_rows: item %d: a bootstrapped reward needs its values and flags, one per row", i);
    g.it[i] = q;
    const int64_t n = q.rows * q.width;
    const bool flat = (q.src_stride == q.width && q.dst_stride == q.width) || q.rows == 1;
    const bool vec = q.kind == PPO_STORE_F32 && flat && n % 4 == 0 && reinterpret_cast<uintptr_t>(q.src) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(q.dst) % 16 == 0;
    if (vec) g.vec |= 1 << i;
    g.block_begin[i] = static_cast<int32_t>(blocks);
    blocks += ceil_div(vec ? n / 4 : n, static_cast<int64_t>(kStorePer));
  }
  g.count = count;
  hipLaunchKernelGGL(store_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kStoreThreads), 0,
                     static_cast<hipStream_t>(stream), g);
  return check_launch("store_rows_kernel");
}
