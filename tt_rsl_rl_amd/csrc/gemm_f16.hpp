// fp32-accurate GEMMs on the fp16 matrix cores for operands whose largest magnitude is known (fp16x3), and the
// bf16-operand mode's kernels, which share their structure.  See gemm.hip for the dispatch.
//
// fp16x3.  Every operand element x is scaled by a power of two s (one per tensor: its largest |x| lands in
// [2^14, 2^15)) and split into two fp16 parts, hi = fp16(s x) and lo = fp16(2^11 (s x - hi)), both rounded to nearest:
// s x = hi + 2^-11 lo with a residual of at most 2^-23 |s x| (2^-24 on average), and of at most 2^-36 where lo is
// subnormal, i.e. 2^-50 of the tensor's largest value (what that means for a tensor of wide range: amax.hpp).  A product
// is taken as hi.hi + 2^-11 (hi.lo + lo.hi): three MFMAs, the hi.hi sums in one accumulator and the cross terms in another
// (added at the end, in fp32); the left-out lo.lo is at most 2^-22 of the product and 2^-24 on average.  This is the
// published scheme of Ootomo and Yokota
// ("Recovering single precision accuracy from Tensor Cores while surpassing the FP32 theoretical peak performance",
// IJHPCA 2022) with the scaling made explicit.  Against bf16x6 (gemm_core.hpp) it issues half the MFMAs, moves two
// 16-bit planes through LDS instead of three and splits in 6 VALU instructions per pair of elements instead of 11; its
// sums round a third as often into the main accumulator, so its error is no larger (measured against fp64 in
// tests/test_gpu_ranged.py).  What it needs is a bound on |x|: the kernels that write the operands leave it behind
// (kAmaxSlots slots with the tensor's range, raised by atomic maxima per wave).
#pragma once

#include "amax.hpp"
#include "gemm_core.hpp"

namespace ppo {
namespace {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// hi and lo parts of two elements, packed (element 0 in the low half): v_fma_mix reads and writes fp16 halves with
// fp32 arithmetic in between, so the scaling costs nothing and s x - hi is exact.
__device__ __forceinline__ void split_f16x2(float x0, float x1, float s, float k2048, uint32_t& hi, uint32_t& lo) {
  float r0, r1;
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(hi) : "v"(x0), "s"(s));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(hi) : "v"(x1), "s"(s));
  asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel_hi:[0,0,1]" : "=v"(r0) : "v"(x0), "s"(s), "v"(hi));
  asm("v_fma_mix_f32 %0, %1, %2, -%3 op_sel:[0,0,1] op_sel_hi:[0,0,1]" : "=v"(r1) : "v"(x1), "s"(s), "v"(hi));
  asm("v_fma_mixlo_f16 %0, %1, %2, 0" : "=v"(lo) : "v"(r0), "s"(k2048));
  asm("v_fma_mixhi_f16 %0, %1, %2, 0" : "+v"(lo) : "v"(r1), "s"(k2048));
}

// How a kernel's operands reach the matrix cores.
enum Arith : int {
  ARITH_F16X3 = 0,  // two fp16 parts, three products, two accumulators
  ARITH_BF16 = 1,   // bf16 operands (PPO_GEMM_BF16_OPERANDS): one part, one product
  ARITH_BF16X6 = 2, // three bf16 parts, six products (gemm_core.hpp): problems whose operands span too much for fp16x3
};

template <int AR>
struct Parts {
  static constexpr int planes = AR == ARITH_F16X3 ? 2 : AR == ARITH_BF16X6 ? 3 : 1;
  static constexpr int accs = AR == ARITH_F16X3 ? 2 : 1;
  static constexpr int products = AR == ARITH_F16X3 ? 3 : AR == ARITH_BF16X6 ? 6 : 1;
};

// Splits 4 consecutive elements and writes each part's 8 bytes (at c and c + plane).
template <int AR>
__device__ __forceinline__ void stage_piece(const f32x4& v, float s, float k2048, unsigned char* c, int plane) {
  if constexpr (AR == ARITH_F16X3) {
    uint32_t h[2], l[2];
    split_f16x2(v[0], v[1], s, k2048, h[0], l[0]);
    split_f16x2(v[2], v[3], s, k2048, h[1], l[1]);
    *reinterpret_cast<u32x2*>(c) = u32x2{h[0], h[1]};
    *reinterpret_cast<u32x2*>(c + plane) = u32x2{l[0], l[1]};
  } else if constexpr (AR == ARITH_BF16X6) {
    uint32_t h[2], m[2], l[2];
    split_bf16x3(v[0], v[1], h[0], m[0], l[0]);
    split_bf16x3(v[2], v[3], h[1], m[1], l[1]);
    *reinterpret_cast<u32x2*>(c) = u32x2{h[0], h[1]};
    *reinterpret_cast<u32x2*>(c + plane) = u32x2{m[0], m[1]};
    *reinterpret_cast<u32x2*>(c + 2 * plane) = u32x2{l[0], l[1]};
  } else {
    *reinterpret_cast<u32x2*>(c) = u32x2{round_bf16x2(v[0], v[1]), round_bf16x2(v[2], v[3])};
  }
}

template <int AR>
__device__ __forceinline__ f32x16 mfma16(const u32x4& a, const u32x4& b, const f32x16& c) {
  if constexpr (AR == ARITH_F16X3)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The products of one 16-deep k-group of a (TM x TN)-tile wave: cross terms into acc[1], hi.hi (or the only part's)
// into acc[0].  NTF: the second operand first (accumulators hold the tile transposed).
template <int AR, int TM, int TN, bool FLIP>
__device__ __forceinline__ void products(f32x16 (&acc)[Parts<AR>::accs][TM][TN], const u32x4 (&fa)[TM][Parts<AR>::planes],
                                         const u32x4 (&fb)[TN][Parts<AR>::planes], int t) {
  constexpr int pa[3] = {1, 0, 0}, pb[3] = {0, 1, 0};
  constexpr int pa6[6] = {2, 1, 0, 1, 0, 0}, pb6[6] = {0, 1, 2, 0, 1, 0};  // (small terms first, as gemm_core.hpp's)
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      if constexpr (AR == ARITH_F16X3) {
        f32x16& c = acc[t < 2 ? 1 : 0][i][j];
        c = FLIP ? mfma16<AR>(fb[j][pb[t]], fa[i][pa[t]], c) : mfma16<AR>(fa[i][pa[t]], fb[j][pb[t]], c);
      } else if constexpr (AR == ARITH_BF16X6) {
        f32x16& c = acc[0][i][j];
        c = FLIP ? mfma16<AR>(fb[j][pb6[t]], fa[i][pa6[t]], c) : mfma16<AR>(fa[i][pa6[t]], fb[j][pb6[t]], c);
      } else {
        f32x16& c = acc[0][i][j];
        c = FLIP ? mfma16<AR>(fb[j][0], fa[i][0], c) : mfma16<AR>(fa[i][0], fb[j][0], c);
      }
    }
}

// acc[0] += 2^-11 acc[1]
template <int AR, int TM, int TN>
__device__ __forceinline__ void join_acc(f32x16 (&acc)[Parts<AR>::accs][TM][TN]) {
  if constexpr (AR == ARITH_F16X3) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v)
          acc[0][i][j][v] = __builtin_fmaf(acc[1][i][j][v], 0x1p-11f, acc[0][i][j][v]);
  }
}

// ------------------------------------------------------------------------------------------------------------------
// NT: C[m,n] = sum_k A[m,k] B[n,k] (forward), or B k-major (BKM: the weights of an input-grad as stored).  One
// 128 x BN tile per block, WM x 2 waves of 128 / WM x BN / 2; 32-deep k-slabs, two LDS stages.  A staged row is read by
// eight lanes, 16 bytes each: whole 128-byte lines.  Slab s + 1 is loaded into registers while slab s's first k-group
// multiplies and is split into the other stage between the MFMAs of its second.  Columns past K (K need not be a
// multiple of anything) are staged as zeros: their loads are clamped to the row's last 16 bytes.
// LDS planes: [row][32 k] halves, the 16-byte chunk index XOR-ed with (row / 4) % 4 (the 16 rows that a ds_read_b128
// serves at a time fall on all 64 banks); BKM's B: [32 k][BN n], as the weight-grad's.
// ------------------------------------------------------------------------------------------------------------------
// fp16x3: a problem with an operand that is not narrow() (amax.hpp) takes its tiles in bf16x6, one slab at a time, three
// planes in the memory of the two stages.  It is there for outliers, and a function of its own so that the usual path keeps
// its registers (as a branch with a loop inside the kernel it cost 17 to 22 spilled ones; as a launch of its own after each
// of these, 3 us and a gap where there is nothing to do).  98,304 rows, 240 -> 512, with an outlier / without / the plain
// kernels: forward 201 / 144 / 164 us, input-grad 179 / 139 / 162, weight-grad 196 / 143 / 162.
using LdsBytes = __attribute__((address_space(3))) unsigned char;
using GroupArgument = const __attribute__((address_space(4))) Group;
template <int BN, int WM, int EPI, bool BKM>
__device__ __attribute__((noinline)) void nt_wide_tile(uint64_t group, LdsBytes* lds);
template <int BN, int WM>
__device__ __attribute__((noinline)) void tn_wide_tile(uint64_t group, LdsBytes* lds);

// Where a kernel whose first argument is a Group finds it: for the functions it calls (evaluated in the kernel itself: the
// kernel-argument pointer is null in a called function).
__device__ __forceinline__ uint64_t group_argument() {
  return reinterpret_cast<uint64_t>((const void*)__builtin_amdgcn_kernarg_segment_ptr());
}
// The same in the called function, with a wave-uniform address.
__device__ __forceinline__ const Group& group_at(uint64_t address) {
  const uint64_t lo = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address)));
  const uint64_t hi = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<uint32_t>(address >> 32)));
  return *(const Group*)(GroupArgument*)((hi << 32) | lo);
}

template <int BN, int WM, int EPI, bool BKM, int AR>
__device__ __forceinline__ void nt_f16_tile(const Group& g, unsigned char* lds) {
  static_assert(EPI == EPI_BIAS || epi_fwd_act(EPI) || epi_act_grad(EPI) || EPI == EPI_STORE, "NT epilogues");
  constexpr int BM = 128, BK = 32, THREADS = WM * 128, TM = 4 / WM, TN = BN / 64, NPL = Parts<AR>::planes;
  constexpr int PLANE_A = BM * BK * 2, PLANE_B = BN * BK * 2;
  constexpr int STAGE = NPL * (PLANE_A + PLANE_B);
  constexpr int PS = 36;

  const TileCoord tc = locate(g);
  const Problem& P = g.p[tc.pi];
  const int64_t lda = P.lda, ldb = P.ldb;
  const int row0 = tc.tm * BM, col0 = tc.tn * BN;
  const int M = P.M, N = P.N, K = P.K;
  const int nk = (K + BK - 1) / BK;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int wm = wave >> 1, wn = wave & 1;

  constexpr int RPP = THREADS / 8, NA = BM / RPP, NB = BN / RPP;
  static_assert(NA >= 1 && NB >= 1, "staging passes");
  const int sr = tid >> 3, sq = tid & 7;  // staged row (+ RPP i), 4-column piece of the slab
  constexpr int CPR = BN / 4, KPP = THREADS / CPR;  // BKM: pieces per k-row, k-rows per pass
  const int bsc = tid % CPR, bsk = tid / CPR;
  const unsigned char* const Ab = reinterpret_cast<const unsigned char*>(P.A);
  const unsigned char* const Bb = reinterpret_cast<const unsigned char*>(P.B);
  uint32_t aoff[NA], boff[NB];  // byte offsets of the lane's rows (operands span less than 4 GiB)
  int la[NA], lb[NB];           // its places in a plane
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    const int r = sr + RPP * i;
    aoff[i] = static_cast<uint32_t>(static_cast<int64_t>(min(row0 + r, M - 1)) * lda * 4);
    la[i] = r * 64 + 16 * ((sq >> 1) ^ ((r >> 2) & 3)) + 8 * (sq & 1);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    if constexpr (BKM) {
      const int kr = bsk + KPP * i;
      boff[i] = static_cast<uint32_t>(min(col0 + 4 * bsc, ((N - 1) >> 2) << 2) * 4);
      lb[i] = tn_chunk_off<BN>(kr, bsc);
    } else {
      const int r = sr + RPP * i;
      boff[i] = static_cast<uint32_t>(static_cast<int64_t>(min(col0 + r, N - 1)) * ldb * 4);
      lb[i] = r * 64 + 16 * ((sq >> 1) ^ ((r >> 2) & 3)) + 8 * (sq & 1);
    }
  }
  const uint32_t ldb4 = static_cast<uint32_t>(ldb * 4);
  const int kc_last = ((K - 1) >> 2) << 2;  // first column of a row's last 16 bytes
  f32x4 va[NA], vb[NB];
  // one piece of slab kt (the look-ahead past the end re-reads the row's last columns)
  auto load_piece = [&](int kt, int o) __attribute__((always_inline)) {
    const int k0 = kt * BK;
    const uint32_t kc = static_cast<uint32_t>(min(k0 + 4 * sq, kc_last) * 4);
    if (o < NA) {
      va[o < NA ? o : 0] = *reinterpret_cast<const f32x4*>(Ab + (aoff[o < NA ? o : 0] + kc));
    } else {
      const int i = o < NA ? 0 : o - NA;
      if constexpr (BKM) {
        const uint32_t kr = static_cast<uint32_t>(min(k0 + bsk + KPP * i, K - 1));  // (rows past K meet zeros of A)
        vb[i] = *reinterpret_cast<const f32x4*>(Bb + (kr * ldb4 + boff[i]));
      } else {
        vb[i] = *reinterpret_cast<const f32x4*>(Bb + (boff[i] + kc));
      }
    }
  };
  // columns at or past K of the last slab become zeros
  auto mask_tail = [&](int kt) __attribute__((always_inline)) {
    if ((kt + 1) * BK <= K) return;
    const int left = K - kt * BK - 4 * sq;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = e < left;
#pragma unroll
      for (int i = 0; i < NA; ++i) va[i][e] = in ? va[i][e] : 0.0f;
      if constexpr (!BKM) {
#pragma unroll
        for (int i = 0; i < NB; ++i) vb[i][e] = in ? vb[i][e] : 0.0f;
      }
    }
  };
#pragma unroll
  for (int o = 0; o < NA + NB; ++o) load_piece(0, o);
  int ea = 0, eb = 0;
  if constexpr (AR == ARITH_F16X3) {
    const Range ra = load_range(P.amax_a, lane), rb = load_range(P.amax_b, lane);
    if (!ra.narrow() || !rb.narrow()) {
      nt_wide_tile<BN, WM, EPI, BKM>(group_argument(), (LdsBytes*)lds);
      return;
    }
    ea = amax_exponent(ra.top);
    eb = amax_exponent(rb.top);
  }
  const float sa = pow2(ea), sb = pow2(eb);
  const float k2048 = 2048.0f;
  auto split_piece = [&](unsigned char* st, int o) __attribute__((always_inline)) {
    if (o < NA)
      stage_piece<AR>(va[o < NA ? o : 0], sa, k2048, st + la[o < NA ? o : 0], PLANE_A);
    else
      stage_piece<AR>(vb[o < NA ? 0 : o - NA], sb, k2048, st + NPL * PLANE_A + lb[o < NA ? 0 : o - NA], PLANE_B);
  };

  f32x16 acc[Parts<AR>::accs][TM][TN];
  auto clear = [&](int a) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][i][j][v] = 0.0f;
  };

  const int fr = lane & 31, fc = lane >> 5;
  auto frag = [&](const unsigned char* pl, int r, int kg) {
    return *reinterpret_cast<const u32x4*>(pl + r * 64 + 16 * ((2 * kg + fc) ^ ((r >> 2) & 3)));
  };
  const int grp = lane >> 4, gi = lane & 3, gr = (lane >> 2) & 3;
  const int rd_k = 8 * (grp >> 1) + gr, rd_c = 4 * (grp & 1) + gi;
  auto frag_t = [&](const unsigned char* pl, int col32, int kg) {
    const int c = col32 / 4 + rd_c;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(pl + tn_chunk_off<BN>(16 * kg + rd_k, c)));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(pl + tn_chunk_off<BN>(16 * kg + rd_k + 4, c)));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    const i16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(u32x4, v);
  };

  constexpr int NT = Parts<AR>::products;
  u32x4 fa[TM][NPL], fb[TN][NPL];
  auto read = [&](const unsigned char* st, int kg) __attribute__((always_inline)) {
#pragma unroll
    for (int pp = 0; pp < NPL; ++pp) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i][pp] = frag(st + pp * PLANE_A, wm * (128 / WM) + 32 * i + fr, kg);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[j][pp] = BKM ? frag_t(st + NPL * PLANE_A + pp * PLANE_B, wn * (BN / 2) + 32 * j, kg)
                       : frag(st + NPL * PLANE_A + pp * PLANE_B, wn * (BN / 2) + 32 * j + fr, kg);
    }
  };
#pragma unroll
  for (int a = 0; a < Parts<AR>::accs; ++a) clear(a);
  if constexpr (AR == ARITH_BF16X6) {  // one slab at a time in one stage
    for (int kt = 0; kt < nk; ++kt) {
      mask_tail(kt);
#pragma unroll
      for (int o = 0; o < NA + NB; ++o) {
        split_piece(lds, o);
        load_piece(kt + 1, o);
      }
      lds_barrier();
#pragma unroll
      for (int kg = 0; kg < 2; ++kg) {
        read(lds, kg);
#pragma unroll
        for (int t = 0; t < NT; ++t) products<AR, TM, TN, true>(acc, fa, fb, t);
      }
      lds_barrier();
    }
  } else {
  if (nk > 0) {
    mask_tail(0);
#pragma unroll
    for (int o = 0; o < NA + NB; ++o) {
      split_piece(lds, o);
      load_piece(1, o);
    }
    lds_barrier();
  }
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const unsigned char* st = lds + (kt & 1) * STAGE;
    unsigned char* nst = lds + ((kt & 1) ^ 1) * STAGE;
    read(st, 0);
    mask_tail(kt + 1);
    // the two k-groups' products, a piece of slab kt + 1 split after each and its registers loaded with slab kt + 2's
    constexpr int PER = (NA + NB + 2 * NT - 1) / (2 * NT);
#pragma unroll
    for (int t = 0; t < 2 * NT; ++t) {
      if (t == NT) read(st, 1);
      products<AR, TM, TN, true>(acc, fa, fb, t % NT);
#pragma unroll
      for (int o = t * PER; o < (t + 1) * PER && o < NA + NB; ++o) {
        split_piece(nst, o);
        load_piece(kt + 2, o);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  }
  if (nk > 0) {  // the last slab: one k-group, or two
    const unsigned char* st = lds + ((nk - 1) & 1) * STAGE;
    for (int kg = 0; kg < 2 && (nk - 1) * BK + 16 * kg < K; ++kg) {
      read(st, kg);
#pragma unroll
      for (int t = 0; t < NT; ++t) products<AR, TM, TN, true>(acc, fa, fb, t);
    }
    lds_barrier();
  }
  join_acc<AR, TM, TN>(acc);
  }
  float* const patch = reinterpret_cast<float*>(lds) + wave * 32 * PS;  // every wave is past the last barrier
  const int rw = row0 + wm * (128 / WM), cw = col0 + wn * (BN / 2);
  if constexpr (AR != ARITH_BF16) {
    const float m = nt_pipe_epilogue_t<TM, TN, EPI, epi_generic(EPI), true>(P, acc[0], rw, cw, patch, lane,
                                                                               pow2(-ea), pow2(-eb));
    if (P.amax_c != nullptr) amax_publish(P.amax_c, m, AR == ARITH_BF16X6, lane, (THREADS / 64) * blockIdx.x + wave);
  } else {
    nt_pipe_epilogue<TM, TN, EPI>(P, acc[0], rw, cw, patch, lane);
  }
}

template <int BN, int WM, int EPI, bool BKM>
__device__ __attribute__((noinline)) void nt_wide_tile(uint64_t group, LdsBytes* lds) {
  nt_f16_tile<BN, WM, EPI, BKM, ARITH_BF16X6>(group_at(group), (unsigned char*)lds);
}

template <int BN, int WM, int OCC, int EPI, bool BKM, int AR>
__global__ __launch_bounds__(WM * 128) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_nt_f16_kernel(
    const Group g) {
  constexpr int STAGES = 2 * Parts<AR>::planes * (128 + BN) * 32 * 2, PATCHES = WM * 2 * 32 * 36 * 4;
  __shared__ __align__(16) unsigned char lds[STAGES > PATCHES ? STAGES : PATCHES];
  nt_f16_tile<BN, WM, EPI, BKM, AR>(g, lds);
}

// ------------------------------------------------------------------------------------------------------------------
// TN (weight-grad): C[m,n] = sum_k A[k,m] B[k,n] over one split's rows, 128 x BN tiles, 32-row k-slabs in two LDS
// stages of k-major planes, fragments by the transposing LDS read (layouts as in gemm_core.hpp's tn_bx6_tile).  The
// last slab of a matrix whose rows are not whole slabs is shifted back to end at the matrix's end, its rows before the
// slab's own start zeroed (and a matrix of fewer than 32 rows re-reads its last row, zeroed).
// ------------------------------------------------------------------------------------------------------------------
template <int BN, int WM, int AR>
__device__ __forceinline__ void tn_f16_tile(const Group& g, const TileCoord tc, unsigned char* lds, int ea = 0, int eb = 0) {
  constexpr int BM = 128, BK = 32, THREADS = WM * 128, TM = 4 / WM, TN = BN / 64, NPL = Parts<AR>::planes;
  constexpr int PLANE_A = BK * BM * 2, PLANE_B = BK * BN * 2, STAGE = NPL * (PLANE_A + PLANE_B);
  const Problem& P = g.p[tc.pi];
  const int64_t lda = P.lda, ldb = P.ldb;
  const int row0 = tc.tm * BM, col0 = tc.tn * BN;
  const int M = P.M, N = P.N, K = P.K;
  const int k_begin = tc.split * P.k_chunk;
  const int k_end = min(K, k_begin + P.k_chunk);
  const int nk = (k_end - k_begin + BK - 1) / BK;
  const int tid = threadIdx.x, lane = tid & 63, wave = wave_id();
  const int wm = wave >> 1, wn = wave & 1;
  const bool want_colsum = P.colsum != nullptr && tc.tn == 0;

  constexpr int KPPA = THREADS / 32, NA = BK / KPPA, CPRB = BN / 4, KPPB = THREADS / CPRB, NB = BK / KPPB;
  const int sc = tid & 31, sk = tid >> 5, bsc = tid % CPRB, bsk = tid / CPRB;
  const int mc_a = min(row0 + 4 * sc, ((M - 1) >> 2) << 2), mc_b = min(col0 + 4 * bsc, ((N - 1) >> 2) << 2);
  uint32_t aoff[NA], boff[NB];  // from the slab's first row (32 rows of an operand span less than 2^31 bytes)
  int la[NA], lb[NB];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    aoff[i] = static_cast<uint32_t>((min(sk + KPPA * i, K - 1) * lda + mc_a) * 4);
    la[i] = tn_chunk_off<BM>(sk + KPPA * i, sc);
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    boff[i] = static_cast<uint32_t>((min(bsk + KPPB * i, K - 1) * ldb + mc_b) * 4);
    lb[i] = tn_chunk_off<BN>(bsk + KPPB * i, bsc);
  }
  f32x4 va[NA], vb[NB];
  auto load_piece = [&](int kt, int o) __attribute__((always_inline)) {
    const int64_t k0 = max(min(k_begin + kt * BK, K - BK), 0);
    if (o < NA) {
      va[o < NA ? o : 0] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const unsigned char*>(P.A + k0 * lda) +
                                                           aoff[o < NA ? o : 0]);
    } else {
      const int i = o < NA ? 0 : o - NA;
      vb[i] = *reinterpret_cast<const f32x4*>(reinterpret_cast<const unsigned char*>(P.B + k0 * ldb) + boff[i]);
    }
  };
  // rows outside [k_begin + 32 kt, k_end): those that a shifted slab repeats, and those past a chunk's end
  auto mask_tail = [&](int kt) __attribute__((always_inline)) {
    const int own = k_begin + kt * BK, k0 = max(min(own, K - BK), 0);
    if (own == k0 && own + BK <= k_end) return;
#pragma unroll
    for (int i = 0; i < NA; ++i) {
      const int k = k0 + sk + KPPA * i;
      if (k < own || k >= k_end) va[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int k = k0 + bsk + KPPB * i;
      if (k < own || k >= k_end) vb[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
  };
#pragma unroll
  for (int o = 0; o < NA + NB; ++o) load_piece(0, o);
  const float sa = pow2(ea), sb = pow2(eb);
  const float k2048 = 2048.0f;
  double colsum_acc[4] = {0.0, 0.0, 0.0, 0.0};
  auto split_piece = [&](unsigned char* st, int o) __attribute__((always_inline)) {
    if (o < NA)
      stage_piece<AR>(va[o < NA ? o : 0], sa, k2048, st + la[o < NA ? o : 0], PLANE_A);
    else
      stage_piece<AR>(vb[o < NA ? 0 : o - NA], sb, k2048, st + NPL * PLANE_A + lb[o < NA ? 0 : o - NA], PLANE_B);
  };
  auto add_colsum = [&](int i) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) colsum_acc[e] += static_cast<double>(va[i][e]);
  };

  f32x16 acc[Parts<AR>::accs][TM][TN];
  auto clear = [&](int a) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[a][i][j][v] = 0.0f;
  };

  const int grp = lane >> 4, gi = lane & 3, gr = (lane >> 2) & 3;
  const int rd_k = 8 * (grp >> 1) + gr, rd_c = 4 * (grp & 1) + gi;
  auto frag = [&](auto w_c, const unsigned char* pl, int col32, int kg) {
    constexpr int W = decltype(w_c)::value;
    const int c = col32 / 4 + rd_c;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(pl + tn_chunk_off<W>(16 * kg + rd_k, c)));
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) i16x4*)(pl + tn_chunk_off<W>(16 * kg + rd_k + 4, c)));
    typedef short i16x8 __attribute__((ext_vector_type(8)));
    const i16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(u32x4, v);
  };

  constexpr int NT = Parts<AR>::products;
  u32x4 fa[TM][NPL], fb[TN][NPL];
  auto read = [&](const unsigned char* st, int kg) __attribute__((always_inline)) {
#pragma unroll
    for (int pp = 0; pp < NPL; ++pp) {
#pragma unroll
      for (int i = 0; i < TM; ++i) fa[i][pp] = frag(IntC<BM>{}, st + pp * PLANE_A, wm * (128 / WM) + 32 * i, kg);
#pragma unroll
      for (int j = 0; j < TN; ++j)
        fb[j][pp] = frag(IntC<BN>{}, st + NPL * PLANE_A + pp * PLANE_B, wn * (BN / 2) + 32 * j, kg);
    }
  };
#pragma unroll
  for (int a = 0; a < Parts<AR>::accs; ++a) clear(a);
  if constexpr (AR == ARITH_BF16X6) {  // (as in nt_f16_tile)
    for (int kt = 0; kt < nk; ++kt) {
      mask_tail(kt);
#pragma unroll
      for (int o = 0; o < NA + NB; ++o) {
        split_piece(lds, o);
        if (o < NA && want_colsum) add_colsum(o < NA ? o : 0);
        load_piece(kt + 1, o);
      }
      lds_barrier();
#pragma unroll
      for (int kg = 0; kg < 2; ++kg) {
        read(lds, kg);
#pragma unroll
        for (int t = 0; t < NT; ++t) products<AR, TM, TN, false>(acc, fa, fb, t);
      }
      lds_barrier();
    }
  } else {
  if (nk > 0) {
    mask_tail(0);
#pragma unroll
    for (int o = 0; o < NA + NB; ++o) {
      split_piece(lds, o);
      if (o < NA && want_colsum) add_colsum(o < NA ? o : 0);
      load_piece(1, o);
    }
    lds_barrier();
  }
  for (int kt = 0; kt + 1 < nk; ++kt) {
    const unsigned char* st = lds + (kt & 1) * STAGE;
    unsigned char* nst = lds + ((kt & 1) ^ 1) * STAGE;
    read(st, 0);
    mask_tail(kt + 1);
    // the two k-groups' products, a piece of slab kt + 1 split after each and its registers loaded with slab kt + 2's
    constexpr int PER = (NA + NB + 2 * NT - 1) / (2 * NT);
#pragma unroll
    for (int t = 0; t < 2 * NT; ++t) {
      if (t == NT) read(st, 1);
      products<AR, TM, TN, false>(acc, fa, fb, t % NT);
#pragma unroll
      for (int o = t * PER; o < (t + 1) * PER && o < NA + NB; ++o) {
        split_piece(nst, o);
        if (o < NA && want_colsum) add_colsum(o < NA ? o : 0);
        load_piece(kt + 2, o);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    lds_barrier();
  }
  if (nk > 0) {
    const unsigned char* st = lds + ((nk - 1) & 1) * STAGE;
    for (int kg = 0; kg < 2; ++kg) {
      read(st, kg);
#pragma unroll
      for (int t = 0; t < NT; ++t) products<AR, TM, TN, false>(acc, fa, fb, t);
    }
  }
  join_acc<AR, TM, TN>(acc);
  }
  [[maybe_unused]] const float ra = pow2(-ea), rb = pow2(-eb);

  const int fr = lane & 31, fc = lane >> 5;
  float* Cs = P.C + static_cast<int64_t>(tc.split) * P.partial_stride;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = col0 + wn * (BN / 2) + 32 * j + fr;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = row0 + wm * (128 / WM) + 32 * i + 8 * (v >> 2) + 4 * fc + (v & 3);
        const float x = AR == ARITH_F16X3 ? acc[0][i][j][v] * ra * rb : acc[0][i][j][v];
        if (m < M && n < N) Cs[static_cast<int64_t>(m) * P.ldc + n] = x;
      }
    }
  if (want_colsum) {  // column 4 sc + e: the row groups sk in order
    double* part = reinterpret_cast<double*>(lds);  // [KPPA][128]
    lds_barrier();
#pragma unroll
    for (int e = 0; e < 4; ++e) part[sk * 128 + 4 * sc + e] = colsum_acc[e];
    lds_barrier();
    if (tid < 128 && row0 + tid < M) {
      double sum = part[tid];
      for (int r = 1; r < KPPA; ++r) sum += part[r * 128 + tid];
      P.colsum[static_cast<int64_t>(tc.split) * M + row0 + tid] = sum;
    }
  }
}

template <int BN, int WM>
__device__ __attribute__((noinline)) void tn_wide_tile(uint64_t group, LdsBytes* lds) {
  const Group& g = group_at(group);
  tn_f16_tile<BN, WM, ARITH_BF16X6>(g, locate(g), (unsigned char*)lds);
}

template <int WM, int OCC, int AR>
__global__ __launch_bounds__(WM * 128) __attribute__((amdgpu_waves_per_eu(OCC, OCC))) void gemm_tn_f16_kernel(
    const Group g) {
  __shared__ __align__(16) unsigned char lds[2 * Parts<AR>::planes * 2 * 32 * 128 * 2];
  const TileCoord tc = locate(g);
  const Problem& P = g.p[tc.pi];
  int ea = 0, eb = 0;
  if constexpr (AR == ARITH_F16X3) {
    const int lane = threadIdx.x & 63;
    const Range ra = load_range(P.amax_a, lane), rb = load_range(P.amax_b, lane);
    if (!ra.narrow() || !rb.narrow()) {
      if (P.tn64) tn_wide_tile<64, WM>(group_argument(), (LdsBytes*)lds);
      else tn_wide_tile<128, WM>(group_argument(), (LdsBytes*)lds);
      return;
    }
    ea = amax_exponent(ra.top);
    eb = amax_exponent(rb.top);
  }
  if (P.tn64) {
    tn_f16_tile<64, WM, AR>(g, tc, lds, ea, eb);
  } else {
    tn_f16_tile<128, WM, AR>(g, tc, lds, ea, eb);
  }
}

}  // namespace
}  // namespace ppo
