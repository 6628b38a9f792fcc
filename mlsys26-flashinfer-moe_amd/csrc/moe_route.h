// Device code of the grouped top-8 routing shared by the routing kernels and by the decode GEMM1 of
// the smallest batches. Its fp32 operations are evaluated exactly as written: the top-k lists
// do not depend on which kernel made them.
#pragma once

#include "moe_internal.h"
#include "moe_device.h"

namespace moe {

__device__ __forceinline__ float load_bias(const void* bias, int dtype, int i) {
  if (dtype == MOE_FP8_BIAS_F32) return reinterpret_cast<const float*>(bias)[i];
  const uint16_t h = reinterpret_cast<const uint16_t*>(bias)[i];
  if (dtype == MOE_FP8_BIAS_BF16) return __uint_as_float((uint32_t)h << 16);
  return (float)__builtin_bit_cast(_Float16, h);
}

// Multiset top-2 merge: (a1 >= a2) and (b1 >= b2) -> the two largest of the four.
__device__ __forceinline__ void top2_merge(float& m1, float& m2, float o1, float o2) {
  const float n1 = fmaxf(m1, o1);
  const float n2 = fmaxf(fminf(m1, o1), fmaxf(m2, o2));
  m1 = n1;
  m2 = n2;
}

// DPP lane permutations (within rows of 16 lanes).
constexpr int kDppXor1 = 0xB1;         // quad_perm [1,0,3,2]
constexpr int kDppXor2 = 0x4E;         // quad_perm [2,3,0,1]
constexpr int kDppHalfMirror = 0x141;  // lane i <-> 7-i within 8
constexpr int kDppMirror = 0x140;      // lane i <-> 15-i within 16

template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false));
}

template <int CTRL>
__device__ __forceinline__ uint64_t dpp_u64(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, 0xF, 0xF, false);
  return ((uint64_t)hi << 32) | lo;
}

// Argmax keys of the routing: a larger fp32 value wins, then the lower expert index (the
// "lowest index on ties" rule of kernel.py:499 and :525): key = ordered(v) << 32 | 0xFFFF - e.
__device__ __forceinline__ int key_index(uint64_t key) { return 0xFFFF - (int)(key & 0xFFFFu); }

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

// Order-preserving map of a float to an unsigned key (after -0 -> +0, so equal values tie):
// a > b as floats <=> ordered(a) > ordered(b).
__device__ __forceinline__ uint32_t ordered(float v) {
  const uint32_t u = __float_as_uint(v + 0.0f);
  return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
constexpr uint32_t kOrderedNegInf = 0x007FFFFFu;   // ordered(-inf)

template <int CTRL>
__device__ __forceinline__ int dpp_i32(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xF, 0xF, false);
}

// DPP row broadcasts across the 16-lane rows of a wavefront (GFX9): lane 15 of each row to
// the next row (rows 1 and 3 take it), lane 31 to rows 2 and 3.
constexpr int kDppRowBcast15 = 0x142;
constexpr int kDppRowBcast31 = 0x143;

template <int CTRL, int ROW_MASK>
__device__ __forceinline__ uint64_t dpp_u64_rows(uint64_t v) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, ROW_MASK, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(v >> 32), CTRL, ROW_MASK, 0xF, false);
  return ((uint64_t)hi << 32) | lo;
}

// Inclusive sum over lanes 0..31 (which must all be active), by DPP row shifts and one row broadcast:
// a shuffle through the data-share unit costs several times a step's latency.
__device__ __forceinline__ int scan32(int v) {
  v += dpp_i32<0x111>(v);   // row_shr:1
  v += dpp_i32<0x112>(v);
  v += dpp_i32<0x114>(v);
  v += dpp_i32<0x118>(v);
  v += __builtin_amdgcn_update_dpp(0, v, kDppRowBcast15, 0xA, 0xF, false);
  return v;
}

// Stable rank of each lane's slot among the wavefront's slots of the same local expert (le < 0: not
// local), and the wavefront's 32 counts in `cnt` (LDS): one ballot per distinct local expert of the
// wavefront, a few of the 32 as a rule. Lane e < 32 gathers expert e's count in a register and stores
// cnt[e] itself, so that it may read it back at once; the other lanes' counts need a barrier. Against
// a ballot for each of the 32 (with the scans by shuffle): layer at T=80 162.0 -> 160.8 us, 128
// 168.7 -> 167.4, 901 239.4 -> 238.8, 8192 583.8 -> 582.2, skewed T=128 220.0 -> 218.7. GEMM1's own
// dispatch keeps its scans by shuffle: with scan32 T=16 68.7 -> 68.5, but skewed T=64 170.4 -> 170.8.
__device__ __forceinline__ int wave_rank(int le, int* cnt) {
  const int lane = lane_id();
  const uint64_t lt = lanemask_lt();
  int rank = 0, n = 0;
  uint64_t todo = __ballot(le >= 0);
  while (todo) {
    const int v = __builtin_amdgcn_readlane(le, __builtin_ctzll(todo));
    const uint64_t m = __ballot(le == v);
    if (le == v) rank = __popcll(m & lt);
    if (lane == v) n = __popcll(m);
    todo &= ~m;
  }
  if (lane < kExpertsLocal) cnt[lane] = n;
  return rank;
}

// Routing of token t by one wavefront (kernel.py:428-542), for small batches: lane l holds
// experts 4l..4l+3, so group g (32 experts) is lanes 8g..8g+7, and every lane does a quarter
// of route_wave's per-token work. The selections are route_wave's: the same argmax keys, the
// group score as the sum of the group's two largest biased scores, the kept groups by (score,
// lower index), the weights summed in selection order with the same fp32 operations, so
// the top-k lists are bit-identical. `lg` holds the lane's four logits. Returns in lanes
// k < 8 the expert of top-k slot k and its weight; other lanes return -1.
__device__ __forceinline__ int route_wide(const RouteParams& p, const float* s_bias, int t, const float4 lg,
                                          float& w_out) {
#pragma clang fp contract(off)
  const int lane = lane_id();
  const float4 cb = reinterpret_cast<const float4*>(s_bias)[lane];
  const float xs[4] = {lg.x, lg.y, lg.z, lg.w}, cs[4] = {cb.x, cb.y, cb.z, cb.w};
  float b[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) b[j] = sigmoid_f32(xs[j]) + cs[j];   // kernel.py:466-467
  // group score (kernel.py:479-488): top-2 of the lane's four, then of the group's 8 lanes
  float m1 = fmaxf(b[0], b[1]), m2 = fminf(b[0], b[1]);
#pragma unroll
  for (int i = 2; i < 4; ++i) {
    const float n2 = __builtin_amdgcn_fmed3f(m1, m2, b[i]);
    m1 = fmaxf(m1, b[i]);
    m2 = n2;
  }
  top2_merge(m1, m2, dpp_f32<kDppXor1>(m1), dpp_f32<kDppXor1>(m2));
  top2_merge(m1, m2, dpp_f32<kDppXor2>(m1), dpp_f32<kDppXor2>(m2));
  top2_merge(m1, m2, dpp_f32<kDppHalfMirror>(m1), dpp_f32<kDppHalfMirror>(m2));
  const float gs = m1 + m2;
  // the 4 best groups (kernel.py:495-501): the eight scores are wave-uniform (lane 8h holds
  // group h's), and a group is kept iff fewer than 4 groups rank before it
  const int g = lane >> 3;
  int rank = 0;
#pragma unroll
  for (int h = 0; h < kNGroup; ++h) {
    const float hs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(gs), 8 * h));
    rank += (hs > gs || (hs == gs && h < g)) ? 1 : 0;
  }
  const bool kept = rank < kTopKGroup;
  // top-8 experts of the kept groups (kernel.py:515-534): 8 rounds of (argmax inside the
  // lane, argmax of the 64-bit keys across the wavefront, removal of the winner)
  uint32_t c[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) c[i] = kept ? ordered(b[i]) : kOrderedNegInf;
  const uint32_t lo_base = 0xFFFFu - 4u * (uint32_t)lane;
  int my_id = -1;
#pragma unroll
  for (int k = 0; k < kTopK; ++k) {
    const bool h01 = c[1] > c[0], h23 = c[3] > c[2];
    const uint32_t v01 = h01 ? c[1] : c[0], v23 = h23 ? c[3] : c[2];
    const uint32_t i01 = h01 ? 1u : 0u, i23 = h23 ? 3u : 2u;
    const bool hi = v23 > v01;
    uint64_t key = ((uint64_t)(hi ? v23 : v01) << 32) | (lo_base - (hi ? i23 : i01));
    key = max_u64(key, dpp_u64<kDppXor1>(key));
    key = max_u64(key, dpp_u64<kDppXor2>(key));
    key = max_u64(key, dpp_u64<kDppHalfMirror>(key));
    key = max_u64(key, dpp_u64<kDppMirror>(key));
    key = max_u64(key, dpp_u64_rows<kDppRowBcast15, 0xA>(key));
    key = max_u64(key, dpp_u64_rows<kDppRowBcast31, 0xC>(key));
    // lane 63 holds the wavefront's largest key
    const uint32_t klo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)key, 63);
    const int e = key_index((uint64_t)klo);
    my_id = (lane == k) ? e : my_id;
    // the winner drops to -inf, where it ties with the other -inf entries (kernel.py:534)
    const uint32_t drop = ((e >> 2) == lane) ? (uint32_t)(e & 3) : 4u;
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = (drop == (uint32_t)i) ? kOrderedNegInf : c[i];
  }
  // weights (kernel.py:537-538), as route_wave: w = s / (s_0 + ... + s_7 + 1e-20) * rsf
  const float sv = (lane < kTopK) ? sigmoid_f32(p.logits[(size_t)t * kExpertsGlobal + my_id]) : 0.0f;
  float sum = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sv), 0));
#pragma unroll
  for (int k = 1; k < kTopK; ++k) sum = sum + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(sv), k));
  sum = sum + 1e-20f;
  w_out = __fdiv_rn(sv, sum) * p.rsf;
  return lane < kTopK ? my_id : -1;
}

// Router bias (fp32, bf16 or fp16) -> fp32 in LDS; the whole work-group calls this.
__device__ __forceinline__ void stage_bias(const RouteParams& p, float* s_bias) {
  if (!p.skip_routing && threadIdx.x < kExpertsGlobal) s_bias[threadIdx.x] = load_bias(p.bias, p.bias_dtype, threadIdx.x);
  __syncthreads();
}

}  // namespace moe
