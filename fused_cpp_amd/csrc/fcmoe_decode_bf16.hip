// fcmoe_decode_bf16.hip -- BF16 and W8A16 MoE layers of a few routes in two
// launches, as fcmoe_decode_tail.hip's for W8A8.
//
//   head: route build + W13 + activation. Workgroup (pair, route) is one wave:
//         it derives every route's sorted position from the ids by a ballot
//         (routes by expert, then by flat route), streams its expert's gate and
//         up tile through a register ring and passes the token's row through
//         row 0 of the MFMA. The pair 0 workgroups write the route metadata.
//   tail: W2 + merge. Workgroup (channel tile, token) has a wave per slot; the
//         slots' values meet in LDS and wave 0 merges them as combine_kernel.
//
// The layer's four launches cost ~3 us of host time each and 3-5 us each on
// the GPU whatever their work. What the two cost instead is that every route
// streams its own expert's weights: nothing extra for one token (its experts
// differ), L2 reads beyond, so the caller bounds routes x expert bytes. Per
// product the K order is the 16-row kernel's, so both give the same bits.
// Arithmetic: csrc/moe/arm/common/fused_moe_bf16_tiled.cpp:1861-1914 (the
// activation), csrc/moe/arm/sve_bf16/route_merge.cpp:47-126 (the merge).
#include <type_traits>
#include <utility>

#include "fcmoe_gemm_common.h"

namespace fcmoe {
namespace {

constexpr int kRing = 8;

// The wave's dot products of one bf16 row with NT 16-channel tiles: chunk c
// pairs a 1 KB weight piece of each tile with 64 bytes of the row (W8A16: 64
// int8 weights a channel with 128 bytes). acc[.][0] of lanes 0..15 is the
// result. Chunks past the last re-load it (never consumed). ONCE: no other
// workgroup reads these weights (one token): nontemporal loads.
template <bool W8, bool ONCE, int NT>
__device__ __forceinline__ void row_times_tiles(const uint8_t* row, const uint8_t* const (&w)[NT], int kc, int lane,
                                                v4f (&acc)[NT]) {
  constexpr int AW = W8 ? 2 : 1;
  v4i bq[kRing][NT], aq[kRing][AW];
  const uint8_t* arow = row + (lane / 16) * 16 * AW;
  auto issue = [&](int c, auto slot_c) {
    constexpr int b = decltype(slot_c)::value;
    const int cc = c < kc ? c : kc - 1;
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const v4i* src = (const v4i*)(w[j] + (int64_t)cc * 1024) + lane;
      bq[b][j] = ONCE ? __builtin_nontemporal_load(src) : *src;
    }
#pragma unroll
    for (int h = 0; h < AW; ++h) aq[b][h] = *(const v4i*)(arow + (int64_t)cc * 64 * AW + h * 16);
  };
#pragma unroll
  for (int j = 0; j < NT; ++j) acc[j] = v4f{0, 0, 0, 0};
  [&]<int... S>(std::integer_sequence<int, S...>) {
    (issue(S, std::integral_constant<int, S>{}), ...);
  }(std::make_integer_sequence<int, kRing - 1>{});
  auto body = [&](int c, auto b_c) {
    constexpr int b = decltype(b_c)::value;
    issue(c + kRing - 1, std::integral_constant<int, (b + kRing - 1) % kRing>{});
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      if constexpr (W8) {
        v4i lo, hi;
        i8x16_to_bf16(bq[b][j], lo, hi);
        acc[j] = mfma(__builtin_bit_cast(v8bf, aq[b][0]), __builtin_bit_cast(v8bf, lo), acc[j]);
        acc[j] = mfma(__builtin_bit_cast(v8bf, aq[b][1]), __builtin_bit_cast(v8bf, hi), acc[j]);
      } else {
        acc[j] = mfma(__builtin_bit_cast(v8bf, aq[b][0]), __builtin_bit_cast(v8bf, bq[b][j]), acc[j]);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  int c0 = 0;
  for (; c0 + kRing <= kc; c0 += kRing) {
    [&]<int... S>(std::integer_sequence<int, S...>) {
      (body(c0 + S, std::integral_constant<int, S>{}), ...);
    }(std::make_integer_sequence<int, kRing>{});
  }
  [&]<int... S>(std::integer_sequence<int, S...>) {
    ((c0 + S < kc ? body(c0 + S, std::integral_constant<int, S>{}) : void()), ...);
  }(std::make_integer_sequence<int, kRing - 1>{});
}

template <bool W8, bool ONCE>
__global__ __launch_bounds__(kWave) void bf16_head_kernel(SmallBatchArgs a) {
  const int lane = threadIdx.x;
  const int j = blockIdx.x, r = blockIdx.y;
  const int tok = ONCE ? 0 : r / a.kt;  // (ONCE is one token: no division ahead of the loads)
  const int routes = ONCE ? a.kt : a.tokens * a.kt;  // at most 64: lane l carries route l
  // every route's expert, validity (route_expert) and combined weight (route_weight_of)
  const int lr = lane < routes ? lane : 0;
  const int lt = ONCE ? 0 : lr / a.kt, ls = lr - lt * a.kt;
  const int idx = ls < a.top_k ? lt * a.top_k + ls : 0;  // (top_k = 0: no ids, only the shared slot)
  const int64_t e = a.top_k == 0 ? 0 : a.ids_is_i64 ? ((const int64_t*)a.ids)[idx] : (int64_t)((const int32_t*)a.ids)[idx];
  float w_l = a.topk_w && a.top_k > 0 ? a.topk_w[idx] : 1.0f;
  if (a.scale_routed) w_l = w_l * a.scale;
  bool ok_l = lane < routes;
  int e_l = a.shared_id;
  if (ls < a.top_k) {
    ok_l = ok_l && e >= 0 && e < a.valid_experts;
    e_l = ok_l ? (int)e : 0;
  } else {
    w_l = 1.0f;
  }
  const int e_r = __builtin_amdgcn_readlane(e_l, r);
  const bool ok_r = __builtin_amdgcn_readlane((int)ok_l, r) != 0;
  const int pos = __popcll(__ballot(ok_l && (e_l < e_r || (e_l == e_r && lane < r))));
  const int n_invalid = __popcll(__ballot(lane < routes && !ok_l));
  if (j == 0 && lane == 0) {
    a.route_pos[r] = ok_r ? pos : -1;
    a.route_weight[r] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w_l), r));
    if (ok_r) {
      a.sorted_routes[pos] = r;
      a.row_token[pos] = tok;
    }
    if (r == 0) store_count(a.invalid, n_invalid);
  }
  if (!ok_r) return;
  const int kc = a.k_chunks13;
  const uint8_t* wg = (const uint8_t*)a.w13 + (int64_t)e_r * a.w13_expert_bytes + (int64_t)j * kc * 1024;
  const uint8_t* const w[2] = {wg, wg + (int64_t)a.n_tiles13 * kc * 1024};
  // the epilogue's channel values, ahead of the stream
  const int64_t f = (int64_t)j * 16 + lane % 16;
  const int64_t fc = f < a.inter ? f : 0;
  const float* cv = W8 ? a.w13_scale : a.w13_bias;
  float cg = 0.0f, cu = 0.0f;
  if (cv) {
    cg = cv[(int64_t)e_r * 2 * a.inter + fc];
    cu = cv[(int64_t)e_r * 2 * a.inter + a.inter + fc];
  }
  v4f acc[2];
  row_times_tiles<W8, ONCE, 2>((const uint8_t*)(a.x + (int64_t)tok * a.hidden), w, kc, lane, acc);
  if (lane >= 16 || f >= a.inter) return;
  float gate = acc[0][0], up = acc[1][0];
  if constexpr (W8) {
    gate = gate * cg;
    up = up * cu;
  } else if (cv) {
    gate = gate + cg;
    up = up + cu;
  }
  a.y[(int64_t)pos * a.inter + f] = f32_to_bf16(act_bf16_mode(gate, up, a.activation));
}

template <bool W8, bool ONCE>
__global__ __launch_bounds__(kDecodeTailSlots * kWave) void bf16_tail_kernel(SmallBatchArgs a) {
  __shared__ float s_val[kDecodeTailSlots][16];
  __shared__ float s_wt[kDecodeTailSlots];
  __shared__ int s_ok[kDecodeTailSlots];
  const int lane = threadIdx.x % kWave;
  const int slot = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int tile = blockIdx.x, t = blockIdx.y;
  const int64_t ch = (int64_t)tile * 16 + lane % 16;
  const bool cvalid = ch < a.hidden;
  const int r = t * a.kt + slot;
  const int pos = a.route_pos[r];  // -1: the id was invalid and the route is dropped
  const int idx = t * a.top_k + (slot < a.top_k ? slot : 0);
  const int eid = a.top_k == 0 ? 0 : a.ids_is_i64 ? (int)((const int64_t*)a.ids)[idx] : ((const int32_t*)a.ids)[idx];
  if (pos >= 0) {
    const int e = slot < a.top_k ? eid : a.shared_id;
    const int64_t cidx = (int64_t)e * a.hidden + (cvalid ? ch : 0);
    const float cs = W8 ? a.w2_scale[cidx] : a.w2_bias ? a.w2_bias[cidx] : 0.0f;
    const float wt = a.route_weight[r];
    const int kc = a.k_chunks2;
    const uint8_t* const w[1] = {(const uint8_t*)a.w2 + (int64_t)e * a.w2_expert_bytes + (int64_t)tile * kc * 1024};
    v4f acc[1];
    row_times_tiles<W8, ONCE, 1>((const uint8_t*)(a.y + (int64_t)pos * a.inter), w, kc, lane, acc);
    if (lane < 16) {
      float v = acc[0][0];
      if constexpr (W8)
        v = v * cs;
      else if (a.w2_bias)
        v = v + cs;
      s_val[slot][lane] = v;
      if (cvalid) a.route_out[(int64_t)r * a.hidden + ch] = v;
    }
    if (lane == 0) {
      s_wt[slot] = wt;
      s_ok[slot] = 1;
    }
  } else if (lane == 0) {
    s_ok[slot] = 0;
  }
  __syncthreads();
  if (slot != 0 || lane >= 16 || !cvalid) return;
  float merged = 0.0f;
  if (a.skip_weighted) {
    merged = s_ok[0] ? s_val[0][lane] : 0.0f;
  } else if (a.kt == 2 || a.kt == 4 || a.kt == 6 || a.kt == 8) {
    float v[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) v[s] = s < a.kt && s_ok[s] ? s_val[s][lane] * s_wt[s] : 0.0f;
    merged = a.kt == 2   ? TreeSum<0, 2>::run(v)
             : a.kt == 4 ? TreeSum<0, 4>::run(v)
             : a.kt == 6 ? TreeSum<0, 6>::run(v)
                         : TreeSum<0, 8>::run(v);
  } else {
    for (int s = 0; s < a.kt; ++s)
      if (s_ok[s]) merged = __builtin_fmaf(s_val[s][lane], s_wt[s], merged);
  }
  a.out[(int64_t)t * a.hidden + ch] = f32_to_bf16(merged);
}

}  // namespace

int small_batch_bf16_launch(const SmallBatchArgs& a, bool w8, bool tail, hipStream_t stream) {
  const int64_t chunk = w8 ? 64 : 32;  // elements of K per chunk
  if (a.tokens <= 0 || a.kt <= 0 || a.kt > kDecodeTailSlots || (int64_t)a.tokens * a.kt > kWave || a.hidden <= 0 ||
      a.inter <= 0 || a.hidden % chunk || a.inter % chunk || a.k_chunks13 * chunk != a.hidden ||
      a.k_chunks2 * chunk != a.inter || a.n_tiles13 != ceil_div(a.inter, 16))
    return fail(FCMOE_EINVAL, "small-batch MoE: shapes outside its domain");
  auto launch = [&](auto w8_c, auto once_c) {
    constexpr bool W8 = decltype(w8_c)::value, ONCE = decltype(once_c)::value;
    if (tail)
      hipLaunchKernelGGL((bf16_tail_kernel<W8, ONCE>), dim3((unsigned)ceil_div(a.hidden, 16), (unsigned)a.tokens),
                         dim3((unsigned)(a.kt * kWave)), 0, stream, a);
    else
      hipLaunchKernelGGL((bf16_head_kernel<W8, ONCE>), dim3((unsigned)a.n_tiles13, (unsigned)(a.tokens * a.kt)),
                         dim3(kWave), 0, stream, a);
  };
  std::true_type yes;
  std::false_type no;
  if (w8)
    a.tokens == 1 ? launch(yes, yes) : launch(yes, no);
  else
    a.tokens == 1 ? launch(no, yes) : launch(no, no);
  return check_launch(tail ? "small_batch_tail" : "small_batch_head");
}

}  // namespace fcmoe
