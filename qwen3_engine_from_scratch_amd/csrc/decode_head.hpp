// The end of a decode head, shared by the kernels that project q, k and v: a
// token's position and pool slot, and QK-RMSNorm + RoPE + the q / K / V store
// of one head row, with the arithmetic and roundings of the pre-attention
// kernel (same lane grouping, same summation order, so the same bits).
#pragma once

#include "common.hpp"

namespace {

constexpr int kHeadD = 128;

struct HeadArgs {
  int M, Hq, Hkv;
  q3::GlobalPtr<const uint16_t> q_w;  // QK-norm weights (128)
  q3::GlobalPtr<const uint16_t> k_w;
  float head_eps;
  q3::GlobalPtr<const float> cos_t;
  q3::GlobalPtr<const float> sin_t;
  int64_t tab_stride, tab_rows;
  q3::GlobalPtr<const int64_t> positions;  // nullable: RoPE at seq_lens[row]
  q3::GlobalPtr<uint16_t> q_out;
  int64_t qo_s0, qo_s1;
  q3::GlobalPtr<uint16_t> k_cache;
  q3::GlobalPtr<uint16_t> v_cache;
  int64_t kc[4], vc[4];
  int64_t num_blocks;
  int layer;
  q3::GlobalPtr<const int32_t> seq_lens;
  q3::GlobalPtr<const int32_t> block_table;
  int64_t bt_stride, max_rows, max_pages;
  q3::GlobalPtr<const int32_t> row_ids;  // nullable: identity
  int bs;
};

// RoPE position, pool block and slot in it of token t; -1 where the tables
// have none.
__device__ __forceinline__ void locate_token(const HeadArgs& a, int t, int64_t& pos,
                                             int64_t& phys, int& off) {
  pos = -1;
  phys = -1;
  off = 0;
  if (t >= a.M) return;
  const int64_t row = a.row_ids ? a.row_ids[t] : t;
  if (row < 0 || row >= a.max_rows) return;
  const int64_t wpos = a.seq_lens[row];
  const int64_t pg = wpos >= 0 ? wpos / a.bs : -1;
  if (pg >= 0 && pg < a.max_pages) {
    phys = a.block_table[row * a.bt_stride + pg];
    off = static_cast<int>(wpos % a.bs);
  }
  pos = a.positions ? a.positions[t] : wpos;
}

// Head `head` of token t (< M): lane j of a 16-lane group holds dims 8j ..
// 8j + 7 of the projection's output (xw).  Called by whole groups; a lane
// whose stores() is false writes nothing (asked for after row_sum).  row_sum: the
// sum over the group's lanes (q3::row16_sum, or its value by other means).
template <typename Stores, typename Sum>
__device__ __forceinline__ void finish_head(const HeadArgs& a, int head, int t, int j,
                                            q3::u32x4 xw, int64_t pos, int64_t phys, int off,
                                            Stores&& stores, Sum&& row_sum) {
  const bool ok_pos = pos >= 0 && pos < a.tab_rows;
  const bool write_pool = ok_pos && phys >= 0 && phys < a.num_blocks;
  const int kv_base = a.Hq + a.Hkv;
  if (head >= kv_base) {  // v: a bit-exact copy into the pool
    if (write_pool && stores())
      q3::st16(a.v_cache + phys * a.vc[0] + static_cast<int64_t>(a.layer) * a.vc[1] +
                   static_cast<int64_t>(head - kv_base) * a.vc[2] + off * a.vc[3] + 8 * j,
               xw);
    return;
  }
  const uint16_t* wn = head < a.Hq ? a.q_w : a.k_w;
  const q3::u32x4 ww = q3::ld16(wn + 8 * j);
  float x[8], w[8];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = q3::bf16_lo(xw[e]);
    x[2 * e + 1] = q3::bf16_hi(xw[e]);
    w[2 * e] = q3::bf16_lo(ww[e]);
    w[2 * e + 1] = q3::bf16_hi(ww[e]);
  }
  float cv[8], sv[8];
  if (ok_pos) {
    const float* cr = a.cos_t + pos * a.tab_stride + 8 * j;
    const float* sr = a.sin_t + pos * a.tab_stride + 8 * j;
    const float4 c0 = *reinterpret_cast<const float4*>(cr);
    const float4 c1 = *reinterpret_cast<const float4*>(cr + 4);
    const float4 s0 = *reinterpret_cast<const float4*>(sr);
    const float4 s1 = *reinterpret_cast<const float4*>(sr + 4);
    const float cc[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
    const float ss_[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      cv[e] = q3::round_bf16(cc[e]);  // cos / sin .to(q.dtype)
      sv[e] = q3::round_bf16(ss_[e]);
    }
  }
  // Squares rounded, then summed (no fused multiply-add), as x.pow(2).mean().
  float ss = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) ss = __fadd_rn(ss, __fmul_rn(x[e], x[e]));
  ss = row_sum(ss);
  const float rmsh = 1.f / sqrtf(ss / static_cast<float>(kHeadD) + a.head_eps);
  uint32_t np[4], pp[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    np[e] = q3::pack_bf16x2((x[2 * e] * rmsh) * w[2 * e], (x[2 * e + 1] * rmsh) * w[2 * e + 1]);
#pragma unroll
  for (int e = 0; e < 4; ++e) pp[e] = q3::dpp_u32<q3::kDppRor8>(np[e]);  // lane j ^ 8
  const float sign = j < 8 ? -1.f : 1.f;  // rotate_half: (-x2, x1)
  q3::u32x4 out = {0u, 0u, 0u, 0u};
  if (ok_pos) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float o[2];
#pragma unroll
      for (int hl = 0; hl < 2; ++hl) {
        const int el = 2 * e + hl;
        const float n = hl ? q3::bf16_hi(np[e]) : q3::bf16_lo(np[e]);
        const float rh = sign * (hl ? q3::bf16_hi(pp[e]) : q3::bf16_lo(pp[e]));
        o[hl] = q3::round_bf16(n * cv[el]) + q3::round_bf16(rh * sv[el]);
      }
      out[e] = q3::pack_bf16x2(o[0], o[1]);
    }
  }
  if (!stores()) return;
  if (head < a.Hq) {
    q3::st16(a.q_out + static_cast<int64_t>(t) * a.qo_s0 +
                 static_cast<int64_t>(head) * a.qo_s1 + 8 * j,
             out);
  } else if (write_pool) {
    q3::st16(a.k_cache + phys * a.kc[0] + static_cast<int64_t>(a.layer) * a.kc[1] +
                 static_cast<int64_t>(head - a.Hq) * a.kc[2] + off * a.kc[3] + 8 * j,
             out);
  }
}
__device__ __forceinline__ void finish_head(const HeadArgs& a, int head, int t, int j,
                                            q3::u32x4 xw, int64_t pos, int64_t phys, int off) {
  finish_head(a, head, t, j, xw, pos, phys, off, []() { return true; },
              [](float ss) { return q3::row16_sum(ss); });
}

}  // namespace
