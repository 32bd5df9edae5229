// The streaming paged decode's partial results: where a launch leaves them in
// the workspace, and how a query head's are combined.
#pragma once

#include "common.hpp"

namespace {

struct StreamLayout {
  int64_t po, plse, pref, meta, total;
};

inline int64_t align256(int64_t x) { return (x + 255) / 256 * 256; }

// Workspace layout of the stream path for `waves` persistent waves and
// groups of G query heads.
inline StreamLayout stream_layout(int B, int64_t waves, int G) {
  constexpr int64_t kD = 128;
  StreamLayout s;
  s.po = 0;
  s.plse = s.po + align256(waves * 2 * G * kD * 4);
  s.pref = s.plse + align256(waves * 2 * G * 4);
  s.meta = s.pref + align256((static_cast<int64_t>(B) + 1) * 4);
  s.total = s.meta + 256;
  return s;
}

struct StreamPartials {
  q3::GlobalPtr<const float> po;      // [W][2][G][128] normalised partial outputs
  q3::GlobalPtr<const float> plse;    // [W][2][G] log2-sum-exp of each
  q3::GlobalPtr<const int32_t> pref;  // [B + 1] exclusive prefix of tiles per sequence
  q3::GlobalPtr<const int32_t> meta;  // [0] tiles per wave
  int Hkv, G;
};

// Query head hq of batch entry b, by one wave: lanes first fetch the LSEs of
// up to 64 covering waves at once, then every lane owns output dims 2 lane,
// 2 lane + 1 (packed in y) and sums the weighted partials kBatch waves at a
// time.  False: a wave has written the head whole.  An empty context is zero.
template <int kBatch = 16>
__device__ __forceinline__ bool merge_partials(const StreamPartials& p, int b, int64_t hq,
                                               int lane, uint32_t& y) {
  constexpr int kD = 128;
  const int G = p.G;
  const int hkv = static_cast<int>(hq / G), g = static_cast<int>(hq % G);
  const int64_t pref_b = p.pref[b];
  const int n = p.pref[b + 1] - static_cast<int32_t>(pref_b);
  if (n == 0) {
    y = 0u;
    return true;
  }
  const int64_t pw = p.meta[0];
  const int64_t S = static_cast<int64_t>(p.Hkv) * pref_b + static_cast<int64_t>(hkv) * n;
  const int64_t E = S + n;
  // (a 64-bit division is a long stretch of code)
  const bool small = E <= 0xffffffffll;
  const int64_t wf = small ? static_cast<uint32_t>(S) / static_cast<uint32_t>(pw) : S / pw;
  const int64_t wl =
      small ? static_cast<uint32_t>(E - 1) / static_cast<uint32_t>(pw) : (E - 1) / pw;
  if (wf == wl) return false;  // written whole by its wave
  const int nw = static_cast<int>(wl - wf + 1);
  const int slot0 = static_cast<int>(wf) * 2 * G + g;  // fewer than 2^18 slots
  const int half0 = wf * pw != S ? G : 0;              // the first wave's second slot
  // The partials kBatch at a time, the first ones fetched with the LSEs; one
  // past the last lies outside the descriptor and reads as zero.
  const int stride = 2 * G * kD * 4;  // bytes from one wave's partial to the next
  const __amdgpu_buffer_rsrc_t po = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(p.po + static_cast<int64_t>(slot0) * kD), 0, (nw - 1) * stride + kD * 4,
      0x00020000);
  q3::u32x2 ov[kBatch];
  auto fetch = [&](int i0) {
    const int off = i0 * stride + 8 * lane;
#pragma unroll
    for (int j = 0; j < kBatch; ++j)
      ov[j] = __builtin_bit_cast(
          q3::u32x2, __builtin_amdgcn_raw_buffer_load_b64(
                         po, off + j * stride + (j == 0 && i0 == 0 ? half0 * kD * 4 : 0), 0, 0));
  };
  auto lse_at = [&](int i) -> float {
    return i < nw ? p.plse[slot0 + i * 2 * G + (i == 0 ? half0 : 0)] : q3::kNegInf;
  };
  fetch(0);
  // Pass 1: global max of the partial LSEs.
  const float lse0 = lse_at(lane);
  float M = lse0;
  for (int i0 = 64; i0 < nw; i0 += 64) M = fmaxf(M, lse_at(i0 + lane));
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) M = fmaxf(M, q3::shfl_xor(M, o));
  const float M_use = M == q3::kNegInf ? 0.f : M;
  // Pass 2: weighted sum of the partial outputs (lane owns dims 2*lane, 2*lane+1).
  float sw = 0.f, o0 = 0.f, o1 = 0.f;
  for (int i0 = 0; i0 < nw; i0 += 64) {
    const float wl_lane = q3::fast_exp2((i0 == 0 ? lse0 : lse_at(i0 + lane)) - M_use);
    float wsum = wl_lane;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) wsum += q3::shfl_xor(wsum, o);
    sw += wsum;
    const int cnt = nw - i0 < 64 ? nw - i0 : 64;
    for (int j0 = 0; j0 < cnt; j0 += kBatch) {
      if (i0 + j0 > 0) fetch(i0 + j0);
#pragma unroll
      for (int j = 0; j < kBatch; ++j) {  // weight 0 past the last
        const float wt =
            __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(wl_lane), j0 + j));
        o0 += wt * __uint_as_float(ov[j][0]);
        o1 += wt * __uint_as_float(ov[j][1]);
      }
    }
  }
  const float inv = sw > 0.f ? 1.f / sw : 0.f;
  y = q3::pack_bf16x2(o0 * inv, o1 * inv);
  return true;
}

}  // namespace
