// Decode-batch QKV projection fused with the pre-attention step: one launch
// computes, for up to 64 tokens,
//   qkv = RMSNorm(h) @ W_qkv^T                 (qwen3/attention.py:81, norm.py:22-26)
//   q, k = RMSNorm_head(q), RMSNorm_head(k)    (qwen3/attention.py:91-92)
//   q, k = RoPE(q, k) at each token's position (qwen3/rope.py:88-110)
// and stores q for the attention kernel and k, v into the paged pool at
// position seq_lens[row] through the resident block table, as the decode
// form of the pre-attention kernel does (qwen3/kernels/paged_attention.py:
// 292-350 for the write).
//
// Work split: one 1024-thread workgroup per (head, 16-token block).  Its 16
// waves are 8 column tiles of the head's 128 weight rows x 2 halves of K;
// each streams 16 weight rows from HBM as the B operand of
// mfma_f32_16x16x32_bf16 (loads coalesced per lane quad, redistributed with
// ds_bpermute).  The A operand, the block's 16 rows of the residual stream h
// after the input RMSNorm (rms from the producer's per-16-column partial
// sums of h^2), is staged once in LDS by the whole workgroup and read from
// there in the operand layout.  The head's 16 x 128 outputs meet in LDS, rounded to bf16 as the
// projection's output is, and 16 lanes per token finish the head with the
// arithmetic of the pre-attention kernel (same lane grouping, same
// summation order, so the same bits).  The 16-token blocks of one head run
// on one XCD (workgroups are dealt round-robin), so its weights come from
// HBM once.
#include "decode_head.hpp"

namespace {

constexpr int kD = 128;
constexpr int kRowsPerBlock = 16;
constexpr int kColTiles = kD / 16;  // 8
constexpr int kKParts = 2;
constexpr int kWavesQ = kColTiles * kKParts;  // 16
constexpr int kThreadsQ = kWavesQ * 64;       // 1024
constexpr int kKStep = 32;
constexpr int kC = 8;  // k-steps per prefetch buffer (weights only)
constexpr int kMaxRows = 64;
constexpr int kMaxK = 4096;  // staged A rows: 16 x (K + 8) bf16 in LDS
constexpr int kXcds = 8;

struct QkvArgs {
  const uint16_t* h;  // residual stream (M x K)
  int64_t h_s;
  const float* ss_in;  // (M x ss_tiles) partial sums of h^2
  int ss_tiles;
  const uint16_t* norm_w;  // input RMSNorm weight (K)
  float eps;
  const uint16_t* w;  // fused qkv weight ((Hq + 2 Hkv) * 128 x K)
  int64_t w_s;
  int M, K;
  HeadArgs hd;
};

__global__ __launch_bounds__(kThreadsQ) void qkv_rope_kernel(QkvArgs a) {
  // The block's 16 normalised A rows, staged once: row r at a_s + r * pitch.
  extern __shared__ uint16_t a_s[];
  __shared__ float rms_s[kRowsPerBlock];
  __shared__ float red[kColTiles][4][64];
  __shared__ uint16_t y_s[kRowsPerBlock][kD];
  __shared__ int64_t pos_s[kRowsPerBlock], phys_s[kRowsPerBlock];
  __shared__ int off_s[kRowsPerBlock];

  const int heads = a.hd.Hq + 2 * a.hd.Hkv;
  const int rbc = (a.M + 15) >> 4;
  const int b = blockIdx.x;
  const int slot = b >> 3;
  const int head = (slot / rbc) * kXcds + (b & (kXcds - 1));
  const int rb = slot % rbc;
  if (head >= heads) return;  // whole workgroup

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int ct = wave % kColTiles;  // column tile of the head
  const int kh = wave / kColTiles;  // half of K
  const int r16 = lane & 15;
  const int kg = 8 * (lane >> 4);
  const int kw = a.K / kKParts;
  const int k0 = kh * kw;
  const int steps = kw / kKStep;
  const int pitch = a.K + 8;  // bf16 elements per staged row (16-byte pad: no bank conflicts)

  // Weights: coalesced loads (lane l: row l / 4, k-group l % 4) moved into
  // the operand layout (lane L: row L % 16, k-group L / 16) by ds_bpermute.
  const int lrow = lane >> 2, lkg = 8 * (lane & 3);
  const int perm_addr = 4 * (4 * r16 + (lane >> 4));
  const uint16_t* wrow =
      a.w + static_cast<int64_t>(head * kD + ct * 16 + lrow) * a.w_s + lkg + k0;
  auto to_mfma = [&](q3::u32x4 v) {
    q3::u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(perm_addr, static_cast<int>(v[e])));
    return o;
  };
  struct Buf {
    q3::u32x4 b[kC];
  };
  auto load = [&](Buf& B, int s0) {
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      if (s0 + u >= steps) break;
      B.b[u] = q3::ld16(wrow + (s0 + u) * kKStep);
    }
  };
  Buf p, q;
  load(p, 0);
  load(q, kC);

  // A rows and norm weight for this thread's first staging chunks (16 rows x
  // K/8 chunks of 8), the rms of every row, and the position and pool slot
  // of every token of the block: all independent of the weights, so their
  // loads overlap them.
  const int cpr = a.K >> 3;  // chunks per row
  const int nchunks = kRowsPerBlock * cpr;
  constexpr int kPre = 2;  // chunks per thread loaded early (all of them for K <= 1024)
  q3::u32x4 hv[kPre], nv[kPre];
  auto chunk_src = [&](int c, q3::u32x4& h, q3::u32x4& n) {
    const int r = c / cpr, cc = c - r * cpr;
    const int row = min(rb * 16 + r, a.M - 1);
    h = q3::ld16(a.h + static_cast<int64_t>(row) * a.h_s + 8 * cc);
    n = q3::ld16(a.norm_w + 8 * cc);
  };
#pragma unroll
  for (int i = 0; i < kPre; ++i)
    if (tid + i * kThreadsQ < nchunks) chunk_src(tid + i * kThreadsQ, hv[i], nv[i]);
  if (wave == 0) {
    const int row = min(rb * 16 + (lane >> 2), a.M - 1);
    const int part = lane & 3;
    const float* sp = a.ss_in + static_cast<int64_t>(row) * a.ss_tiles;
    float s = 0.f;
    if (a.ss_tiles == 64) {
      float4 f[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) f[j] = reinterpret_cast<const float4*>(sp + 16 * part)[j];
#pragma unroll
      for (int j = 0; j < 4; ++j) s += ((f[j].x + f[j].y) + f[j].z) + f[j].w;
    } else {
      for (int t = part; t < a.ss_tiles; t += 4) s += sp[t];
    }
    s += q3::dpp_f32<q3::kDppXor1>(s);  // lane ^ 1
    s += q3::dpp_f32<q3::kDppXor2>(s);  // lane ^ 2
    if (part == 0) rms_s[lane >> 2] = 1.f / sqrtf(s / static_cast<float>(a.K) + a.eps);
  } else if (wave == 1 && lane < kRowsPerBlock) {
    int64_t pos, phys;
    int off;
    locate_token(a.hd, rb * 16 + lane, pos, phys, off);
    pos_s[lane] = pos;
    phys_s[lane] = phys;
    off_s[lane] = off;
  }
  __syncthreads();
  // a = bf16((h * rms) * w), the input RMSNorm (qwen3/norm.py:22-26)
  auto chunk_store = [&](int c, const q3::u32x4& h, const q3::u32x4& n) {
    const int r = c / cpr, cc = c - r * cpr;
    const float rr = rms_s[r];
    q3::u32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      o[e] = q3::pack_bf16x2((q3::bf16_lo(h[e]) * rr) * q3::bf16_lo(n[e]),
                             (q3::bf16_hi(h[e]) * rr) * q3::bf16_hi(n[e]));
    *reinterpret_cast<q3::u32x4*>(a_s + r * pitch + 8 * cc) = o;
  };
#pragma unroll
  for (int i = 0; i < kPre; ++i)
    if (tid + i * kThreadsQ < nchunks) chunk_store(tid + i * kThreadsQ, hv[i], nv[i]);
  for (int c = tid + kPre * kThreadsQ; c < nchunks; c += kThreadsQ) {
    q3::u32x4 h, n;
    chunk_src(c, h, n);
    chunk_store(c, h, n);
  }
  __syncthreads();

  // A fragment of step s: lane L reads row L % 16, k = k0 + 32 s + 8 (L / 16).
  const uint16_t* arow = a_s + r16 * pitch + k0 + kg;
  q3::f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  auto compute = [&](const Buf& B, int s0) {
#pragma unroll
    for (int u = 0; u < kC; ++u) {
      if (s0 + u >= steps) break;
      const q3::u32x4 av = *reinterpret_cast<const q3::u32x4*>(arow + (s0 + u) * kKStep);
      acc = q3::mfma16x16x32(q3::as_bf16x8(av), q3::as_bf16x8(to_mfma(B.b[u])), acc);
    }
  };
  for (int s0 = 0; s0 < steps; s0 += 2 * kC) {
    compute(p, s0);
    load(p, s0 + 2 * kC);
    compute(q, s0 + kC);
    load(q, s0 + 3 * kC);
  }

  // Sum the two halves of K in order (first half + second half) and round to
  // bf16, the projection's output type: y_s[token][column].
  if (kh == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) red[ct][i][lane] = acc[i];
  }
  __syncthreads();
  if (kh == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      y_s[4 * (lane >> 4) + i][ct * 16 + r16] = q3::bf16_bits(acc[i] + red[ct][i][lane]);
  }
  __syncthreads();

  // Finish the head: 16 lanes per token, 8 dims per lane (lane j: dims
  // 8j .. 8j+7), the pre-attention kernel's grouping.
  if (tid >= kRowsPerBlock * 16) return;
  const int r = tid >> 4, j = tid & 15;
  const int t = rb * 16 + r;
  if (t >= a.M) return;  // whole 16-lane groups
  const q3::u32x4 xw = *reinterpret_cast<const q3::u32x4*>(&y_s[r][8 * j]);
  finish_head(a.hd, head, t, j, xw, pos_s[r], phys_s[r], off_s[r]);
}

}  // namespace

extern "C" int qwen3_decode_qkv_rope_bf16(
    const void* h, int64_t h_row_stride, const float* ss_in, int ss_in_tiles,
    const void* norm_weight, float eps, const void* qkv_weight, int64_t weight_row_stride, int M,
    int K, int num_heads, int num_kv_heads, int head_dim, const void* q_norm_weight,
    const void* k_norm_weight, float head_eps, const float* cos_table, const float* sin_table,
    int64_t table_row_stride, int64_t table_rows, const int64_t* positions, void* q_out,
    const int64_t q_out_strides[2], void* k_cache, const int64_t k_cache_strides[4],
    void* v_cache, const int64_t v_cache_strides[4], int64_t num_blocks, int layer_idx,
    int num_layers,
    const int32_t* seq_lens, const int32_t* block_table, int64_t bt_row_stride, int64_t max_rows,
    int64_t max_pages, const int32_t* row_ids, int block_size, void* stream) {
  const char* who = "qwen3_decode_qkv_rope_bf16";
  if (!h || !ss_in || !norm_weight || !qkv_weight || !q_norm_weight || !k_norm_weight ||
      !cos_table || !sin_table || !q_out || !q_out_strides || !k_cache || !k_cache_strides ||
      !v_cache || !v_cache_strides || !seq_lens || !block_table)
    return q3::fail(QWEN3_EINVAL, "%s: null pointer argument", who);
  if (head_dim != kD)
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: head_dim %d not supported (built for %d)", who,
                    head_dim, kD);
  if (M < 0 || M > kMaxRows || K <= 0 || num_heads <= 0 || num_kv_heads <= 0 ||
      ss_in_tiles <= 0 || block_size <= 0 || num_blocks <= 0 || layer_idx < 0 ||
      layer_idx >= num_layers ||
      table_rows < 0 || max_rows <= 0 || max_pages <= 0 || bt_row_stride < max_pages ||
      !(eps >= 0.f) || !(head_eps >= 0.f))
    return q3::fail(QWEN3_EINVAL, "%s: bad sizes (M must be <= %d)", who, kMaxRows);
  if (K % (kKParts * kKStep) != 0 || K > kMaxK)
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: K must be a multiple of %d and <= %d", who,
                    kKParts * kKStep, kMaxK);
  bool ok = q3::aligned16(h) && q3::aligned16(ss_in) && q3::aligned16(norm_weight) &&
            q3::aligned16(qkv_weight) && q3::aligned16(q_norm_weight) &&
            q3::aligned16(k_norm_weight) && q3::aligned16(cos_table) &&
            q3::aligned16(sin_table) && q3::aligned16(q_out) && q3::aligned16(k_cache) &&
            q3::aligned16(v_cache) && h_row_stride % 8 == 0 && weight_row_stride % 8 == 0 &&
            ss_in_tiles % 4 == 0 && table_row_stride % 4 == 0;
  const int64_t strides[] = {q_out_strides[0], q_out_strides[1], k_cache_strides[0],
                             k_cache_strides[1], k_cache_strides[2], k_cache_strides[3],
                             v_cache_strides[0], v_cache_strides[1], v_cache_strides[2],
                             v_cache_strides[3]};
  for (int64_t s : strides) ok = ok && s % 8 == 0;
  if (!ok)
    return q3::fail(QWEN3_EALIGN, "%s: tensors need 16-byte aligned rows", who);
  if (M == 0) return QWEN3_OK;
  QkvArgs a{};
  a.h = static_cast<const uint16_t*>(h);
  a.h_s = h_row_stride;
  a.ss_in = ss_in;
  a.ss_tiles = ss_in_tiles;
  a.norm_w = static_cast<const uint16_t*>(norm_weight);
  a.eps = eps;
  a.w = static_cast<const uint16_t*>(qkv_weight);
  a.w_s = weight_row_stride;
  a.M = M;
  a.K = K;
  HeadArgs& hd = a.hd;
  hd.M = M;
  hd.Hq = num_heads;
  hd.Hkv = num_kv_heads;
  hd.q_w = static_cast<const uint16_t*>(q_norm_weight);
  hd.k_w = static_cast<const uint16_t*>(k_norm_weight);
  hd.head_eps = head_eps;
  hd.cos_t = cos_table;
  hd.sin_t = sin_table;
  hd.tab_stride = table_row_stride;
  hd.tab_rows = table_rows;
  hd.positions = positions;
  hd.q_out = static_cast<uint16_t*>(q_out);
  hd.qo_s0 = q_out_strides[0];
  hd.qo_s1 = q_out_strides[1];
  hd.k_cache = static_cast<uint16_t*>(k_cache);
  hd.v_cache = static_cast<uint16_t*>(v_cache);
  for (int i = 0; i < 4; ++i) {
    hd.kc[i] = k_cache_strides[i];
    hd.vc[i] = v_cache_strides[i];
  }
  hd.num_blocks = num_blocks;
  hd.layer = layer_idx;
  hd.seq_lens = seq_lens;
  hd.block_table = block_table;
  hd.bt_stride = bt_row_stride;
  hd.max_rows = max_rows;
  hd.max_pages = max_pages;
  hd.row_ids = row_ids;
  hd.bs = block_size;
  const int heads = num_heads + 2 * num_kv_heads;
  const int64_t blocks = q3::cdiv(heads, kXcds) * kXcds * ((M + 15) / 16);
  q3::clear_error();
  const size_t lds = static_cast<size_t>(kRowsPerBlock) * (K + 8) * sizeof(uint16_t);
  hipLaunchKernelGGL(qkv_rope_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreadsQ), lds,
                     static_cast<hipStream_t>(stream), a);
  return q3::launch_status(who);
}
