// The dense work between two attention launches of a decode step, for at most
// 16 rows, in one launch:
//   merge     the streaming attention's partial results -> o     (paged_decode_merge.hpp)
//   o_proj    h_mid = h + o @ W_o^T                              (qwen3/attention.py:187, decoder.py:49)
//   gate_up   act = SwiGLU(RMSNorm(h_mid) @ W_gu^T)              (qwen3/mlp.py:31-36)
//   down      h = h_mid + act @ W_down^T                         (qwen3/decoder.py:55)
//   qkv       the next layer's q, k, v: RMSNorm, projection, QK-norm, RoPE and
//             the K/V pool write (as decode_qkv.hip)
// with the arithmetic, K splits and summation orders of the separate kernels
// (decode_linear.hip, decode_qkv.hip), so the same bits.
//
// Why: with few rows each of these is a few microseconds of latency -- about
// 2.3 us of launch and end-of-kernel write-back, then weights, activations and
// the cross-wave sum waited for in turn -- and five of them make up most of a
// small batch's step.  Here every workgroup issues its weight loads first and
// then waits for the phase before its own, so the layer's 30 MB stream in while
// the first phases run and each further phase costs its hand-off instead of a
// launch.
//
// Hand-off: the blocks of a phase are numbered after those of the phase
// before it.  A block publishes its results with device-scope (sc1) stores,
// waits until they are complete, and sets its own flag words to the launch's
// number; a block of the next phase polls that phase's flags, 256 at a time, and
// then reads the results with device-scope loads.  (Counters instead of flags:
// an add takes about 80 ns on its line, 2.4 us for 192 blocks on eight lines.
// Eight copies of the flags, each polled by an eighth of the blocks: device-scope
// loads of one line are served about 10 ns apart, 2.5 us a round for 192
// blocks.)  No fence: those write back and invalidate the whole L2.
//
// Progress: a block never depends on another one being resident.  The dispatcher
// starts the blocks in order on each XCD, but not across XCDs, and other work
// (another such launch on another stream, another process, a CU mask) may hold
// the slots that a waited-for block needs.  So a wait that is not answered within
// wait_ticks ends, and the block runs the missing blocks' work itself, lowest
// phase first, and then its own again (next_item).  That is sound because every
// block's work is a function of its number whose inputs do not change while
// anyone may still need them: running it twice, even at the same time, stores
// the same bits.  (The one input that the launch overwrites, h_in where h_out is
// the same buffer: an o_proj block first loads its residual and then looks at its
// own flag; unset, what it loaded is from before any down block could store;
// set, its work is done and it stores nothing.)  Nothing is put back to zero for
// the next launch, which would have to know that no late block still comes:
// flags and exchanged sums carry the launch's number, which the last block to
// arrive advances.
//
// Before they wait, gate_up, down and qkv blocks run their phase once without
// data and without storing anything: the weights passing through have evicted
// the code since the last launch, and a first pass over a phase's
// instructions takes a microsecond or more longer than the second.  They ask
// for their weights after that, when the merge's loads and o_proj's are out.
// (o_proj has no such pass: it would end after the merge.)
//
// Qwen3-0.6B, one row at 900 tokens: merge done 6.2 us after the start, o_proj
// 9.9, gate_up 14, down 17.5, qkv 22.5; as separate launches 5.0, 5.9, 7.4,
// 5.9 and 13.5 each (24.4 for the launch as a kernel trace counts it).  A step
// with them: 1448 -> 1033 us, of which a flag that carries the launch's number,
// where the flags were put back to zero and a wait could fail for good, is
// 10.  The rare path is code of its own behind the usual one: a loop around both
// would hold what it shares in more registers than there are.
#include "decode_head.hpp"
#include "paged_decode_merge.hpp"

namespace {

constexpr int kThreads = 512;
constexpr int kWaves = kThreads / 64;
constexpr int kKStep = 32;      // k per MFMA
constexpr int kMaxSteps = 12;   // k-steps of a wave's weights held in registers
constexpr int kAhead = 8;       // activation k-steps in flight
constexpr int kRows = 16;
constexpr int kQkvSteps = 16;   // k-steps of half of K, at most
constexpr int kMaxHidden = 2 * kQkvSteps * kKStep;  // 1024
constexpr int kMaxBlocks = 1024;
constexpr int kMaxNormHeads = 64;  // q and k heads
constexpr int kSc1 = 16;        // buffer cache policy: device scope
// A wait's limit, in ticks of the 100 MHz clock: 200 us, ten times the longest
// wait of a launch that has the device to itself.
constexpr int64_t kWaitTicks = 20000;

enum Phase : int { kMerge = 0, kO = 1, kGateUp = 2, kDown = 3, kQkv = 4, kPhases = 5 };
// Sync words, each part on lines (128 bytes) of its own: the number of launches
// so far, the counts of blocks that have arrived (kArriveLines lines, then
// the lines that are complete), kCopies flags per block, and the sums that the
// two blocks of a q or k head exchange (8 bytes: launch number, sum).
constexpr int kCopies = 8;
constexpr int kLine = 32;
constexpr int kArriveLines = 32;
constexpr int kArriveWord = kLine;
constexpr int kFlagWord = kArriveWord + (kArriveLines + 1) * kLine;
constexpr int kSumWord = kFlagWord + kCopies * kMaxBlocks;  // [head][half of it][row][2]
constexpr int kSums = kMaxNormHeads * 2 * kRows * 2;
constexpr int kMaxRowBlocks = 4;  // of the qkv kernel
constexpr int kSyncWords = kSumWord + 2 * kMaxRowBlocks * kSums;

// How a run of one block's work ended: stored, or a wait was not answered.
enum Run : int { kDone = 0, kPhaseMissing = 1, kPartnerMissing = 2 };

struct ChainArgs {
  int M, K, I, KO;          // rows, hidden, intermediate, Hq * 128
  int first[kPhases + 1];   // first block of each phase
  int last_phase;           // kQkv, or kDown for the last layer
  float eps;
  StreamPartials parts;     // merge phase (its block count may be 0)
  q3::GlobalPtr<uint16_t> o;              // M x KO, row stride o_s
  int64_t o_s;
  q3::GlobalPtr<const uint16_t> o_w;
  int64_t o_ws;
  q3::GlobalPtr<const uint16_t> h_in;     // residual streams (M x K, contiguous)
  q3::GlobalPtr<uint16_t> h_mid;
  q3::GlobalPtr<uint16_t> h_out;
  q3::GlobalPtr<float> ss_mid;            // (M x K / 16) sums of squares
  q3::GlobalPtr<float> ss_out;
  q3::GlobalPtr<const uint16_t> post_w;
  q3::GlobalPtr<const uint16_t> gu_w;     // gate rows 0.., up rows I..
  int64_t gu_ws;
  q3::GlobalPtr<uint16_t> act;            // M x I, contiguous
  q3::GlobalPtr<const uint16_t> down_w;
  int64_t down_ws;
  int64_t h_s;              // row stride of h_out for the qkv phase
  q3::GlobalPtr<const uint16_t> in_w;     // next layer
  q3::GlobalPtr<const uint16_t> qkv_w;
  int64_t qkv_ws;
  HeadArgs hd;
  q3::GlobalPtr<uint32_t> sync;           // kSyncWords, zero before the first launch
  int64_t wait_ticks;
};

// Of one workgroup, in LDS.
struct Shared {
  uint32_t launch;  // this launch's number
  bool arrived;     // of wave kTagWave's own
  int run;          // of the current run: its Run so far
  int item;         // the next item to run
};

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void* p, int64_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes),
                                           0x00020000);
}
__device__ __forceinline__ q3::u32x4 ld16_dev(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return __builtin_bit_cast(q3::u32x4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, kSc1));
}
// k-step u of a lane's row (the row and k-group in `off`, so that the step is
// the instruction's own offset).  Steps past the last go through an empty
// descriptor and read as zero: they add nothing and need no branch.
struct Rows {
  const void* p;
  int bytes, steps;
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t at(int u) const {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, u < steps ? bytes : 0,
                                             0x00020000);
  }
  __device__ __forceinline__ q3::u32x4 weight(uint32_t off, int u) const {
    return __builtin_bit_cast(q3::u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             at(u), off + u * kKStep * 2, 0, 0));
  }
  __device__ __forceinline__ q3::u32x4 activation(uint32_t off, int u) const {
    return __builtin_bit_cast(q3::u32x4, __builtin_amdgcn_raw_buffer_load_b128(
                                             at(u), off + u * kKStep * 2, 0, kSc1));
  }
};
__device__ __forceinline__ void st16b_dev(uint16_t* p, uint16_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ uint32_t ld_dev(const uint32_t* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(uint32_t* p, uint32_t v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint32_t add_dev(uint32_t* p) {
  return __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// x, unknown to the compiler: what is derived from it is computed where it is
// used (hoisted out of the pass loops, the offsets of all k-steps would need
// more registers than there are).
__device__ __forceinline__ uint32_t fresh(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}

// The wave that reads the launch's number and reports the block's arrival: it
// has nothing to do while wave 0 waits, stores or polls.
constexpr int kTagWave = kWaves - 1;

// The launch's number, never 0, read once per block, by wave kTagWave into LDS;
// the other waves use it after the block's next barrier.  (It comes round after
// 2^32 - 1 launches, days of decoding; a word is then taken for set only if no
// launch since has used it.)
__device__ __forceinline__ uint32_t read_launch(const uint32_t* sync) {
  return threadIdx.x == kTagWave * 64 ? max(ld_dev(sync) + 1u, 1u) : 0u;
}
__device__ __forceinline__ void share_launch(Shared& sh, uint32_t launch) {
  if (launch != 0u) {
    sh.launch = launch;
    sh.arrived = false;
  }
}

// Reports that this block has read the launch's number (wave kTagWave, after
// share_launch; once).  The last of all blocks advances the number: no block of
// this launch can read it any more, and the next launch begins after all of
// them have ended.
__device__ __forceinline__ void arrive(const ChainArgs& a, Shared& sh) {
  if (threadIdx.x != kTagWave * 64 || sh.arrived) return;
  sh.arrived = true;
  const int line = blockIdx.x % kArriveLines;
  const int lines = min(static_cast<int>(gridDim.x), kArriveLines);
  const int n = (static_cast<int>(gridDim.x) - line + kArriveLines - 1) / kArriveLines;
  uint32_t* count = a.sync + kArriveWord + line * kLine;
  uint32_t* all = a.sync + kArriveWord + kArriveLines * kLine;
  if (add_dev(count) == static_cast<uint32_t>(n - 1)) {
    st_dev(count, 0u);
    if (add_dev(all) == static_cast<uint32_t>(lines - 1)) {
      st_dev(all, 0u);
      st_dev(a.sync, sh.launch);
    }
  }
}

__device__ __forceinline__ const uint32_t* flags_of(const ChainArgs& a) {
  return a.sync + kFlagWord + blockIdx.x % kCopies * kMaxBlocks;
}

// Whether a wait since t0 is over, after `polls` that were not answered (a
// negative limit: after the first).
__device__ __forceinline__ bool too_long(const ChainArgs& a, uint64_t t0, int polls) {
  return ((polls & 3) == 0 || a.wait_ticks < 0) &&
         static_cast<int64_t>(wall_clock64() - t0) > a.wait_ticks;
}

// Waits for the blocks of phase `ph`; afterwards sh.run tells whether it was
// answered.  Every thread of the block calls it.
template <bool kFirst>
__device__ __forceinline__ void wait_phase(const ChainArgs& a, Shared& sh, int ph) {
  const int tid = static_cast<int>(fresh(threadIdx.x));
  if (tid < 64) {
    const uint32_t* flags = flags_of(a);
    const uint32_t tag = sh.launch;
    const int end = a.first[ph + 1];
    int at = a.first[ph] + tid;
    const uint64_t t0 = wall_clock64();
    int polls = 0;
    while (__any(at < end)) {  // the flags below `at` are set
      uint32_t off = 0u;       // of 256 blocks, in one round trip
#pragma unroll
      for (int i = 0; i < 4; ++i)
        off |= at + 64 * i < end ? ld_dev(flags + at + 64 * i) ^ tag : 0u;
      if (__all(off == 0u)) {
        at += 256;
        continue;
      }
      if (too_long(a, t0, ++polls)) break;
    }
    const bool answered = !__any(at < end);
    if (tid == 0) sh.run = answered ? kDone : kPhaseMissing;
  } else if (kFirst && ph > kMerge) {  // (o_proj may not have that long to wait)
    arrive(a, sh);
  }
  __syncthreads();
}

// One wave of the block, after the block's stores to device memory: they are
// complete before the flag shows the item.
__device__ __forceinline__ void set_flag(const ChainArgs& a, const Shared& sh, int item) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  const int lane = static_cast<int>(fresh(threadIdx.x)) & 63;
  if (lane < kCopies) st_dev(a.sync + kFlagWord + lane * kMaxBlocks + item, sh.launch);
}

// What a block runs next after a wait that was not answered (or after such a
// missing item): the other half of its head (`partner`), or an item without a
// flag in the first incomplete phase before its own -- all its inputs are there
// -- and otherwise its own again.  The blocks look from different places, so
// that they help with different items.  Called by every thread of the block.
__device__ __forceinline__ int next_item(const ChainArgs& a, Shared& sh, int own, bool partner) {
  __syncthreads();  // the run before this is over in every wave
  if (partner) return a.first[kQkv] + ((own - a.first[kQkv]) ^ 1);
  const int lane = static_cast<int>(fresh(threadIdx.x));
  if (lane < 64) {
    const uint32_t* flags = flags_of(a);
    int next = own;
#pragma unroll
    for (int ph = 0; ph < kPhases - 1; ++ph) {
      if (own < a.first[ph + 1]) break;  // not before its own
      const int n = a.first[ph + 1] - a.first[ph];
      for (int i = 0; i < n && next == own; i += 64) {
        const int item = a.first[ph] + (i + lane + own) % n;
        const uint64_t missing = __ballot(i + lane < n && ld_dev(flags + item) != sh.launch);
        if (missing) next = __shfl(item, __ffsll(static_cast<unsigned long long>(missing)) - 1, 64);
      }
    }
    if (lane == 0) sh.item = next;
  }
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(sh.item);
}

// rms of this lane's MFMA row (row lane % 16 of the block's rows) from the
// producer's partial sums: four lanes per row take every fourth group of
// tiles, then the butterfly of the separate kernels, so the same bits.
__device__ __forceinline__ float row_rms(const ChainArgs& a, const float* ss, int M, int lane) {
  const int tiles = a.K / 16;
  const int row = min(lane >> 2, M - 1), part = lane & 3;
  const __amdgpu_buffer_rsrc_t r = rsrc_of(ss, static_cast<int64_t>(M) * tiles * 4);
  float s = 0.f;
  if (tiles == 64) {
    q3::u32x4 f[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) f[j] = ld16_dev(r, (row * 64 + 16 * part + 4 * j) * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j)
      s += ((__uint_as_float(f[j][0]) + __uint_as_float(f[j][1])) + __uint_as_float(f[j][2])) +
           __uint_as_float(f[j][3]);
  } else {
    for (int t = part; t < tiles; t += 4)
      s += __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (row * tiles + t) * 4, 0, kSc1));
  }
  s += q3::dpp_f32<q3::kDppXor1>(s);  // lane ^ 1
  s += q3::dpp_f32<q3::kDppXor2>(s);  // lane ^ 2
  const float rms = 1.f / sqrtf(s / static_cast<float>(a.K) + a.eps);
  return __shfl(rms, 4 * (lane & 15), 64);
}

// 2, unknown to the compiler: the dry pass and the real one share their code.
__device__ __forceinline__ int two() {
  int n = 2;
  asm volatile("" : "+s"(n));
  return n;
}

__device__ __forceinline__ q3::u32x4 to_mfma(q3::u32x4 v, int perm_addr) {
  q3::u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = static_cast<uint32_t>(__builtin_amdgcn_ds_bpermute(perm_addr, static_cast<int>(v[e])));
  return o;
}

__device__ __forceinline__ q3::u32x4 normed(q3::u32x4 h, q3::u32x4 w, float rms) {
  q3::u32x4 o;
#pragma unroll
  for (int e = 0; e < 4; ++e)
    o[e] = q3::pack_bf16x2((q3::bf16_lo(h[e]) * rms) * q3::bf16_lo(w[e]),
                           (q3::bf16_hi(h[e]) * rms) * q3::bf16_hi(w[e]));
  return o;
}

// One 16-column tile of o_proj, gate_up or down.  Each wave holds its share of
// the tile's weights before it waits: an eighth of K of the one weight tile
// (o_proj, down), or a quarter of K of the gate or of the up tile (gate_up).
template <int kPh, bool kFirst>
__device__ __forceinline__ int linear_phase(const ChainArgs& a, Shared& sh, int tile,
                                            uint32_t launch, q3::f32x4 (*red)[64],
                                            uint16_t* nw_s) {
  constexpr bool kNorm = kPh == kGateUp;
  constexpr int kSteps = kNorm ? kMaxHidden / 4 / kKStep : kMaxSteps;
  constexpr int kParts = kNorm ? kWaves / 2 : kWaves;  // waves sharing one weight tile's K
  const int tid = static_cast<int>(fresh(threadIdx.x)), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = 8 * (lane >> 4);
  const int lrow = lane >> 2, lkg = 8 * (lane & 3);
  const int perm_addr = 4 * (4 * r16 + (lane >> 4));
  const int n0 = tile * 16;
  const int K = kPh == kO ? a.KO : kPh == kGateUp ? a.K : a.I;
  const int kw = K / kParts;
  const int k0 = (wave % kParts) * kw;
  const int steps = kw / kKStep;  // at most kSteps
  const uint16_t* w = kPh == kO ? a.o_w : kPh == kGateUp ? a.gu_w : a.down_w;
  const int64_t ws = kPh == kO ? a.o_ws : kPh == kGateUp ? a.gu_ws : a.down_ws;
  const Rows wr{w + (n0 + (kNorm && wave >= kParts ? a.I : 0)) * ws,
                static_cast<int>((15 * ws + K) * 2), steps};
  const uint32_t woff = static_cast<uint32_t>((lrow * ws + lkg + k0) * 2);
  q3::u32x4 b[kSteps];
  auto load_weights = [&]() {
#pragma unroll
    for (int u = 0; u < kSteps; ++u) b[u] = wr.weight(woff, u);
  };
  // gate_up and down ask for theirs after the dry pass: 26 MB asked for at
  // once would hold up the merge's loads and o_proj's
  uint32_t res[4] = {0u, 0u, 0u, 0u};
  bool done = false;  // o_proj: by another block already
  if constexpr (kPh == kO) {  // the residual comes from the launch before this one
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * (lane >> 4) + i;
        if (row < a.M) res[i] = a.h_in[static_cast<int64_t>(row) * a.K + n0 + r16];
      }
    }
    load_weights();
    if constexpr (kFirst) share_launch(sh, launch);
    uint32_t flag = 0u;
    if (wave == 0) {  // the residual is here; after that, whether it still was h_in
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(res[i])::"memory");
      const uint32_t* flags = a.sync + kFlagWord + a.first[kO] + tile;  // every copy
      flag = ld_dev(flags + (lane % kCopies) * kMaxBlocks);
    }
    __syncthreads();  // sh.launch
    done = __any(flag == sh.launch);
  } else {
#pragma unroll
    for (int u = 0; u < kSteps; ++u) b[u] = q3::u32x4{0u, 0u, 0u, 0u};
    if constexpr (kFirst) share_launch(sh, launch);  // (the dry pass has a barrier)
  }
  if constexpr (kNorm) {
    for (int i = tid; i < a.K / 8; i += kThreads)
      *reinterpret_cast<q3::u32x4*>(nw_s + 8 * i) = q3::ld16(a.post_w + 8 * i);
  }
  const uint16_t* x = kPh == kO ? a.o : kPh == kGateUp ? a.h_mid : a.act;
  const int64_t xs = kPh == kO ? a.o_s : K;
  // straight into the operand layout (few rows: there is little to coalesce,
  // and a permute here would be on the critical path); rows past M repeat
  // the last
  const uint32_t xoff0 = static_cast<uint32_t>((min(r16, a.M - 1) * xs + kg + k0) * 2);
  for (int pass = kPh == kO ? 1 : 0; pass < two(); ++pass) {
    if (pass) {
      if constexpr (kPh != kO) load_weights();
      // into the operand layout while there is nothing else to do
#pragma unroll
      for (int u = 0; u < kSteps; ++u) b[u] = to_mfma(b[u], perm_addr);
      wait_phase<kFirst>(a, sh, kPh - 1);
    }
    // (the dry pass asks for nothing: an empty descriptor)
    const Rows xr{x, static_cast<int>(((a.M - 1) * xs + K) * 2), pass ? steps : 0};
    const uint32_t xoff = fresh(xoff0);
    const uint16_t* nwp = nw_s + fresh(k0 + kg);
    q3::u32x4 xv[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) xv[u] = xr.activation(xoff, u);
    if constexpr (kPh == kDown) {
      if (wave == 0) {
        const __amdgpu_buffer_rsrc_t hr = rsrc_of(a.h_mid, static_cast<int64_t>(a.M) * a.K * 2);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int row = min(4 * (lane >> 4) + i, a.M - 1);
          res[i] = __builtin_amdgcn_raw_buffer_load_b16(hr, (row * a.K + n0 + r16) * 2, 0, kSc1);
        }
      }
    }
    float rms = 0.f;
    if constexpr (kNorm) rms = row_rms(a, a.ss_mid, a.M, lane);
    q3::f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kSteps; ++u) {
      q3::u32x4 av = xv[u % kAhead];
      if (u + kAhead < kSteps) xv[u % kAhead] = xr.activation(xoff, u + kAhead);
      if constexpr (kNorm)  // (a step past the last: 0 x a weight of step 0)
        av = normed(av, *reinterpret_cast<const q3::u32x4*>(nwp + (u < steps ? u : 0) * kKStep), rms);
      acc = q3::mfma16x16x32(q3::as_bf16x8(av), q3::as_bf16x8(b[u]), acc);
    }
    // Cross-wave sum in wave order; wave 0 runs the epilogue.
    red[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
      const bool stores = pass && sh.run == kDone && !done;
      q3::f32x4 v = red[0][lane], up = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int w2 = 1; w2 < kParts; ++w2) v += red[w2][lane];
      if constexpr (kNorm) {
        up = red[kParts][lane];
#pragma unroll
        for (int w2 = kParts + 1; w2 < kWaves; ++w2) up += red[w2][lane];
      }
      const int col = n0 + r16;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 4 * (lane >> 4) + i;
        const bool live = stores && row < a.M;
        if constexpr (kNorm) {
          const uint16_t y = q3::swiglu_bf16(v[i], up[i]);
          if (live) st16b_dev(a.act + static_cast<int64_t>(row) * a.I + col, y);
        } else {
          uint16_t* dst = kPh == kO ? a.h_mid : a.h_out;
          float* ss = kPh == kO ? a.ss_mid : a.ss_out;
          float h = 0.f;
          if (live) {
            h = q3::add_residual(res[i], v[i]);
            st16b_dev(dst + static_cast<int64_t>(row) * a.K + col, q3::bf16_bits(h));
          }
          float sq = __fmul_rn(h, h);
          sq = q3::row16_sum(sq);
          if (live && r16 == 0)
            __hip_atomic_store(ss + static_cast<int64_t>(row) * (a.K / 16) + tile, sq,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
      if (stores && kPh != a.last_phase) set_flag(a, sh, a.first[kPh] + tile);
    }
  }
  return sh.run;
}

// Adds up the 16 lanes of a token's head (lane j: 8 of its dims, squared and
// summed) when this block has only quads hf and hf + 2 of them: each quad sum
// goes to the head's other block, which has the other two.  Quads 0 + 1 and
// 2 + 3 are added first, as row16_sum does, so the same bits in both blocks.
// `late` is set where they do not come in time.
__device__ __forceinline__ float exchange_sum(const ChainArgs& a, uint32_t tag, int rb, int head,
                                              int hf, int row, int j, float v, bool& late) {
  v += q3::dpp_f32<q3::kDppXor1>(v);
  v += q3::dpp_f32<q3::kDppXor2>(v);
  const bool mine = ((j >> 2) & 1) == hf;
  uint64_t* word = reinterpret_cast<uint64_t*>(a.sync + kSumWord) + rb * kSums +
                   ((head * 2 + (mine ? hf : 1 - hf)) * kRows + row) * 2 + (j >> 3);
  const bool first = (j & 3) == 0;
  if (first && mine)
    __hip_atomic_store(word, static_cast<uint64_t>(tag) << 32 | __float_as_uint(v),
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool reads = first && !mine;
  uint64_t got = static_cast<uint64_t>(tag) << 32;
  const uint64_t t0 = wall_clock64();
  for (int polls = 1;; ++polls) {
    if (reads) got = __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__all(static_cast<uint32_t>(got >> 32) == tag)) break;
    if (too_long(a, t0, polls)) {
      late = true;
      break;
    }
  }
  constexpr int kQuadFirst = 0x00;  // quad_perm [0,0,0,0]
  const float theirs =
      q3::dpp_f32<kQuadFirst>(__uint_as_float(static_cast<uint32_t>(got)));
  v = mine ? v : theirs;
  v += q3::dpp_f32<q3::kDppHalfMirror>(v);
  v += q3::dpp_f32<q3::kDppMirror>(v);
  return v;
}

// Half a head of the next layer's q, k, v: dims 32 hf .. + 31 and 64 + 32 hf
// .. + 31, so that RoPE's pairs are inside; the two halves exchange their sums
// of squares.  Wave w has 16 of the 64 weight rows (w % 4) and a half of K (w /
// 4), all of it in registers while it waits.  (A whole head in one block: its
// 256 KB do not fit the registers, and what was left to read after the wait
// took 2.5 us at the 46 GB/s of one CU.)  kAlone: a launch of its own, rows
// 16 rb .. of h.
template <bool kAlone, bool kFirst>
__device__ __forceinline__ int qkv_phase(const ChainArgs& a, Shared& sh, int blk, int rb,
                                         uint32_t launch, q3::f32x4 (*red)[64], uint16_t* a_s,
                                         uint16_t* nw_s) {
  __shared__ float rms_s[kRows];
  __shared__ __attribute__((aligned(16))) uint16_t y_s[kRows][kHeadD / 2];
  __shared__ int64_t pos_s[kRows], phys_s[kRows];
  __shared__ int off_s[kRows];
  const int head = blk >> 1, hf = blk & 1;
  const int M = kAlone ? min(kRows, a.M - kRows * rb) : a.M;
  const uint16_t* h = a.h_out + static_cast<int64_t>(kRows * rb) * a.h_s;
  const float* ss = a.ss_out + kRows * rb * (a.K / 16);
  const int tid = static_cast<int>(fresh(threadIdx.x)), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ct = wave & 3, kh = wave >> 2;
  const int r16 = lane & 15;
  const int lrow = lane >> 2, lkg = 8 * (lane & 3);
  const int perm_addr = 4 * (4 * r16 + (lane >> 4));
  const int steps = a.K / 2 / kKStep;  // at most kQkvSteps
  const int pitch = a.K + 8;
  const int wrow = head * kHeadD + (ct < 2 ? 0 : kHeadD / 2 - 32) + 32 * hf + 16 * ct;
  const Rows wr{a.qkv_w + wrow * a.qkv_ws, static_cast<int>((15 * a.qkv_ws + a.K) * 2), steps};
  const uint32_t woff = static_cast<uint32_t>((lrow * a.qkv_ws + lkg + kh * (a.K / 2)) * 2);
  q3::u32x4 b[kQkvSteps];
#pragma unroll
  for (int u = 0; u < kQkvSteps; ++u)
    b[u] = kAlone ? wr.weight(woff, u) : q3::u32x4{0u, 0u, 0u, 0u};
  if (wave == 1 && lane < kRows) {
    int64_t pos, phys;
    int off;
    locate_token(a.hd, kRows * rb + lane, pos, phys, off);
    pos_s[lane] = pos;
    phys_s[lane] = phys;
    off_s[lane] = off;
  }
  for (int i = tid; i < a.K / 8; i += kThreads)
    *reinterpret_cast<q3::u32x4*>(nw_s + 8 * i) = q3::ld16(a.in_w + 8 * i);
  if constexpr (kFirst) share_launch(sh, launch);  // (there are barriers before its use)
  if (kAlone && tid == 0) sh.run = kDone;
  for (int pass = kAlone ? 1 : 0; pass < two(); ++pass) {
    if (!kAlone && pass) {
#pragma unroll
      for (int u = 0; u < kQkvSteps; ++u) b[u] = wr.weight(woff, u);
#pragma unroll
      for (int u = 0; u < kQkvSteps; ++u) b[u] = to_mfma(b[u], perm_addr);
      wait_phase<kFirst>(a, sh, kDown);
    }
    // The rows of h: chunk c = tid + i * threads of the M x K / 8 16-byte
    // chunks, at most four per thread.  Rows past M stay unwritten: a row of the
    // product depends on its own row only.
    constexpr int kPer = kRows * kMaxHidden / 8 / kThreads;
    const int tp = static_cast<int>(fresh(tid));
    const int cpr = a.K >> 3, nch = M * cpr;
    q3::u32x4 hv[kPer];
    const __amdgpu_buffer_rsrc_t hr =
        rsrc_of(h, pass ? ((M - 1) * a.h_s + a.K) * 2 : 0);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {  // (past the rows: zero)
      const int c = tp + i * kThreads, r = c / cpr;
      hv[i] = ld16_dev(hr, static_cast<uint32_t>((r * a.h_s + 8 * (c - r * cpr)) * 2));
    }
    if (wave == 0) {
      const float rms = row_rms(a, ss, M, tp & 63);
      if (lane < kRows) rms_s[lane] = rms;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int c = tp + i * kThreads;
      if (c >= nch) continue;
      const int r = c / cpr, cc = c - r * cpr;
      *reinterpret_cast<q3::u32x4*>(a_s + r * pitch + 8 * cc) =
          normed(hv[i], *reinterpret_cast<const q3::u32x4*>(nw_s + 8 * cc), rms_s[r]);
    }
    __syncthreads();
    const uint16_t* arow = a_s + (tp & 15) * pitch + 8 * ((tp & 63) >> 4) + kh * (a.K / 2);
    if constexpr (kAlone)
#pragma unroll
      for (int u = 0; u < kQkvSteps; ++u) b[u] = to_mfma(b[u], perm_addr);
    q3::f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < kQkvSteps; ++u)
      acc = q3::mfma16x16x32(q3::as_bf16x8(*reinterpret_cast<const q3::u32x4*>(
                                 arow + (u < steps ? u : 0) * kKStep)),
                             q3::as_bf16x8(b[u]), acc);
    // first half of K + second, rounded to bf16, as decode_qkv.hip
    if (kh == 1) red[ct][lane] = acc;
    __syncthreads();
    if (kh == 0) {
      const q3::f32x4 other = red[ct][lane];
#pragma unroll
      for (int i = 0; i < 4; ++i)
        y_s[4 * (lane >> 4) + i][ct * 16 + r16] = q3::bf16_bits(acc[i] + other[i]);
    }
    __syncthreads();
  }
  // 16 lanes per token as for a whole head; the quads of the other block are
  // zero here.
  if (sh.run == kDone) {  // uniform
    const int r = tid >> 4, j = tid & 15;
    if (r < M) {  // whole 16-lane groups
      const bool mine = ((j >> 2) & 1) == hf;
      const int at = 8 * (j & 3) + (j >> 3) * 32;
      const q3::u32x4 xw = mine ? *reinterpret_cast<const q3::u32x4*>(&y_s[r][at])
                                : q3::u32x4{0u, 0u, 0u, 0u};
      bool late = false;
      if (mine || head < a.hd.Hq + a.hd.Hkv)
        finish_head(a.hd, head, kRows * rb + r, j, xw, pos_s[r], phys_s[r], off_s[r],
                    [&]() { return mine && !late; }, [&](float v) {
                      return exchange_sum(a, sh.launch, rb, head, hf, r, j, v, late);
                    });
      if (late && (tid & 63) == 0) sh.run = kPartnerMissing;
    }
    if constexpr (kAlone && kFirst) arrive(a, sh);  // (this wave has no rows)
    __syncthreads();  // sh.run
  }
  return sh.run;
}

template <bool kFirst>
__device__ __forceinline__ int merge_phase(const ChainArgs& a, Shared& sh, int item,
                                           uint32_t launch) {
  const int tid = static_cast<int>(fresh(threadIdx.x)), lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hq_n = a.KO / kHeadD;
  const int task = item * kWaves + wave;  // one wave per (row, query head)
  const int b = task / hq_n, hq = task - b * hq_n;
  uint32_t y;
  if (b < a.M && merge_partials<32>(a.parts, b, hq, lane, y))
    st_dev(reinterpret_cast<uint32_t*>(a.o + b * a.o_s + hq * kHeadD + 2 * lane), y);
  if constexpr (kFirst) share_launch(sh, launch);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this wave's stores are complete
  __syncthreads();
  if (wave == 0) set_flag(a, sh, item);
  return kDone;
}

// kFirst: a block's first run, of its own item.
template <bool kFirst>
__device__ __forceinline__ int run_item(const ChainArgs& a, Shared& sh, int item,
                                        uint32_t launch, q3::f32x4 (*red)[64], uint16_t* a_s,
                                        uint16_t* nw_s) {
  if (item < a.first[kO]) return merge_phase<kFirst>(a, sh, item, launch);
  if (item < a.first[kGateUp])
    return linear_phase<kO, kFirst>(a, sh, item - a.first[kO], launch, red, nw_s);
  if (item < a.first[kDown])
    return linear_phase<kGateUp, kFirst>(a, sh, item - a.first[kGateUp], launch, red, nw_s);
  if (item < a.first[kQkv])
    return linear_phase<kDown, kFirst>(a, sh, item - a.first[kDown], launch, red, nw_s);
  return qkv_phase<false, kFirst>(a, sh, item - a.first[kQkv], 0, launch, red, a_s, nw_s);
}

// The kernel's argument (the first, at offset 0), read anew: the rare path that
// runs another block's work keeps nothing in registers across the usual one.
__device__ __forceinline__ const ChainArgs& item_args() {
  typedef const __attribute__((address_space(4))) ChainArgs kernarg;
  kernarg* p = (kernarg*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *(const ChainArgs*)p;
}

// Two blocks per CU.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void decode_chain_kernel(ChainArgs args) {
  __shared__ q3::f32x4 red[kWaves][64];
  __shared__ __attribute__((aligned(16))) uint16_t a_s[kRows * (kMaxHidden + 8)];
  __shared__ __attribute__((aligned(16))) uint16_t nw_s[kMaxHidden];
  __shared__ Shared sh;
  const int own = blockIdx.x;
  const uint32_t launch = read_launch(args.sync);
  int item = own, run = run_item<true>(args, sh, item, launch, red, a_s, nw_s);
  while (__builtin_expect(run != kDone || item != own, 0)) {
    const ChainArgs& a = item_args();
    // the other half of the head, or what the phases before this one lack
    item = next_item(a, sh, own, run == kPartnerMissing && item == own);
    run = run_item<false>(a, sh, item, 0u, red, a_s, nw_s);
  }
  arrive(args, sh);  // (where it has not waited)
}

// The qkv phase as a launch of its own, for up to 64 rows: block (half head,
// 16-row block), the row blocks of a half head on one XCD (blocks are dealt to
// the eight in turn) where their weights meet in its L2.
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(4, 4)))
void decode_qkv_half_kernel(ChainArgs args) {
  __shared__ q3::f32x4 red[kWaves][64];
  __shared__ __attribute__((aligned(16))) uint16_t a_s[kRows * (kMaxHidden + 8)];
  __shared__ __attribute__((aligned(16))) uint16_t nw_s[kMaxHidden];
  __shared__ Shared sh;
  const int rbc = (args.M + kRows - 1) / kRows;
  const int halves = 2 * (args.hd.Hq + 2 * args.hd.Hkv);
  const int slot = static_cast<int>(blockIdx.x >> 3);
  const int half = (slot / rbc) * 8 + static_cast<int>(blockIdx.x & 7);
  const uint32_t launch = read_launch(args.sync);
  if (half < halves) {
    int item = half;
    int run = qkv_phase<true, true>(args, sh, item, slot % rbc, launch, red, a_s, nw_s);
    while (__builtin_expect(run != kDone || item != half, 0)) {
      const ChainArgs& a = item_args();
      item = run == kPartnerMissing && item == half ? half ^ 1 : half;
      __syncthreads();  // the run before this is over in every wave
      run = qkv_phase<true, false>(a, sh, item, slot % rbc, 0u, red, a_s, nw_s);
    }
  } else {
    share_launch(sh, launch);
  }
  arrive(args, sh);
}

// Blocks of the kernel resident at once on the current device (0: unknown).
int resident_blocks(void (*kernel)(ChainArgs), int (&cached)[64]) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
  if (cached[dev] == 0) {
    int cus = 0, per = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per, reinterpret_cast<const void*>(kernel), kThreads, 0) != hipSuccess)
      return 0;
    cached[dev] = cus * per;
  }
  return cached[dev];
}
// Larger grids would be answered too, but their waits would run out.
int chain_blocks() {
  static int cached[64] = {0};
  return resident_blocks(decode_chain_kernel, cached);
}
int qkv_half_blocks() {
  static int cached[64] = {0};
  return resident_blocks(decode_qkv_half_kernel, cached);
}

// Blocks per phase; false for shapes the kernel does not hold.
bool phase_blocks(int M, int hidden, int inter, int num_heads, int num_kv_heads, bool merge,
                  bool qkv, int (&first)[kPhases + 1]) {
  const int64_t KO = static_cast<int64_t>(num_heads) * kHeadD;
  if (M < 1 || M > kRows || hidden <= 0 || inter <= 0 || num_heads <= 0 || num_kv_heads <= 0 ||
      num_heads % num_kv_heads != 0 || num_heads + num_kv_heads > kMaxNormHeads)
    return false;
  // whole k-steps per wave, held in registers; rows of one head staged in
  // LDS; o_proj and down split K over eight waves, as decode_linear does from
  // 2048 on (fewer would sum in another order)
  if (hidden % (4 * kKStep) != 0 || hidden > kMaxHidden || hidden / 4 / kKStep > kMaxSteps ||
      KO < 2048 || KO % (kWaves * kKStep) != 0 || KO / kWaves / kKStep > kMaxSteps ||
      inter < 2048 || inter % (kWaves * kKStep) != 0 || inter / kWaves / kKStep > kMaxSteps)
    return false;
  const int n[kPhases] = {merge ? (M * num_heads + kWaves - 1) / kWaves : 0, hidden / 16,
                          inter / 16, hidden / 16, qkv ? 2 * (num_heads + 2 * num_kv_heads) : 0};
  first[0] = 0;
  for (int p = 0; p < kPhases; ++p) first[p + 1] = first[p] + n[p];
  return first[kPhases] <= kMaxBlocks;
}

// The next layer's part of the arguments.
int fill_qkv(ChainArgs& a, const qwen3_decode_chain_args* c, const char* who) {
  if (!c->in_norm_weight || !c->q_norm_weight || !c->k_norm_weight || !c->cos_table ||
      !c->sin_table || !c->q_out || !c->k_cache || !c->v_cache || !c->seq_lens ||
      !c->block_table)
    return q3::fail(QWEN3_EINVAL, "%s: null pointer argument", who);
  if (c->block_size <= 0 || c->num_blocks <= 0 || c->layer_idx < 0 ||
      c->layer_idx >= c->num_layers || c->table_rows < 0 || c->max_rows <= 0 ||
      c->max_pages <= 0 || c->bt_row_stride < c->max_pages || !(c->head_eps >= 0.f))
    return q3::fail(QWEN3_EINVAL, "%s: bad sizes", who);
  bool ok = q3::aligned16(c->in_norm_weight) && q3::aligned16(c->qkv_weight) &&
       q3::aligned16(c->q_norm_weight) && q3::aligned16(c->k_norm_weight) &&
       q3::aligned16(c->cos_table) && q3::aligned16(c->sin_table) && q3::aligned16(c->q_out) &&
       q3::aligned16(c->k_cache) && q3::aligned16(c->v_cache) && c->qkv_row_stride % 8 == 0 &&
       c->table_row_stride % 4 == 0 && c->q_out_strides[0] % 8 == 0 &&
       c->q_out_strides[1] % 8 == 0;
  HeadArgs& hd = a.hd;
  for (int i = 0; i < 4; ++i) {
    ok = ok && c->k_cache_strides[i] % 8 == 0 && c->v_cache_strides[i] % 8 == 0;
    hd.kc[i] = c->k_cache_strides[i];
    hd.vc[i] = c->v_cache_strides[i];
  }
  a.in_w = static_cast<const uint16_t*>(c->in_norm_weight);
  a.qkv_w = static_cast<const uint16_t*>(c->qkv_weight);
  a.qkv_ws = c->qkv_row_stride;
  hd.M = c->M;
  hd.Hq = c->num_heads;
  hd.Hkv = c->num_kv_heads;
  hd.q_w = static_cast<const uint16_t*>(c->q_norm_weight);
  hd.k_w = static_cast<const uint16_t*>(c->k_norm_weight);
  hd.head_eps = c->head_eps;
  hd.cos_t = c->cos_table;
  hd.sin_t = c->sin_table;
  hd.tab_stride = c->table_row_stride;
  hd.tab_rows = c->table_rows;
  hd.positions = c->positions;
  hd.q_out = static_cast<uint16_t*>(c->q_out);
  hd.qo_s0 = c->q_out_strides[0];
  hd.qo_s1 = c->q_out_strides[1];
  hd.k_cache = static_cast<uint16_t*>(c->k_cache);
  hd.v_cache = static_cast<uint16_t*>(c->v_cache);
  hd.num_blocks = c->num_blocks;
  hd.layer = c->layer_idx;
  hd.seq_lens = c->seq_lens;
  hd.block_table = c->block_table;
  hd.bt_stride = c->bt_row_stride;
  hd.max_rows = c->max_rows;
  hd.max_pages = c->max_pages;
  hd.row_ids = c->row_ids;
  hd.bs = c->block_size;
  if (!ok) return q3::fail(QWEN3_EALIGN, "%s: tensors need 16-byte aligned rows", who);
  return QWEN3_OK;
}

}  // namespace

extern "C" size_t qwen3_decode_chain_sync_bytes(void) { return kSyncWords * sizeof(uint32_t); }

extern "C" int qwen3_decode_chain_supported(int M, int hidden, int intermediate, int num_heads,
                                            int num_kv_heads) {
  int first[kPhases + 1];
  return phase_blocks(M, hidden, intermediate, num_heads, num_kv_heads, true, true, first) &&
                 first[kPhases] <= chain_blocks()
             ? 1
             : 0;
}

extern "C" int qwen3_decode_chain_bf16(const qwen3_decode_chain_args* c, void* stream) {
  const char* who = "qwen3_decode_chain_bf16";
  if (!c || !c->o || !c->o_weight || !c->h_in || !c->h_mid || !c->h_out || !c->ss_mid ||
      !c->ss_out || !c->post_norm_weight || !c->gate_up_weight || !c->act || !c->down_weight ||
      !c->sync)
    return q3::fail(QWEN3_EINVAL, "%s: null pointer argument", who);
  if (c->M == 0) return QWEN3_OK;
  const bool merge = c->attn_workspace != nullptr, qkv = c->qkv_weight != nullptr;
  ChainArgs a{};
  if (!phase_blocks(c->M, c->hidden, c->intermediate, c->num_heads, c->num_kv_heads, merge, qkv,
                    a.first))
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: %d rows, hidden %d, intermediate %d, heads %d / %d "
                    "not supported", who, c->M, c->hidden, c->intermediate, c->num_heads,
                    c->num_kv_heads);
  if (c->h_in == c->h_mid || c->h_mid == c->h_out || !(c->eps >= 0.f))
    return q3::fail(QWEN3_EINVAL, "%s: h_mid must be a buffer of its own, eps >= 0", who);
  bool ok = q3::aligned16(c->o) && q3::aligned16(c->o_weight) && q3::aligned16(c->h_in) &&
            q3::aligned16(c->h_mid) && q3::aligned16(c->h_out) && q3::aligned16(c->ss_mid) &&
            q3::aligned16(c->ss_out) && q3::aligned16(c->post_norm_weight) &&
            q3::aligned16(c->gate_up_weight) && q3::aligned16(c->act) &&
            q3::aligned16(c->down_weight) && q3::aligned16(c->sync) && c->o_row_stride % 8 == 0 &&
            c->o_weight_row_stride % 8 == 0 && c->gate_up_row_stride % 8 == 0 &&
            c->down_row_stride % 8 == 0;
  a.M = c->M;
  a.K = c->hidden;
  a.I = c->intermediate;
  a.KO = c->num_heads * kHeadD;
  a.last_phase = qkv ? kQkv : kDown;
  a.eps = c->eps;
  if (merge) {
    const int64_t waves = c->attn_waves;
    const StreamLayout L = stream_layout(c->M, waves, c->num_heads / c->num_kv_heads);
    if (waves <= 0 || static_cast<size_t>(L.total) > c->attn_workspace_bytes)
      return q3::fail(QWEN3_EWORKSPACE, "%s: attention workspace of %lld bytes needed, %zu given",
                      who, static_cast<long long>(L.total), c->attn_workspace_bytes);
    const char* ws = static_cast<const char*>(c->attn_workspace);
    ok = ok && q3::aligned16(ws);
    a.parts = {reinterpret_cast<const float*>(ws + L.po),
               reinterpret_cast<const float*>(ws + L.plse),
               reinterpret_cast<const int32_t*>(ws + L.pref),
               reinterpret_cast<const int32_t*>(ws + L.meta), c->num_kv_heads,
               c->num_heads / c->num_kv_heads};
  }
  a.o = static_cast<uint16_t*>(c->o);
  a.o_s = c->o_row_stride;
  a.o_w = static_cast<const uint16_t*>(c->o_weight);
  a.o_ws = c->o_weight_row_stride;
  a.h_in = static_cast<const uint16_t*>(c->h_in);
  a.h_mid = static_cast<uint16_t*>(c->h_mid);
  a.h_out = static_cast<uint16_t*>(c->h_out);
  a.ss_mid = c->ss_mid;
  a.ss_out = c->ss_out;
  a.post_w = static_cast<const uint16_t*>(c->post_norm_weight);
  a.gu_w = static_cast<const uint16_t*>(c->gate_up_weight);
  a.gu_ws = c->gate_up_row_stride;
  a.act = static_cast<uint16_t*>(c->act);
  a.down_w = static_cast<const uint16_t*>(c->down_weight);
  a.down_ws = c->down_row_stride;
  a.sync = c->sync;
  a.wait_ticks = c->wait_ticks ? c->wait_ticks : kWaitTicks;
  a.h_s = c->hidden;
  if (qkv)
    if (const int rc = fill_qkv(a, c, who)) return rc;
  if (!ok) return q3::fail(QWEN3_EALIGN, "%s: tensors need 16-byte aligned rows", who);
  // rows of o and of a weight tile inside 32-bit offsets, and not overlapping
  const int64_t strides[5][2] = {{c->o_weight_row_stride, a.KO}, {c->gate_up_row_stride, a.K},
                                 {c->down_row_stride, a.I},
                                 {qkv ? c->qkv_row_stride : a.K, a.K},
                                 {c->M > 1 ? c->o_row_stride : a.KO, a.KO}};
  for (const auto& st : strides)
    if (st[0] < st[1] || st[0] > (int64_t{1} << 24))
      return q3::fail(QWEN3_EINVAL, "%s: row stride %lld of %lld columns", who,
                      static_cast<long long>(st[0]), static_cast<long long>(st[1]));
  if (a.first[kPhases] > chain_blocks())
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: %d blocks cannot be resident at once", who,
                    a.first[kPhases]);
  q3::clear_error();
  hipLaunchKernelGGL(decode_chain_kernel, dim3(static_cast<unsigned>(a.first[kPhases])),
                     dim3(kThreads), 0, static_cast<hipStream_t>(stream), a);
  return q3::launch_status(who);
}

namespace {
// Blocks of the half-head launch; 0 for shapes the kernel does not hold.
int64_t half_blocks(int M, int hidden, int num_heads, int num_kv_heads) {
  if (M < 1 || M > kMaxRowBlocks * kRows || num_heads <= 0 || num_kv_heads <= 0 ||
      num_heads + num_kv_heads > kMaxNormHeads || hidden <= 0 || hidden % (2 * kKStep) != 0 ||
      hidden > kMaxHidden)
    return 0;
  return q3::cdiv(2 * (num_heads + 2 * num_kv_heads), 8) * 8 * ((M + kRows - 1) / kRows);
}
}  // namespace

extern "C" int qwen3_decode_qkv_half_supported(int M, int hidden, int num_heads,
                                               int num_kv_heads) {
  const int64_t blocks = half_blocks(M, hidden, num_heads, num_kv_heads);
  return blocks > 0 && blocks <= qkv_half_blocks() ? 1 : 0;
}

extern "C" int qwen3_decode_qkv_half_bf16(const qwen3_decode_chain_args* c, int64_t h_row_stride,
                                          void* stream) {
  const char* who = "qwen3_decode_qkv_half_bf16";
  if (!c || !c->h_out || !c->ss_out || !c->qkv_weight || !c->sync)
    return q3::fail(QWEN3_EINVAL, "%s: null pointer argument", who);
  if (c->M == 0) return QWEN3_OK;
  const int64_t blocks = half_blocks(c->M, c->hidden, c->num_heads, c->num_kv_heads);
  if (blocks == 0)
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: %d rows, hidden %d, heads %d / %d not supported", who,
                    c->M, c->hidden, c->num_heads, c->num_kv_heads);
  if (h_row_stride < c->hidden || h_row_stride > (int64_t{1} << 24) ||
      c->qkv_row_stride < c->hidden || c->qkv_row_stride > (int64_t{1} << 24) || !(c->eps >= 0.f))
    return q3::fail(QWEN3_EINVAL, "%s: bad row strides or eps", who);
  ChainArgs a{};
  a.M = c->M;
  a.K = c->hidden;
  a.eps = c->eps;
  a.h_out = static_cast<uint16_t*>(c->h_out);
  a.h_s = h_row_stride;
  a.ss_out = c->ss_out;
  a.sync = c->sync;
  a.wait_ticks = c->wait_ticks ? c->wait_ticks : kWaitTicks;
  if (const int rc = fill_qkv(a, c, who)) return rc;
  if (!q3::aligned16(c->h_out) || !q3::aligned16(c->ss_out) || !q3::aligned16(c->sync) ||
      h_row_stride % 8 != 0)
    return q3::fail(QWEN3_EALIGN, "%s: tensors need 16-byte aligned rows", who);
  if (blocks > qkv_half_blocks())
    return q3::fail(QWEN3_EUNSUPPORTED, "%s: %lld blocks cannot be resident at once", who,
                    static_cast<long long>(blocks));
  q3::clear_error();
  hipLaunchKernelGGL(decode_qkv_half_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0,
                     static_cast<hipStream_t>(stream), a);
  return q3::launch_status(who);
}
