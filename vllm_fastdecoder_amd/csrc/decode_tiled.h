// Shared device code of the two tiled decode kernels (decode_valu.hip and
// decode_mfma.hip): launch parameters, task decomposition, the K/V stream
// helpers and the cross-wave merge.
//
// Semantics follow the reference's host-tier kernel decode_attn
// (fastdecode/csrc/cpu_attn.cpp:298-411) and the GPU-tier FlashAttention
// decode call it is merged with (fastdecode/backend.py:305-316): for every
// (sequence i, query head h) the softmax-weighted sum of V over the tokens of
// the listed blocks, plus the natural-log LSE of the scaled scores, with
// out = 0 and lse = -inf for an empty row (cpu_attn.cpp:324-331).
//
// A launch covers one KV tier (a partial, as in the reference) or two: the
// fused split path walks a row's HBM-tier blocks and then its host-tier
// blocks as one list, so the tier merge of backend.py:354-356 happens inside
// the kernel. Each tier has its own cache pointers, strides, block table and
// lengths; the tier of a block is wave-uniform.
//
// Work decomposition (memory-bound design):
//   * a task = (sequence, kv head, range of up to `split_blocks` blocks) is
//     one 256-thread workgroup; its 4 wavefronts take the range's blocks
//     round-robin and each keeps its own softmax state, merged once through
//     LDS at the end. Longer rows are split and a small combine kernel merges
//     the split partials;
//   * the next block's K and V are in flight (register double buffer) while
//     the current block is reduced; 16-byte buffer loads with a non-temporal
//     hint (each byte is read once);
//   * the G = H/KVH query heads of a kv head share every K/V load.
#pragma once

#include <string.h>

#include <atomic>
#include <type_traits>

#include "fd_common.h"

namespace fd {

constexpr int kTileTokens = 16;         // tokens per block in the tiled kernels
constexpr int kWavesPerTask = 4;        // wavefronts sharing one task
constexpr int kMaxWaveBlocks = kWave;   // a wave's block ids of a task fit one VGPR
constexpr int kMaxSplitBlocks = kWavesPerTask * kMaxWaveBlocks;
constexpr int kMaxDevices = 64;         // per-device launch settings cached
constexpr int kMaxHeadGroup = 512;      // largest H / KVH the tiled kernels take (in passes)
constexpr int kMaxBlockSize = 1024;     // largest cache block size they take (16-token tiles)

// One KV tier as the tiled kernels see it (16-bit elements).
struct TierParams {
  const uint16_t* k;
  const uint16_t* v;
  int64_t sb, sh, st;  // element strides: block, head, token
  int64_t num_blocks;
  uint32_t run_bytes;    // extent of one (block, head) run: (15 * st + D) elements
  uint32_t k_run_bytes;  // extent of the K resource: run_bytes, or the K + V run if kv_adj
  bool kv_adj;           // V follows K in every token row (v == k + D): one load reads both
  const int32_t* bt;
  int64_t bt_stride;
  int32_t bt_width;
  const int32_t* lens;
};

struct TiledParams {
  const uint16_t* q;
  int64_t q_ss, q_sh;
  TierParams tier[2];    // tier[1] is read by two-tier launches only
  const int32_t* order;  // optional processing order of the sequences
  int32_t n, H, KVH;
  int32_t D;       // head size (<= the kernel's D; lanes past it only stand by)
  int32_t BS;      // cache block size: tpb 16-token tiles, each handled as a kernel block
  int32_t tpb;     // tiles per cache block (BS / 16)
  int32_t hpk;     // query heads per kv head (H / KVH)
  int32_t passes;  // head groups per kv head: ceil(hpk / the kernel's G)
  float scale_log2;  // softmax scale * log2(e)
  void* out;
  int64_t out_ss, out_sh;
  bool out_f32;
  float* lse;
  int64_t lse_sh;
  float* part_o;    // [n, H, S, D] fp32 (normalised partial outputs)
  float* part_lse;  // [n, H, S] fp32 (natural-log LSE of each partial)
  // balanced cuts: [slots, H, D] sums of p V and [slots, H, 2] (max, sum of p)
  int32_t S;        // max splits per (sequence, kv head)
  int32_t split_blocks;
  int32_t wave_blocks;  // blocks per working wave (0: every wave works; wave_blocks())
  int32_t bal_parts;  // > 0: balanced cuts (balanced_task()): parts per kv-head pass aimed at
  int32_t bal_min;    // balanced cuts: blocks per part at least
  int32_t bal_whole;  // balanced cuts: blocks a cut has to save (whole rows otherwise)
  int32_t host_wgs;   // balanced cuts of two tiers: workgroups that take tier 1's blocks alone
                      // (balanced_task()), 0: tasks over both tiers' blocks
  float bal_share;    // balanced cuts: blocks of one task's own rate in the time in which HBM
                      // delivers one block of every row of all kv-head passes together
  uint64_t* counters; // balanced cuts: arrivals per (sequence, kv-head pass) (count_arrival())
  uint64_t launch;    // balanced cuts: this launch's number, kArrivalBits up
  int32_t counter_stride;  // balanced cuts: counters are this many words apart
  bool tier_waves;  // two tiers: a task's waves are divided between them (wave_blocks())
  bool xcd_group;   // adjacent kv heads of a row on one XCD (xcd_task)
  uint64_t* timeline;  // measurement only: kTimelineSlots stamps per workgroup (NULL: none)
};

// Time stamps of one workgroup in a timeline launch (s_memrealtime, 100 MHz):
// task start, wave 0's block ids in registers, each wave's end of its block
// loop, the end of the task, and a word with the task's block count (bits
// 0-15), working waves (16-23) and sequence (32-63).
constexpr int kTimelineSlots = 8;
enum TimelineSlot { kTlStart = 0, kTlIds = 1, kTlLoop0 = 2, kTlEnd = 6, kTlInfo = 7 };

// Launchers of the kernel families (decode_valu.hip, decode_mfma.hip,
// decode_mm.hip, decode_f32.hip).
hipError_t launch_valu(const TiledParams& tp, unsigned tasks, const SplitPlan& sp, int kv_dtype,
                       int D, int G, bool two_tiers, hipStream_t s);
hipError_t launch_mfma(const TiledParams& tp, unsigned tasks, const SplitPlan& sp, int kv_dtype,
                       int D, int G, bool two_tiers, hipStream_t s);
hipError_t launch_mm(const TiledParams& tp, unsigned tasks, const SplitPlan& sp, int kv_dtype,
                     int D, bool two_tiers, hipStream_t s);
hipError_t launch_f32(const TiledParams& tp, unsigned tasks, const SplitPlan& sp, int D, int G,
                      bool two_tiers, hipStream_t s);

// Dynamic LDS that caps `kernel` at `wgs` workgroups per CU (decode_partial.hip).
unsigned cap_lds(const void* kernel, int wgs, std::atomic<int>* cache);
// Workgroups of `kernel` one CU holds at once without a cap, 0 if unknown
// (decode_partial.hip).
int natural_wgs_per_cu(const void* kernel, std::atomic<int>* cache);

// Launches `Kernel` with the occupancy cap when the plan asks for it. The
// kernel is a template argument so that each kernel has its own settings
// cache: the reserve depends on the kernel's static LDS (every kernel here
// has the type void(TiledParams), so a cache keyed by the pointer's type
// would hand the first kernel's reserve to all the others). A plan with an
// occupancy query launches nothing: it only reports the kernel's occupancy.
template <void (*Kernel)(TiledParams)>
hipError_t launch_capped(const TiledParams& tp, unsigned tasks, const SplitPlan& sp,
                         hipStream_t s) {
  if (sp.occupancy_query != nullptr) {
    static std::atomic<int> occupancy[kMaxDevices] = {};
    *sp.occupancy_query = natural_wgs_per_cu(reinterpret_cast<const void*>(Kernel), occupancy);
    return hipSuccess;
  }
  static std::atomic<int> cache[kMaxDevices] = {};
  const unsigned lds =
      sp.wg_cap > 0 ? cap_lds(reinterpret_cast<const void*>(Kernel), sp.wg_cap, cache) : 0;
  hipLaunchKernelGGL(Kernel, dim3(tasks), dim3(kWave * kWavesPerTask), lds, s, tp);
  return hipGetLastError();
}

// ---------------------------------------------------------------- loads

// 16 bytes of 16-bit elements (8 values).
struct Vec8 {
  uint32_t w[4];
};

__device__ __forceinline__ Vec8 ld16(const uint16_t* p) {
  const uint4 u = *reinterpret_cast<const uint4*>(p);
  return Vec8{{u.x, u.y, u.z, u.w}};
}

// Buffer resource over `bytes` bytes at `base` (gfx9 raw buffer, dword data
// format); loads past `bytes` return zero instead of touching memory.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const uint16_t* base,
                                                           uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(base), (short)0, (int)bytes,
                                           0x00020000);
}

// Cache policy of the KV stream: non-temporal (each byte is read once; the
// hint keeps the stream from displacing other lines). Measured +7.6 % at the
// vicuna-7b shape over the default policy.
constexpr int kKvLoadPolicy = 2;
// The default policy, for loads whose cache lines are read again soon by
// another load: a line split between two loads of one wave (the matrix-core
// kernel's K column slices at head sizes other than 64 and 128) or between
// the runs of neighbouring heads (K + V runs of 4D bytes that are not whole
// lines in vLLM's layout, e.g. D = 80). There, non-temporal lines are often
// gone before their second reader comes and are fetched twice.
constexpr int kKvLoadKeep = 0;

// 16 bytes at byte `off` (per lane) + `soff` (wave-uniform) of the resource.
template <int POL = kKvLoadPolicy>
__device__ __forceinline__ Vec8 buffer_ld16(__amdgpu_buffer_rsrc_t r, uint32_t off,
                                            uint32_t soff = 0) {
  const auto u = __builtin_amdgcn_raw_buffer_load_b128(r, off, soff, POL);
  return Vec8{{(uint32_t)u[0], (uint32_t)u[1], (uint32_t)u[2], (uint32_t)u[3]}};
}

// Loads that read K and V of a token together (a kv_adj tier) leave K and V
// interleaved in each pair of loads x, y. At D = 128 (16-lane rows, two
// tokens per load) x = [K a, V a, K b, V b] and y = [K c, V c, K d, V d]; one
// v_permlane16_swap per dword regroups them into x = [K a, K c, K b, K d] and
// y = [V a, V c, V b, V d], the layout of separate K and V loads. At D = 256
// (one token per load) v_permlane32_swap does the same with 32-lane halves:
// x = [K a, V a], y = [K c, V c] -> x = [K a, K c], y = [V a, V c].
template <int D>
__device__ __forceinline__ void split_kv(Vec8& x, Vec8& y) {
  static_assert(D == 128 || D == 256, "K and V halves of 16 or 32 lanes");
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if constexpr (D == 128) {
      const auto r = __builtin_amdgcn_permlane16_swap(x.w[e], y.w[e], false, false);
      x.w[e] = r[0];
      y.w[e] = r[1];
    } else {
      const auto r = __builtin_amdgcn_permlane32_swap(x.w[e], y.w[e], false, false);
      x.w[e] = r[0];
      y.w[e] = r[1];
    }
  }
}

// 16 bytes at `p` through a global load with the non-temporal hint (the
// same cache policy as kKvLoadPolicy). Callers keep `p` inside the cache.
__device__ __forceinline__ Vec8 global_ld16(const char* p) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 u = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return Vec8{{u[0], u[1], u[2], u[3]}};
}

template <typename T>
__device__ __forceinline__ float dot8(const Vec8& a, const Vec8& b, float acc) {
  acc = dot2(T{}, a.w[0], b.w[0], acc);
  acc = dot2(T{}, a.w[1], b.w[1], acc);
  acc = dot2(T{}, a.w[2], b.w[2], acc);
  acc = dot2(T{}, a.w[3], b.w[3], acc);
  return acc;
}

template <typename T>
__device__ __forceinline__ void axpy8(float p, const Vec8& v, float* acc) {
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    acc[2 * e] = __builtin_fmaf(p, lo_f32(T{}, v.w[e]), acc[2 * e]);
    acc[2 * e + 1] = __builtin_fmaf(p, hi_f32(T{}, v.w[e]), acc[2 * e + 1]);
  }
}

// Writes 8 consecutive outputs starting at element `off` of `out` (fp32
// when `f32` is set or the KV is fp32, else the 16-bit KV type).
template <typename T>
__device__ __forceinline__ void store8(void* out, int64_t off, bool f32, const float* o) {
  if (std::is_same<T, F32>::value || f32) {
    float4* p = reinterpret_cast<float4*>(static_cast<float*>(out) + off);
    p[0] = make_float4(o[0], o[1], o[2], o[3]);
    p[1] = make_float4(o[4], o[5], o[6], o[7]);
  } else if constexpr (!std::is_same<T, F32>::value) {
    uint4 u;
    u.x = to_out(T{}, o[0]) | (uint32_t(to_out(T{}, o[1])) << 16);
    u.y = to_out(T{}, o[2]) | (uint32_t(to_out(T{}, o[3])) << 16);
    u.z = to_out(T{}, o[4]) | (uint32_t(to_out(T{}, o[5])) << 16);
    u.w = to_out(T{}, o[6]) | (uint32_t(to_out(T{}, o[7])) << 16);
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + off) = u;
  }
}

// The same for 4 outputs.
template <typename T>
__device__ __forceinline__ void store4(void* out, int64_t off, bool f32, const float* o) {
  if (std::is_same<T, F32>::value || f32) {
    *reinterpret_cast<float4*>(static_cast<float*>(out) + off) =
        make_float4(o[0], o[1], o[2], o[3]);
  } else if constexpr (!std::is_same<T, F32>::value) {
    uint2 u;
    u.x = to_out(T{}, o[0]) | (uint32_t(to_out(T{}, o[1])) << 16);
    u.y = to_out(T{}, o[2]) | (uint32_t(to_out(T{}, o[3])) << 16);
    *reinterpret_cast<uint2*>(static_cast<uint16_t*>(out) + off) = u;
  }
}

// ---------------------------------------------------------------- tasks

// One task of a tiled launch: (sequence i, kv head kh, split) and the range
// [b_begin, b_end) of the row's nb blocks it covers. With two tiers the row's
// blocks are tier 0's nba blocks followed by tier 1's.
struct Task {
  int i, kh, split;
  int h0;      // first query head of the task: kh * hpk + its head group * G
  int gcount;  // query heads of the task (<= G; the kernel's other head slots
               // repeat the last one and write nothing)
  int la, lb;  // tokens of the row in tier 0 / tier 1 (<= 0: none)
  int nba, nb;
  int b_begin, b_end, nsplit;
  bool range_bad;  // a length needs more blocks than its table has
  int kp, slot0;   // balanced cuts: kv-head pass of the task, first part of its row,
  int pos;         // and the row's place in the launch's list of rows
};

// blockIdx.x -> task: kv head fastest, then head group (one unless a kv head
// has more query heads than the kernel's G), then sequence (in the caller's order
// when one is given, e.g. longest rows first so the last workgroups dispatched
// are short ones), split slowest. Split-major order matters on this GPU:
// workgroups are dealt round-robin to the XCDs and, inside an XCD, to its
// shader engines, so interleaving each row's splits (most of whose later
// splits are empty) would hand the empty workgroups to a fixed half of the
// engines and idle them; split-major keeps the empty ones together at the end.
// False when the workgroup has nothing to do: an order entry outside [0, n),
// or a split past the row's last block.
// Workgroups are dealt round-robin to the GPU's 8 XCDs, each with its own
// L2. With p.xcd_group set, within every 32 consecutive workgroups XCD x
// receives four (dispatch rounds 0-3) and they take logical tasks 4x .. 4x+3
// of the 32, i.e. four adjacent kv heads of one row. Where a token's K + V
// runs of adjacent heads share 128-byte lines (2 D elements of 2 bytes, not
// a multiple of 128 bytes: D = 80, 112, ...), the shared lines are then read
// by tasks of one XCD at about the same time (four heads span 16 D bytes,
// always whole lines); measured +2-3 % at D = 80 / 96 / 112, but -0.7 % at
// D = 128 and -3 % on small batches, so the host sets the flag only for
// head sizes that are not multiples of 64. A trailing partial group of 32
// keeps the identity order; the longest-first row order holds at a
// granularity of 32 workgroups.
constexpr int kXcds = 8;
constexpr int kXcdHeads = 4;
__device__ __forceinline__ int xcd_task(int b, int tasks) {
  constexpr int kGroup = kXcds * kXcdHeads;
  const int g = b / kGroup, r = b % kGroup;
  return (g + 1) * kGroup <= tasks ? g * kGroup + kXcdHeads * (r % kXcds) + r / kXcds : b;
}

// Balanced cuts: how the launch's tasks are drawn from the rows' lengths
// themselves, on the device. The launch wants at most S = bal_parts parts per
// kv-head pass (as many workgroups as the CUs take at once, one round): a
// part holds at most c blocks, a row of nb blocks is cut into ceil(nb / c)
// parts of equal size (+-1), a row without blocks is one part, and c is the
// first size tried at which all rows make at most S parts. Then all tasks
// start together and stream about the same share, however uneven the rows
// and however wide the table is. The host cannot do this: it sees neither
// the lengths nor (without a token total) their sum. Whatever c the search
// ends at, there are at most S + n parts (c >= N / S for the N blocks of all
// rows), or N / 256 + n when parts reach the 256 blocks a task can hold: the
// grid's bound. Workgroups past the last part return.
//
// Two tiers, tier 1 over the link (p.host_wgs > 0): a CU returns vector loads
// in order, so a wave that waits for the link holds up every HBM load of its
// CU, and a launch whose tasks read both took about the sum of both times.
// There the first host_wgs workgroups take all of tier 1's blocks, each of
// their waves a part of its own at a time (adjacent waves adjacent kv heads
// of the same blocks, one run in the host tier's layout), and the parts above
// are cut from tier 0's blocks alone. A row's parts of both kinds merge the
// same way. Parts of tier 1 hold ceil(N1 P / waves) blocks of its N1 blocks
// and P kv-head passes, at most the 64 ids a wave holds.
//
// Every wave works the cut out by itself from the n lengths (one load per 64
// rows, all in flight together, then DPP scans): the same chain of dependent
// loads as a task with a dispatch order, lengths -> block ids -> K.
constexpr int kBalChunks = 8;                  // lengths a lane holds
constexpr int kMaxBalRows = kBalChunks * kWave;  // rows of a balanced launch
constexpr int kMaxBalPairs = FD_DECODE_COUNTERS / 2;  // (sequence, kv-head pass) counters

// Inclusive prefix sum over the wave: row shifts within each 16 lanes, then
// the rows' last lanes broadcast to the rows after them.
__device__ __forceinline__ int wave_scan(int x) {
  x += __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false);  // row_shr:1
  x += __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false);  // row_shr:2
  x += __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false);  // row_shr:4
  x += __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false);  // row_shr:8
  x += __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1, 3
  x += __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2, 3
  return x;
}

__device__ __forceinline__ int wave_max_int(int x) {  // of values >= 0
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x111, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x112, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x114, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x118, 0xF, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x142, 0xA, 0xF, false));
  x = max(x, __builtin_amdgcn_update_dpp(0, x, 0x143, 0xC, 0xF, false));
  return __builtin_amdgcn_readlane(x, kWave - 1);
}

// Blocks of a row of la / lb tokens, of tier 0 alone or of both (0 when a
// length is past its table: such a row is one part, which writes its NaN).
template <bool TWO>
__device__ __forceinline__ int row_blocks(const TiledParams& p, int la, int lb, bool both) {
  if (la > p.tier[0].bt_width * p.BS || (TWO && lb > p.tier[1].bt_width * p.BS)) return 0;
  return (max(la, 0) + kTileTokens - 1) / kTileTokens +
         (TWO && both ? (max(lb, 0) + kTileTokens - 1) / kTileTokens : 0);
}

// a / d for 0 <= a < 2^22 and d > 0, rcp = 1 / d within a few ulp: the
// product is within one of the quotient (the compiler's general division is
// ~20 dependent instructions, and a task's start waits for several).
__device__ __forceinline__ int small_div(int a, int d, float rcp) {
  int q = (int)((float)a * rcp);
  const int r = a - q * d;
  q += r >= d ? 1 : 0;
  q -= r < 0 ? 1 : 0;
  return q;
}
__device__ __forceinline__ float fast_rcp(int d) { return __builtin_amdgcn_rcpf((float)d); }

constexpr int kMaxBalBlocks = 1 << 20;  // table width of a balanced launch, in 16-token tiles
constexpr int kBalTries = 6;            // part sizes tried

// Task f of a balanced launch: part f / P of kv-head pass f % P. TIERED: the
// launch has host workers; tier 0's parts, or with `host` set tier 1's, their
// blocks counted within the tier.
template <int G, bool TWO, bool TIERED, int kBalChunks>
__device__ __forceinline__ bool balanced_task(const TiledParams& p, Task& t, int f, bool host) {
  const int lane = threadIdx.x & (kWave - 1);
  static_assert(TWO || !TIERED, "host workers take a second tier");
  int row[kBalChunks], la[kBalChunks], lb[kBalChunks];
  int parts[kBalChunks];  // of the row's blocks (tiered: of tier 0's)
  bool skips = false;     // the caller's order lists an entry outside [0, n)
#pragma unroll
  for (int c = 0; c < kBalChunks; ++c) {
    row[c] = c * kWave + lane;
    la[c] = lb[c] = 0;
    if (c == 0 || c * kWave < p.n) {
      const int r = min(c * kWave + lane, p.n - 1);
      la[c] = p.tier[0].lens[r];
      if constexpr (TWO) lb[c] = p.tier[1].lens[r];
      if (p.order != nullptr) skips |= (unsigned)p.order[r] >= (unsigned)p.n;
    }
  }
  const int P = p.KVH * p.passes;
  const int j = small_div(f, P, fast_rcp(P));  // part; kv-head passes run fastest
  t.kp = f - j * P;
  const int pass = small_div(t.kp, p.KVH, fast_rcp(p.KVH));
  t.kh = t.kp - pass * p.KVH;
  t.h0 = t.kh * p.hpk + pass * G;
  t.gcount = min(G, p.hpk - pass * G);
  // A permutation of the rows changes nothing here; an order with entries
  // outside [0, n) leaves the rows it does not list to the caller.
  if (__ballot(skips) != 0) {
#pragma unroll
    for (int c = 0; c < kBalChunks; ++c) {
      row[c] = c * kWave + lane < p.n ? p.order[c * kWave + lane] : p.n;
      const bool on = (unsigned)row[c] < (unsigned)p.n;
      la[c] = on ? p.tier[0].lens[row[c]] : 0;
      if constexpr (TWO) lb[c] = on ? p.tier[1].lens[row[c]] : 0;
    }
  }
  auto listed = [&](int c) -> bool { return (unsigned)row[c] < (unsigned)p.n; };
  // blocks of lane's row of chunk c: those the parts are cut from, and tier
  // 1's where it has parts of its own
  auto blocks = [&](int c) -> int {
    return listed(c) ? row_blocks<TWO>(p, la[c], lb[c], !TIERED) : 0;
  };
  auto host_blocks = [&](int c) -> int {
    return TIERED && listed(c) && row_blocks<TWO>(p, la[c], lb[c], true) > 0
               ? (max(lb[c], 0) + kTileTokens - 1) / kTileTokens
               : 0;
  };
  int sum = 0, longest = 0, hsum = 0;
#pragma unroll
  for (int c = 0; c < kBalChunks; ++c) {
    parts[c] = 0;
    if (c == 0 || c * kWave < p.n) {
      const int nb = blocks(c);
      sum += nb;
      longest = max(longest, nb);
      if constexpr (TIERED) hsum += host_blocks(c);
    }
  }
  const int total = __builtin_amdgcn_readlane(wave_scan(sum), kWave - 1);
  // First size: as many parts as wanted if rows end half a part short of a
  // whole one on average; then larger by the share of parts too many.
  const int want = p.bal_parts;
  int size = (int)((float)total * __builtin_amdgcn_rcpf((float)want - 0.5f * (float)min(want, p.n)));
  size = max(max(size, p.bal_min), (total + want - 1) / want);
  // Whole rows where cutting saves less than the parts' merge costs: the
  // longest row at a task's own rate against the parts, or HBM's time for all
  // rows if that is longer.
  if (wave_max_int(longest) <= max(size, (int)(p.bal_share * (float)total)) + p.bal_whole)
    size = kMaxSplitBlocks;
  size = __builtin_amdgcn_readfirstlane(min(size, kMaxSplitBlocks));
  for (int tries = 0;; ++tries) {
    const float rcp = fast_rcp(size);
    int count = 0;
#pragma unroll
    for (int c = 0; c < kBalChunks; ++c) {
      if (c == 0 || c * kWave < p.n) {
        // (a row all in tier 1 has no part of tier 0; an empty one has one part)
        const int least = listed(c) && (!TIERED || host_blocks(c) == 0) ? 1 : 0;
        parts[c] = max(least, small_div(blocks(c) + size - 1, size, rcp));
        count += parts[c];
      }
    }
    const int all = __builtin_amdgcn_readlane(wave_scan(count), kWave - 1);
    if (all <= want || size >= kMaxSplitBlocks || tries >= kBalTries) break;
    const float grow = (float)size * (float)(all - want) * __builtin_amdgcn_rcpf((float)want);
    size = __builtin_amdgcn_readfirstlane(min(size + 1 + (int)(0.5f * grow), kMaxSplitBlocks));
  }
  int hsize = 1;  // tier 1's blocks per part
  if constexpr (TIERED) {
    const int htotal = __builtin_amdgcn_readlane(wave_scan(hsum), kWave - 1);
    hsize = (int)((float)htotal * (float)P *
                  __builtin_amdgcn_rcpf((float)(kWavesPerTask * p.host_wgs))) + 1;
    hsize = __builtin_amdgcn_readfirstlane(min(max(hsize, 1), kMaxWaveBlocks));
  }
  const float hrcp = fast_rcp(hsize);
  int base = 0, hbase = 0;  // parts of the rows before chunk c, of either kind
#pragma unroll
  for (int c = 0; c < kBalChunks; ++c) {
    if (c > 0 && c * kWave >= p.n) break;
    const int nh = TIERED ? host_blocks(c) : 0;
    const int hparts = TIERED ? small_div(nh + hsize - 1, hsize, hrcp) : 0;
    const int upto = base + wave_scan(parts[c]);  // parts up to and with this lane's row
    const int hupto = TIERED ? hbase + wave_scan(hparts) : 0;
    const int end = __builtin_amdgcn_readlane(upto, kWave - 1);
    const int hend = TIERED ? __builtin_amdgcn_readlane(hupto, kWave - 1) : 0;
    if (j < (host ? hend : end)) {
      // the lane of part j's row
      const int at = __popcll(host ? __ballot(hupto <= j) : __ballot(upto <= j));
      t.i = __builtin_amdgcn_readlane(row[c], at);
      t.pos = c * kWave + at;
      t.la = __builtin_amdgcn_readlane(la[c], at);
      t.lb = __builtin_amdgcn_readlane(lb[c], at);
      t.nba = t.la > 0 ? (t.la + kTileTokens - 1) / kTileTokens : 0;
      const int np = __builtin_amdgcn_readlane(parts[c], at);
      const int nhp = TIERED ? __builtin_amdgcn_readlane(hparts, at) : 0;
      const int first = __builtin_amdgcn_readlane(upto, at) - np;
      const int hfirst = TIERED ? __builtin_amdgcn_readlane(hupto, at) - nhp : 0;
      const int nbh = TIERED ? __builtin_amdgcn_readlane(nh, at) : 0;
      const int nb0 = __builtin_amdgcn_readlane(blocks(c), at);  // blocks the np parts are cut from
      t.nb = nb0 + nbh;
      t.nsplit = np + nhp;
      t.slot0 = first + hfirst;
      const int k = host ? j - hfirst : j - first;
      const int of = host ? nhp : np, nbk = host ? nbh : nb0;
      t.split = host ? np + k : k;
      // the first `more` parts hold one block more than the others
      const int each = small_div(nbk, of, fast_rcp(of));
      const int more = nbk - each * of;
      t.b_begin = k * each + min(k, more);
      t.b_end = t.b_begin + each + (k < more ? 1 : 0);
      t.range_bad = t.la > p.tier[0].bt_width * p.BS || (TWO && t.lb > p.tier[1].bt_width * p.BS);
      return true;
    }
    base = end;
    hbase = hend;
  }
  return false;
}

// BAL: the kernel takes balanced cuts (tasks of at most 16 heads do).
template <int G, bool TWO, bool BAL = true>
__device__ __forceinline__ bool decode_task(const TiledParams& p, Task& t) {
  if (BAL && p.bal_parts > 0)
    return p.n <= kWave ? balanced_task<G, TWO, false, 1>(p, t, blockIdx.x, false)
                        : balanced_task<G, TWO, false, kBalChunks>(p, t, blockIdx.x, false);
  const int task = p.xcd_group ? xcd_task(blockIdx.x, gridDim.x) : (int)blockIdx.x;
  t.kh = task % p.KVH;
  int rest = task / p.KVH;
  // a kv head with more than G query heads is done in passes of up to G
  // heads, each its own task over the same blocks
  const int pass = rest % p.passes;
  rest /= p.passes;
  t.h0 = t.kh * p.hpk + pass * G;
  t.gcount = min(G, p.hpk - pass * G);
  t.split = rest / p.n;
  int i = rest % p.n;
  if (p.order != nullptr) {
    i = p.order[i];
    if ((unsigned)i >= (unsigned)p.n) return false;
  }
  t.i = i;
  t.la = p.tier[0].lens[i];
  t.lb = TWO ? p.tier[1].lens[i] : 0;
  t.nba = t.la > 0 ? (t.la + kTileTokens - 1) / kTileTokens : 0;
  const int nbb = t.lb > 0 ? (t.lb + kTileTokens - 1) / kTileTokens : 0;
  t.nb = t.nba + nbb;
  t.b_begin = t.split * p.split_blocks;
  if (t.split > 0 && t.b_begin >= t.nb) return false;
  t.b_end = min(t.nb, t.b_begin + p.split_blocks);
  t.nsplit = t.nb > 0 ? (t.nb + p.split_blocks - 1) / p.split_blocks : 1;
  t.range_bad = t.la > p.tier[0].bt_width * p.BS || (TWO && t.lb > p.tier[1].bt_width * p.BS);
  return true;
}

// Which of the launch's tiers a task's blocks lie in (the kernels' TWO, false
// or true, is the first or second).
enum TierSet { kFirstTier = 0, kBothTiers = 1, kSecondTier = 2 };

// Valid tokens of the row's block u (< 16 only for the last block of a tier).
template <int TS>
__device__ __forceinline__ int block_tokens(const Task& t, int u) {
  constexpr bool TWO = TS == kBothTiers;
  if (TS == kSecondTier) return min(kTileTokens, t.lb - u * kTileTokens);
  if (TWO && u >= t.nba) return min(kTileTokens, t.lb - (u - t.nba) * kTileTokens);
  return min(kTileTokens, t.la - u * kTileTokens);
}

// Empty row (out = 0, lse = -inf) or a length past its table (NaN), written
// by one wave of split 0.
template <typename T, int D, int G>
__device__ __forceinline__ void write_empty(const TiledParams& p, const Task& t, int lane) {
  constexpr int LPT = D / 8;
  if (lane >= LPT || lane * 8 >= p.D) return;
  const float fill = t.range_bad ? qnan() : 0.f;
  for (int g = 0; g < t.gcount; ++g) {  // gcount <= G
    const int h = t.h0 + g;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = fill;
    store8<T>(p.out, (int64_t)t.i * p.out_ss + (int64_t)h * p.out_sh + lane * 8, p.out_f32, o);
    if (lane == 0) p.lse[(int64_t)h * p.lse_sh + t.i] = t.range_bad ? qnan() : neg_inf();
  }
}

// A wave's blocks of its task are b_begin + wave + s k, s = the task's
// working waves (4 unless p.wave_blocks says fewer). Their ids are read
// once, one per lane (at most 64), range-checked together against their
// tier's cache and later picked with v_readlane; a bad id is replaced by 0
// (every read stays inside the cache) and flags the row. The wave's blocks
// from index k1 on are in tier 1.
struct WaveBlocks {
  int first;   // the wave's first block index in the row
  int stride;  // block index step between the wave's blocks (the task's working waves)
  int nw;      // blocks of this wave
  int k1;      // first of the wave's blocks in tier 1 (>= nw: none)
  int my_bid;  // lane k: id of the cache block holding the wave's k-th tile
  int my_sub;  // lane k: that tile's index inside its cache block (0 when BS = 16)
  bool bad;
};

// With p.wave_blocks > 0 a task works with as many of its waves as give
// each about that many blocks (at least one, at most four); the rest only
// take part in the merge. A short row then keeps fewer blocks in flight than
// a long one.
// A host worker wave (TS == kSecondTier) has its task to itself.
template <int TS>
__device__ __forceinline__ WaveBlocks wave_blocks(const TiledParams& p, const Task& t, int wave,
                                                  int lane) {
  constexpr bool TWO = TS == kBothTiers;
  WaveBlocks w;
  int ws = kWavesPerTask;
  if (TS == kSecondTier) {
    ws = 1;
    wave = 0;
  }
  if (TS != kSecondTier && p.wave_blocks > 0) {
    // (each wave's block ids fit its 64 lanes: nblk <= split_blocks <= 256)
    const int nblk = t.b_end - t.b_begin;
    ws = max((nblk + p.wave_blocks - 1) / p.wave_blocks,
             (nblk + kMaxWaveBlocks - 1) / kMaxWaveBlocks);
    ws = min(kWavesPerTask, max(1, ws));
  }
  w.stride = ws;
  w.first = t.b_begin + wave;
  w.nw = wave < ws && w.first < t.b_end ? (t.b_end - w.first + ws - 1) / ws : 0;
  w.k1 = TWO ? (t.nba > w.first ? (t.nba - w.first + ws - 1) / ws : 0) : w.nw;
  if constexpr (TWO) {
    // A range with blocks of both tiers, in a launch of many tasks
    // (p.tier_waves): the last `h` waves take tier 1's (one to three waves, by
    // its share of the blocks), the others tier 0's: a wave that waits for the
    // link holds up no HBM blocks, and the link is busy from the start.
    // Measured without -> with (HIP graph replay, us; the newest block of each
    // row in the host tier, 7.5 %, 30 %): 100 x U[300, 900], 32/8, bf16 89 -> 85,
    // 303 -> 301, 1312 -> 1285; 100 x U[200, 900], 32/8, fp32 178 -> 163, 565 ->
    // 570, 2698 -> 2504; 120 x U[200, 900], 16/8, D = 256 189 -> 172, 656 -> 662,
    // 2915 -> 2902; 90 x U[100, 600], 32/32 249 -> 241, 562 -> 557, 2628 -> 2608.
    // Where the tasks are fewer, the few waves on the link are what the launch
    // waits for: 8 x U[128, 1024], 32/32, fp32 54 -> 69, 177 -> 195, 799 -> 783;
    // 40 x U[200, 1500], 16/8, D = 256 87 -> 108, 354 -> 392, 1488 -> 1507; 20 x
    // U[200, 900], 64/32 79 -> 85. 24 x U[256, 1024], 32/32, three tasks per CU:
    // 83 -> 78 us. The line lies there.
    const int na = min(t.nba, t.b_end) - t.b_begin;
    const int nh = t.b_end - t.b_begin - na;
    const int h = min(kWavesPerTask - 1, max(1, (4 * nh + (na + nh) / 2) / max(na + nh, 1)));
    const int wa = kWavesPerTask - h;
    if (p.tier_waves && na > 0 && nh > 0 && ws == kWavesPerTask && na <= wa * kMaxWaveBlocks &&
        nh <= h * kMaxWaveBlocks) {
      const bool host = wave >= wa;
      w.stride = host ? h : wa;
      w.first = host ? t.b_begin + na + wave - wa : t.b_begin + wave;
      const int end = host ? t.b_end : t.b_begin + na;
      w.nw = w.first < end ? (end - w.first + w.stride - 1) / w.stride : 0;
      w.k1 = host ? 0 : w.nw;
    }
  }
  int bid = 0, sub = 0;
  bool my_bad = false;
  if (lane < w.nw) {
    // tile u of the row: tile u % tpb of the row's cache block u / tpb
    const int u = w.first + w.stride * lane;
    if (TWO && u >= t.nba) {
      const TierParams& tp = p.tier[1];
      const int ut = u - t.nba;
      bid = tp.bt[(int64_t)t.i * tp.bt_stride + ut / p.tpb];
      sub = ut % p.tpb;
      my_bad = bid < 0 || (int64_t)bid >= tp.num_blocks;
    } else {
      const TierParams& tp = p.tier[TS == kSecondTier ? 1 : 0];
      bid = tp.bt[(int64_t)t.i * tp.bt_stride + u / p.tpb];
      sub = u % p.tpb;
      my_bad = bid < 0 || (int64_t)bid >= tp.num_blocks;
    }
  }
  w.bad = __ballot(my_bad) != 0;
  w.my_bid = my_bad ? 0 : bid;
  w.my_sub = my_bad ? 0 : sub;
  return w;
}

// Per-wave softmax states (log2-domain max, sum, unnormalised accumulator)
// for the cross-wave merge.
template <int D, int G>
struct WaveStates {
  float acc[kWavesPerTask][G][D];
  float m[kWavesPerTask][G];
  float l[kWavesPerTask][G];
  int bad[kWavesPerTask];
  int last;  // balanced cuts: this task is its row's last to arrive
};

// Folds the TPW = 64 / LPT lane-rows of a wave (each with its own softmax
// state per head: log2-domain max m, sum l, accumulator of its 8 dims) into
// the wave's state and publishes it in `ws` for finish_task.
template <int D, int G>
__device__ __forceinline__ void publish_wave_state(WaveStates<D, G>& ws, int wave, int lane,
                                                   const float* m, const float* l,
                                                   const float (*acc)[8], bool bad) {
  constexpr int LPT = D / 8;
  const int chunk = lane % LPT;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float M = m[g];
    if constexpr (LPT < kWave) M = xor_max<LPT>(M);
    const float Ms = M == neg_inf() ? 0.f : M;
    const float w = fast_exp2(m[g] - Ms);
    float lt = l[g] * w;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = acc[g][e] * w;
    if constexpr (LPT < kWave) {
      lt = xor_sum<LPT>(lt);
#pragma unroll
      for (int e = 0; e < 8; ++e) o[e] = xor_sum<LPT>(o[e]);
    }
    if (lane < LPT) {
      float4* dst = reinterpret_cast<float4*>(&ws.acc[wave][g][chunk * 8]);
      dst[0] = make_float4(o[0], o[1], o[2], o[3]);
      dst[1] = make_float4(o[4], o[5], o[6], o[7]);
    }
    if (lane == 0) {
      ws.m[wave][g] = M;
      ws.l[wave][g] = lt;
    }
  }
  if (lane == 0) ws.bad[wave] = bad ? 1 : 0;
}

// Split partials of balanced cuts are written and read at agent scope (sc1:
// past the XCD's own L2), as a row's tasks run on several XCDs.
constexpr int kAgentScope = 16;
typedef unsigned int part_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int part_u32x2 __attribute__((ext_vector_type(2)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t part_rsrc(const float* base, int64_t elems) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)(elems * 4),
                                           0x00020000);
}

__device__ __forceinline__ void normalise(float (&o)[8], float l) {
  const float inv = 1.f / l;
#pragma unroll
  for (int e = 0; e < 8; ++e) o[e] *= inv;
}

// Writes a split task's partial of 8 dims of query head h from its sums of
// p V, running max M (log2 domain) and sum of p. Cut by table width: the
// normalised output and, with d0 == 0, the LSE. Balanced cuts keep the sums
// and (M, l) as they are: a weight exp2(M - max) made from an LSE, a number
// of about 10 in fp32, has its rounding in every bit of the merged row.
// Distance from 64 bits (fp32 out; kept as LSEs, then as sums): 12 x
// U[64, 1500], 32/8, fp32 KV 2.0 -> 1.7e-7 (LSE 4.8 -> 3.9e-8); 4 x
// U[3000, 9000], 32/32, fp16 3.1 -> 2.2e-7. A part whose weight underflows
// still shows a NaN or infinity in its V, as in a row of one task.
template <bool BAL = true>
__device__ __forceinline__ void store_partial(const TiledParams& p, const Task& t, int h, int d0,
                                              float (&o)[8], float M, float l) {
  if (BAL && p.bal_parts > 0) {
    // (resources of the whole task: one of each lane's head would not be
    // uniform, and cost a loop over the heads per store)
    const int64_t pidx = (int64_t)(t.slot0 + t.split) * p.H + t.h0;
    const __amdgpu_buffer_rsrc_t ro = part_rsrc(p.part_o + pidx * p.D, (int64_t)t.gcount * p.D);
    const int off = (h - t.h0) * p.D + d0;
#pragma unroll
    for (int e = 0; e < 8; e += 4) {
      const part_u32x4 u = {__float_as_uint(o[e]), __float_as_uint(o[e + 1]),
                            __float_as_uint(o[e + 2]), __float_as_uint(o[e + 3])};
      __builtin_amdgcn_raw_buffer_store_b128(u, ro, (off + e) * 4, 0, kAgentScope);
    }
    if (d0 == 0) {
      const part_u32x2 u = {__float_as_uint(M), __float_as_uint(l)};
      __builtin_amdgcn_raw_buffer_store_b64(u, part_rsrc(p.part_lse + pidx * 2, 2 * t.gcount),
                                            (h - t.h0) * 8, 0, kAgentScope);
    }
  } else {
    const int64_t pidx = ((int64_t)t.i * p.H + h) * p.S + t.split;
    normalise(o, l);
    store8<F32>(p.part_o, pidx * p.D + d0, true, o);
    if (d0 == 0) p.part_lse[pidx] = (M + fast_log2(l)) * kLn2;
  }
}

// Wave 0, after the workgroup barrier: merges the waves' states with the
// log-sum-exp rule and writes the final result, or this split's partial for
// the combine pass.
template <typename T, int D, int G>
__device__ __forceinline__ void finish_task(const TiledParams& p, const Task& t,
                                            const WaveStates<D, G>& ws, int lane) {
  constexpr int LPT = D / 8;
  const int chunk = lane % LPT;
  bool bad = false;
#pragma unroll
  for (int w = 0; w < kWavesPerTask; ++w) bad |= ws.bad[w] != 0;
  const bool write_final = t.nsplit == 1;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float M = ws.m[0][g];
#pragma unroll
    for (int w = 1; w < kWavesPerTask; ++w) M = fmaxf(M, ws.m[w][g]);
    const float Ms = M == neg_inf() ? 0.f : M;
    float lt = 0.f;
    float o[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = 0.f;
    // every lane reads its chunk's slice of every wave's state at once (lanes
    // past LPT repeat a chunk's reads and store nothing): the LDS reads issue
    // together instead of one wave's after another's
    float4 sa[kWavesPerTask], sb[kWavesPerTask];
#pragma unroll
    for (int w = 0; w < kWavesPerTask; ++w) {
      const float4* src = reinterpret_cast<const float4*>(&ws.acc[w][g][chunk * 8]);
      sa[w] = src[0];
      sb[w] = src[1];
    }
#pragma unroll
    for (int w = 0; w < kWavesPerTask; ++w) {
      const float sc = fast_exp2(ws.m[w][g] - Ms);  // 0 for a wave without blocks
      lt += sc * ws.l[w][g];
      o[0] += sc * sa[w].x;
      o[1] += sc * sa[w].y;
      o[2] += sc * sa[w].z;
      o[3] += sc * sa[w].w;
      o[4] += sc * sb[w].x;
      o[5] += sc * sb[w].y;
      o[6] += sc * sb[w].z;
      o[7] += sc * sb[w].w;
    }
    if (bad) lt = qnan();  // and with it the row's output and LSE
    const int h = t.h0 + g;
    if (g < t.gcount && lane < LPT && chunk * 8 < p.D) {
      if (write_final) {
        normalise(o, lt);
        store8<T>(p.out, (int64_t)t.i * p.out_ss + (int64_t)h * p.out_sh + chunk * 8,
                  p.out_f32, o);
        if (lane == 0) p.lse[(int64_t)h * p.lse_sh + t.i] = (M + fast_log2(lt)) * kLn2;
      } else {
        store_partial(p, t, h, chunk * 8, o, M, lt);
      }
    }
  }
}

// Arrivals of a row's parts: one thread of a task calls start_count() before
// the part's stores and, once they are waited for, count_arrival(), which is
// true for the row's last. Rows are counted by their place in the launch's
// list: an order with entries outside [0, n) may list a row twice, and each
// listing is cut, counted and merged by itself.
//
// A counter holds the number of a launch above its arrivals (kArrivalBits).
// Numbers rise from launch to launch, so start_count()'s maximum starts the
// count anew whatever an earlier launch left (one that overlapped another on
// the same counters leaves a count behind), and changes nothing otherwise; the
// last arrival takes its count back out, for replays of a graph, which keep
// the number they were captured with. The tasks of a row finish together, and
// atomics on one line go one by one, so the maximum goes out beside the
// part's stores (a host worker wave's before its blocks are read), and counters of a launch with few of them lie in lines of
// their own. A row of 900 tokens, 32/8, eight counters of 32 parts each (HIP
// graph replay): both atomics at the end 8.29 us with the counters side by
// side and 7.58 with them 256 bytes apart; the maximum beside the stores takes
// another 0.2 off, and 14.7 -> 13.5 off 3 rows of 2,678 to 10,717 tokens, 8/1
// (85 parts each).
constexpr int kArrivalBits = 24;  // parts of a row: below 2^22 (cut_balanced)

__device__ __forceinline__ uint64_t* arrivals(const TiledParams& p, const Task& t) {
  return p.counters + (t.pos * p.KVH * p.passes + t.kp) * p.counter_stride;
}

__device__ __forceinline__ void start_count(const TiledParams& p, const Task& t) {
  __hip_atomic_fetch_max(arrivals(p, t), p.launch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

__device__ __forceinline__ bool count_arrival(const TiledParams& p, const Task& t) {
  constexpr uint64_t kCount = (1ull << kArrivalBits) - 1;
  uint64_t* c = arrivals(p, t);
  const uint64_t before =
      __hip_atomic_fetch_add(c, 1ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool done = (uint32_t)(before & kCount) == (uint32_t)t.nsplit - 1;
  if (done) __hip_atomic_store(c, before & ~kCount, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return done;
}

// This wave's partial stores are done (vmcnt(0)). The fences emit nothing:
// they keep the compiler from moving the stores, or the arrival, across the
// wait.
__device__ __forceinline__ void partial_written() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_s_waitcnt(0x0F70);
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
}

// Whether the tasks of this row still to come leave the merge to this one: a
// balanced launch has no combine pass; the last of a row's parts to arrive
// merges them. Called by the whole workgroup once its partial is written;
// true on every thread of the last one. The partial's stores go through to memory (sc1) and
// are waited for before the arrival is counted, and the last task reads the
// parts with sc1 loads, so no cache is written back or invalidated (an
// agent-scope release / acquire pair does both, and held launches up to 2x).
__device__ __forceinline__ bool last_to_arrive(const TiledParams& p, const Task& t, int* last) {
  partial_written();
  __syncthreads();
  if (threadIdx.x == 0) *last = count_arrival(p, t) ? 1 : 0;
  __syncthreads();
  const bool merge = __builtin_amdgcn_readfirstlane(*last) != 0;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // no part is read before
  return merge;
}

// Merges the row's parts and writes its result (thread `tid` of `threads`: the
// workgroup, or host worker wave, of the row's last task): a thread takes 4
// dims of a head and folds the parts in order, kPartsInFlight of them read
// together, as each round of reads is a trip past the L2. The order is fixed,
// whichever task arrives last.
constexpr int kPartsInFlight = 8;

template <typename T, int D>
__device__ __forceinline__ void merge_parts(const TiledParams& p, const Task& t, int tid,
                                            int threads) {
  constexpr int LPT = D / 4;  // threads per head
  const int64_t first = (int64_t)t.slot0 * p.H + t.h0;
  const int64_t heads = (int64_t)(t.nsplit - 1) * p.H + t.gcount;
  const __amdgpu_buffer_rsrc_t ro = part_rsrc(p.part_o + first * p.D, heads * p.D);
  const __amdgpu_buffer_rsrc_t rl = part_rsrc(p.part_lse + first * 2, heads * 2);
  for (int it = tid; it < t.gcount * LPT; it += threads) {
    const int g = it / LPT;
    const int d0 = (it % LPT) * 4;
    if (d0 >= p.D) continue;
    float M = neg_inf(), l = 0.f, acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < t.nsplit; k0 += kPartsInFlight) {
      part_u32x2 ml[kPartsInFlight];
      part_u32x4 x[kPartsInFlight];
#pragma unroll
      for (int u = 0; u < kPartsInFlight; ++u) {
        // a part past the last reads the last one again, to no effect
        const uint32_t pi = (uint32_t)(min(k0 + u, t.nsplit - 1) * p.H + g);
        ml[u] = __builtin_amdgcn_raw_buffer_load_b64(rl, pi * 8, 0, kAgentScope);
        x[u] = __builtin_amdgcn_raw_buffer_load_b128(
            ro, (pi * (uint32_t)p.D + (uint32_t)d0) * 4, 0, kAgentScope);
      }
      float mn = M;
#pragma unroll
      for (int u = 0; u < kPartsInFlight; ++u) mn = fmaxf(mn, __uint_as_float(ml[u][0]));
      const float ms = mn == neg_inf() ? 0.f : mn;
      const float alpha = fast_exp2(M - ms);
      l *= alpha;
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[e] *= alpha;
#pragma unroll
      for (int u = 0; u < kPartsInFlight; ++u) {
        const bool on = k0 + u < t.nsplit;
        const float w = fast_exp2(__uint_as_float(ml[u][0]) - ms);
        l = __builtin_fmaf(w, on ? __uint_as_float(ml[u][1]) : 0.f, l);
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[e] = __builtin_fmaf(w, on ? __uint_as_float(x[u][e]) : 0.f, acc[e]);
      }
      M = mn;
    }
    const float inv = 1.f / l;
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[e] *= inv;
    const int h = t.h0 + g;
    store4<T>(p.out, (int64_t)t.i * p.out_ss + (int64_t)h * p.out_sh + d0, p.out_f32, acc);
    // (M, about 10, is rounded once: with the product)
    if (d0 == 0)
      p.lse[(int64_t)h * p.lse_sh + t.i] = __builtin_fmaf(M, kLn2, fast_log2(l) * kLn2);
  }
}

// The end of a task of the kernels whose waves publish WaveStates: the waves
// merge, and in a balanced launch a row's last task merges its parts.
template <typename T, int D, int G>
__device__ __forceinline__ void end_task(const TiledParams& p, const Task& t, WaveStates<D, G>& ws,
                                         int wave, int lane) {
  const bool part = p.bal_parts > 0 && t.nsplit > 1;
  if (part && threadIdx.x == 0) start_count(p, t);
  __syncthreads();
  if (wave == 0) finish_task<T, D, G>(p, t, ws, lane);
  if (!part) return;
  if (last_to_arrive(p, t, &ws.last))
    merge_parts<T, D>(p, t, threadIdx.x, kWave * kWavesPerTask);
}

// After a host worker wave's part is written: merges the row if it was the
// row's last.
template <typename T, int D>
__device__ __forceinline__ void end_solo_part(const TiledParams& p, const Task& t, int lane) {
  if (t.nsplit == 1) return;
  partial_written();
  int last = 0;
  if (lane == 0) last = count_arrival(p, t) ? 1 : 0;
  const bool merge = __builtin_amdgcn_readfirstlane(last) != 0;
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // no part is read before
  if (merge) merge_parts<T, D>(p, t, lane, kWave);
}

// Query head of the task's head slot g: slots past the task's heads repeat
// its last head (their results are never written).
__device__ __forceinline__ int task_head(const Task& t, int g) {
  return t.h0 + min(g, t.gcount - 1);
}

// The cache run of a wave's block k: K and V buffer resources over its
// (block, kv head) run in the tier it lies in, and that tier (wave-uniform;
// the kernel picks its per-lane offsets for the tier).
struct BlockSrc {
  __amdgpu_buffer_rsrc_t k, v;
  const char* kp;  // the K run's first byte (global loads of a kv_adj tier)
  bool t1;
};

// A tier-1 block's resources end with its last valid token (a tier's last
// block may be partial): rows past it read as zero and cost no traffic, which
// counts over the link, where a row's newest block is often all it has (33
// rows with one host block each, 2.2 -> 1.2 MB over the link). In HBM the
// extra scalar work per block costs more than the bytes (full batch of 256
// grouped-query rows: 387 -> 401 us), so tier 0 keeps whole blocks.
template <int TS>
__device__ __forceinline__ BlockSrc block_src(const TiledParams& p, const WaveBlocks& wb,
                                              const Task& t, int k) {
  constexpr bool TWO = TS != kFirstTier;
  const bool t1 = TS == kSecondTier || (TS == kBothTiers && k >= wb.k1);
  const int bid = __builtin_amdgcn_readlane(wb.my_bid, k);
  const int sub = __builtin_amdgcn_readlane(wb.my_sub, k);
  const TierParams& a = p.tier[0];
  const TierParams& b = p.tier[TWO ? 1 : 0];
  const int64_t base = (int64_t)bid * (t1 ? b.sb : a.sb) + (int64_t)t.kh * (t1 ? b.sh : a.sh) +
                       (int64_t)sub * kTileTokens * (t1 ? b.st : a.st);
  uint32_t cut = 0;  // bytes of the block's rows past its tokens
  if (t1)
    cut = (uint32_t)(kTileTokens - block_tokens<TS>(t, wb.first + wb.stride * k)) *
          (uint32_t)b.st * 2;
  BlockSrc s;
  s.k = make_rsrc((t1 ? b.k : a.k) + base, (t1 ? b.k_run_bytes : a.k_run_bytes) - cut);
  s.v = make_rsrc((t1 ? b.v : a.v) + base, (t1 ? b.run_bytes : a.run_bytes) - cut);
  s.kp = reinterpret_cast<const char*>((t1 ? b.k : a.k) + base);
  s.t1 = t1;
  return s;
}

}  // namespace fd
