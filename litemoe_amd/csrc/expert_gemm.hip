// Grouped expert GEMMs for prefill-sized route counts, on MFMA with LDS tiles:
//
//   gate_up: act[r, j] = bf16(silu(bf16(x_t . W13[e, j])) * bf16(x_t . W13[e, I + j]))
//   down:    y[r, n]   = bf16(act[r] . W2[e, n])
//
// over the route blocks of lm_moe_align (routes sorted by expert; a block is
// at most kTM routes of one expert, found on the device from the offsets).
// y is in route order r = t*topk + branch, as on the decode path; act is in
// route order for the public gate_up / down entry points and in sorted order
// (row = position in the expert-sorted route list) between the two GEMMs of
// one fused call, so that down reads each route block's act rows as one
// contiguous run instead of gathering 128-byte pieces of rows spread over
// the whole buffer.
//
// Workgroup = (output column tile, route block). It computes a kTM x kTN
// fp32 tile (see the tiles below): for gate_up the B tile is kTN/2 gate rows
// and the kTN/2 up rows of the same j, so silu(g)*u is formed in registers.
// The waves sit in kWM x kWN, each (kTM/kWM) x (kTN/kWN) as 16 x 16 tiles of
// v_mfma_f32_16x16x32_bf16.
//
// K runs in steps of 64. The next step's A rows (gathered through the route
// list: each lane's copy has its own address) and B rows are copied from
// global memory straight into another of the LDS stages
// (global_load_lds_dwordx4, lds_copy16) while the MFMAs run on the current
// one. An LDS row is 64 bf16 = 8 chunks of 16 bytes; chunk c of tile row r sits
// at position c ^ (r & 7), so the 16 rows read by one MFMA fragment load spread
// over the banks, and each wave instruction fills 1 KB contiguously.
//
// Reference: the expert math of litemoe/ops.py:43-47 (reference_experts) and
// vLLM fused_experts at litemoe/ep.py:40-41.
#include <algorithm>
#include <type_traits>

#include "internal.h"

namespace lm {
namespace {

constexpr int kBK = 64;   // K per stage
constexpr int kXcds = 8;  // MI355X: 8 XCDs, each with its own L2
constexpr int kRowBytes = kBK * 2;  // 128
constexpr int kLdsBytes = 160 * 1024;  // per CU

template <int TM, int TN, int WMv, int WNv, int StagesV>
struct TileCfg {
  static constexpr int M = TM, N = TN, WM = WMv, WN = WNv, Stages = StagesV;
};
// Workgroup tiles, chosen per call by r, the mean routes per expert (what the
// host knows). An expert's last block is partly padding, so the tile's height
// follows r; every tile sums K in the same order, so the choice changes no
// bits. Measured alone on one box, us per launch, gate_up / down, at 40
// experts, hidden 1536, uniform routes ("before": one 128 x 128 tile on 4
// waves with register staging below r = 1024, the grid's blocks dealt to the
// XCDs, 256 x 256 above):
//      r    before        64 rows     192 rows    256 x 256
//     30    37.7 / 23.5   29.0 / 12.7  37.9 / 14.6   39.0 / 19.0
//    140    58.1 / 30.2   44.3 / 23.2  43.5 / 18.2   43.7 / 20.8
//    400    84.1 / 46.8   80.6 / 44.4  70.3 / 44.9   83.0 / 40.7
//   1200   161.4 / 96.0      -        156.1 / 99.9  169.3 / 96.1
// - Low: the weights are read once per block and bound the launch; gate_up
//   (24 K steps) takes three stages so that two steps' loads are in flight,
//   down (8 steps) two.
// - Mid: gate_up 192 x 128 on 8 waves of 48 x 64, 80 KB: two workgroups share
//   a CU and one computes while the other waits at its barrier. down (one
//   third of the K steps, three times the output) 192 x 256, whose activation
//   rows are read by half as many column tiles.
// - High: 256 x 256 on 8 waves, a wave's 12 fragment reads feed 32 MFMAs:
//   down 128 x 64 waves (665 -> 655 us at r = 9400, skewed routes, against
//   64 x 128), gate_up 64 x 128 (978 against 985 us).
using GateLow = TileCfg<64, 256, 2, 4, 3>;
using GateMid = TileCfg<192, 128, 4, 2, 2>;
using DownLow = TileCfg<64, 128, 2, 2, 2>;
using DownMid = TileCfg<192, 256, 4, 2, 2>;
using DownMidNarrow = TileCfg<192, 128, 4, 2, 2>;  // hidden not a multiple of 256
using GateHigh = TileCfg<256, 256, 4, 2, 2>;
using DownHigh = TileCfg<256, 256, 2, 4, 2>;
constexpr int64_t kLowBelow = 96, kHighFrom = 1024, kGateHighAlways = 2048;

// The route block of workgroup `lin` (blocks of at most bm routes of one
// expert, from the offsets lm_moe_align writes: exclusive prefix of the
// per-expert counts), numbered so that each XCD takes an eighth of the blocks
// there are: workgroups are dealt to the 8 XCDs round-robin in launch order,
// so workgroup lin is number lin / 8 of XCD lin % 8, and takes block (that
// XCD's first) + number / cols. The grid is sized for the most blocks the
// routes can make; dealing out the grid's blocks instead of the existing ones
// would leave the last XCDs the empty ones (gate/up at 300 tokens over 40
// experts: 55 of 80 blocks exist).
// Lane l takes expert e0 + l's block count; an inclusive prefix sum over the
// lanes gives each expert's first block, and the expert holding the block is
// the one lane whose range contains it. (A scalar walk over the experts waits
// on one load per expert.)
__device__ __forceinline__ bool block_of(const int32_t *__restrict__ offsets, int experts, int bm,
                                         int lin, int cols, int &e_out, int &r0, int &r1) {
  const int lane = threadIdx.x % kWave;
  auto counts = [&](int e0, int &o0, int &o1, int &incl) {  // returns the lane's own count
    const int e = e0 + lane;
    o0 = e < experts ? offsets[e] : 0;
    o1 = e < experts ? offsets[e + 1] : 0;
    const int nb = (o1 - o0 + bm - 1) / bm;
    incl = nb;
#pragma unroll
    for (int d = 1; d < kWave; d *= 2) {
      const int up = __shfl_up(incl, d, kWave);
      if (lane >= d) incl += up;
    }
    return nb;
  };
  int o0, o1, incl;
  int nb = counts(0, o0, o1, incl);
  int total = __shfl(incl, kWave - 1, kWave);
  for (int e0 = kWave; e0 < experts; e0 += kWave) {
    int p0, p1, more;
    counts(e0, p0, p1, more);
    total += __shfl(more, kWave - 1, kWave);
  }
  const int per_xcd = (total + kXcds - 1) / kXcds, j = lin / kXcds / cols;
  const int b = (lin % kXcds) * per_xcd + j;
  if (j >= per_xcd || b >= total) return false;
  int before = 0;  // blocks of the experts below e0
  for (int e0 = 0;;) {
    const int first = before + incl - nb;
    const uint64_t hit = __ballot(b >= first && b < first + nb);
    if (hit) {
      const int l = __ffsll((unsigned long long)hit) - 1;
      e_out = e0 + l;
      r0 = __shfl(o0, l, kWave) + (b - __shfl(first, l, kWave)) * bm;
      r1 = min(__shfl(o1, l, kWave), r0 + bm);
      return true;
    }
    before += __shfl(incl, kWave - 1, kWave);
    e0 += kWave;
    if (e0 >= experts) return false;
    nb = counts(e0, o0, o1, incl);
  }
}

// Byte offset in an operand tile of (row, 16-byte chunk).
__device__ __forceinline__ int frag_offset(int row, int chunk) {
  return row * kRowBytes + ((chunk ^ (row & 7)) << 4);
}

// kGateUp: B rows [0, kTN/2) are W13[e, j0 + r], [kTN/2, kTN) are
// W13[e, I + j0 + r - kTN/2], output act; otherwise B rows are W2[e, n0 + r],
// output y. Waves sit in kWM x kWN; wave (wr, wc) owns rows wr*kTM/kWM .. and,
// for gate_up, the gate and up rows of the same kTN/(2*kWN) columns j.
// kPacked: weights in the fragment layout of lm_expert_pack (a load
// instruction then reads eight whole 128-byte runs: the 8 rows of one
// (k-step, k-group) are adjacent there).
// kSortedAct: act row of sorted position p is p (gate_up writes, down reads).
template <bool kGateUp, int kTM, int kTN, int kWM, int kWN, int kStages, bool kPacked,
          bool kSortedAct>
__global__ void __launch_bounds__(64 * kWM * kWN)
expert_gemm_kernel(const bf16 *__restrict__ a_src, const bf16 *__restrict__ w,
                   const int32_t *__restrict__ offsets, const int32_t *__restrict__ sorted,
                   int topk, int K, int out_cols, int inter, int experts,
                   bf16 *__restrict__ out) {
  constexpr int kWaves = kWM * kWN, kThreadsT = 64 * kWaves;
  constexpr int kWaveRows = kTM / kWM, kWaveCols = kTN / kWN;
  constexpr int kRB = kWaveRows / 16, kCB = kWaveCols / 16;  // 16-row / 16-column blocks per wave
  constexpr int kLA = kTM / (8 * kWaves), kLB = kTN / (8 * kWaves);  // 16-byte copies per lane
  static_assert(kLA * 8 * kWaves == kTM && kLB * 8 * kWaves == kTN, "tile rows per copy round");
  static_assert(!kGateUp || kCB % 2 == 0, "gate/up waves hold gate and up blocks in pairs");
  constexpr int kABytes = kTM * kRowBytes, kStageBytes = (kTM + kTN) * kRowBytes;
  // two stages are two arrays, three one array
  __shared__ __align__(16) char smem[kStages == 2 ? kStageBytes : kStages * kStageBytes];
  __shared__ __align__(16) char smem1[kStages == 2 ? kStageBytes : 16];
  constexpr int kOutCols = kGateUp ? kTN / 2 : kTN, kOB = kOutCols * 2;  // output row bytes
  constexpr int kHalfRows = (kStages == 2 ? 1 : kStages) * kStageBytes / kOB;  // staged output rows in smem
  static_assert(kTM * kOB <= kStages * kStageBytes, "output tile fits the LDS stages");
  // The output rows' routes (all forms but gate_up on sorted act), for the
  // epilogue only: in the stages behind the staged output tile where there is
  // room, since the 192 x 128 tile's two workgroups per CU need all 160 KB for
  // their stages (1200 routes per expert, us: gate_up on route-order act at
  // hidden 1536, 40 experts, 193 -> 144, down at hidden 384, 32 experts, 29.5
  // -> 23.6).
  constexpr bool kRouteList = !(kGateUp && kSortedAct);
  constexpr int kTileEnd = kTM * kOB, kListBytes = kTM * 4, kSmem1 = kStages == 2 ? kStageBytes : 0;
  constexpr bool kBehind0 = kTileEnd + kListBytes <= (int)sizeof(smem);
  constexpr int kUsed1 = kTM > kHalfRows ? (kTM - kHalfRows) * kOB : 0;
  constexpr bool kBehind1 = !kBehind0 && kUsed1 + kListBytes <= kSmem1;
  constexpr bool kOwnList = kRouteList && !kBehind0 && !kBehind1;
  static_assert(!kOwnList || 2 * kStages * kStageBytes > kLdsBytes, "the list takes the second workgroup's room");
  __shared__ int list_own[kOwnList ? kTM : 1];
  int *const route_of = kBehind0   ? reinterpret_cast<int *>(smem + kTileEnd)
                        : kBehind1 ? reinterpret_cast<int *>(smem1 + kUsed1)
                                   : list_own;
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  // Each XCD takes a contiguous range of route blocks with all their column
  // tiles (block_of): a block's gathered A rows are then fetched into one L2,
  // and an expert's weight rows mostly into one or two.
  const int cols = gridDim.x;
  const int lin = blockIdx.y * cols + blockIdx.x;
  const int tile_x = lin / kXcds % cols;  // gridDim.y is a multiple of kXcds
  int e, r0, r1;
  if (!block_of(offsets, experts, kTM, lin, cols, e, r0, r1)) return;
  const int n = r1 - r0;
  const int c0 = tile_x * (kGateUp ? kTN / 2 : kTN);  // first output column
  // This thread's entry of the route list, requested ahead of the K loop.
  static_assert(kTM <= kThreadsT, "a list entry per thread");
  [[maybe_unused]] int my_route = 0;
  if constexpr (kRouteList) my_route = sorted[r0 + min((int)threadIdx.x, n - 1)];

  // Load instruction i of wave w fills LDS rows 8*(w*L+i) .. +7 of an
  // operand (1 KB, lane l at byte 16*l): row 8*(w*L+i) + l/8, position l%8,
  // holding chunk (l%8) ^ (l/8), which is frag_offset's swizzle.
  const int chunk = (lane & 7) ^ (lane >> 3);
  int oa[kLA], ob[kLB];  // element offsets (< 2^31 at the supported sizes)
#pragma unroll
  for (int i = 0; i < kLA; ++i) {
    const int t = 8 * (wave * kLA + i) + lane / 8;
    if constexpr (!kGateUp && kSortedAct) {
      oa[i] = (r0 + min(t, n - 1)) * K + chunk * 8;
    } else {
      const int route = sorted[r0 + min(t, n - 1)];
      oa[i] = (kGateUp ? route / topk : route) * K + chunk * 8;
    }
  }
#pragma unroll
  for (int i = 0; i < kLB; ++i) {
    const int row = 8 * (wave * kLB + i) + lane / 8;
    const int wrow = kGateUp ? e * 2 * inter + (row < kTN / 2 ? c0 + row : inter + c0 + row - kTN / 2)
                             : e * out_cols + c0 + row;
    ob[i] = (int)wofs<kPacked>(wrow, chunk * 8, K);
  }
  // element advance of one kBK step of B (two 32-wide k-steps when packed)
  constexpr int kBStep = kPacked ? (int)(kBK / 32 * wstep<true>()) : kBK;
  // A step's rows from global memory straight into an LDS stage (byte
  // offsets: the element offsets are below 2^31).
  const uint32_t uw = __builtin_amdgcn_readfirstlane(wave);
  auto issue_a = [&](int kt, const char *stage) {
    const bf16 *ak = a_src + kt * kBK;
    const uint32_t la = lds_address(stage) + uw * kLA * 1024;
#pragma unroll
    for (int i = 0; i < kLA; ++i) lds_copy16(ak, (uint32_t)oa[i] * 2, la + i * 1024);
  };
  auto issue_b = [&](int kt, const char *stage) {
    const bf16 *wk = w + kt * kBStep;
    const uint32_t lb = lds_address(stage) + kABytes + uw * kLB * 1024;
#pragma unroll
    for (int i = 0; i < kLB; ++i) lds_copy16(wk, (uint32_t)ob[i] * 2, lb + i * 1024);
  };

  const int wr = wave / kWN, wc = wave % kWN;
  const int fr = lane % 16, fk = lane / 16;
  constexpr int kGateCols = kWaveCols / 2;  // gate/up: gate (and up) columns of a wave
  int brow[kCB];
#pragma unroll
  for (int cb = 0; cb < kCB; ++cb)
    brow[cb] = kGateUp ? (cb < kCB / 2 ? wc * kGateCols + cb * 16
                                       : kTN / 2 + wc * kGateCols + (cb - kCB / 2) * 16)
                       : wc * kWaveCols + cb * 16;
  f32x4 acc[kRB][kCB];
#pragma unroll
  for (int i = 0; i < kRB; ++i)
#pragma unroll
    for (int jj = 0; jj < kCB; ++jj) acc[i][jj] = f32x4{0.f, 0.f, 0.f, 0.f};

  // One 32-wide half of a k step.
  auto compute_kk = [&](const char *as, int kk) {
    const char *bs = as + kABytes;
    {
      // B fragments stay in registers for the whole k step; A fragments are
      // read one row block at a time.
      u32x4 bfr[kCB];
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb)
        bfr[cb] = *reinterpret_cast<const u32x4 *>(bs + frag_offset(brow[cb] + fr, kk * 4 + fk));
#pragma unroll
      for (int rb = 0; rb < kRB; ++rb) {
        const u32x4 af =
            *reinterpret_cast<const u32x4 *>(as + frag_offset(wr * kWaveRows + rb * 16 + fr, kk * 4 + fk));
        // weights as the first operand: the tile is computed transposed
#pragma unroll
        for (int cb = 0; cb < kCB; ++cb) acc[rb][cb] = mfma16x16x32(bfr[cb], af, acc[rb][cb]);
      }
    }
  };
  auto compute = [&](const char *as) {
#pragma unroll
    for (int kk = 0; kk < kBK / 32; ++kk) compute_kk(as, kk);
  };

  const int nk = K / kBK;
  if constexpr (kStages == 2) {
    // Before a stage is read: this wave's copies have landed (vmcnt) and the
    // barrier has seen every wave's, and every wave has left the step that
    // last read the stage the next copy goes into.
    // The next step's copies go out in two groups, one before each 32-wide
    // half of the current step's MFMAs, instead of all eight before the
    // first: gate/up issues its weight rows first, down its activation rows
    // (the cfg 4 prefill 99.0-99.6 -> 98.8-98.9 ms, the MoE 1.95-1.97 ->
    // 1.945-1.949 ms per layer with uniform routes; A/B on one box, three
    // runs each; the other orders and an even split of both within 1%).
    static_assert(kBK / 32 == 2, "two halves per k step");
    auto issue_first = [&](int kt, const char *stage) {
      if constexpr (kGateUp) issue_b(kt, stage); else issue_a(kt, stage);
    };
    auto issue_second = [&](int kt, const char *stage) {
      if constexpr (kGateUp) issue_a(kt, stage); else issue_b(kt, stage);
    };
    issue_a(0, smem);
    issue_b(0, smem);
    for (int kt = 0; kt < nk; kt += 2) {
      lds_copy_wait();
      __syncthreads();
      if (kt + 1 < nk) issue_first(kt + 1, smem1);
      __builtin_amdgcn_sched_barrier(0);
      compute_kk(smem, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (kt + 1 < nk) issue_second(kt + 1, smem1);
      __builtin_amdgcn_sched_barrier(0);
      compute_kk(smem, 1);
      if (kt + 1 < nk) {
        lds_copy_wait();
        __syncthreads();
        if (kt + 2 < nk) issue_first(kt + 2, smem);
        __builtin_amdgcn_sched_barrier(0);
        compute_kk(smem1, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 2 < nk) issue_second(kt + 2, smem);
        __builtin_amdgcn_sched_barrier(0);
        compute_kk(smem1, 1);
      }
    }
  } else {
    // A ring: the copies of kStages - 1 steps are in flight; a step waits for
    // its own only (they complete in issue order), and one barrier tells that
    // every wave's copies have landed and that every wave has left the step
    // whose slot the next copy goes into.
    static_assert(kStages == 3, "the wait below leaves one later step in flight");
    constexpr int kL = kLA + kLB;  // copies of one step per wave
    auto issue = [&](int kt, const char *stage) {
      issue_a(kt, stage);
      issue_b(kt, stage);
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s)
      if (s < nk) issue(s, smem + s * kStageBytes);
    int cur = 0, nxt = (kStages - 1) * kStageBytes;
    for (int kt = 0; kt < nk; ++kt) {
      if (kt + 1 < nk) vm_wait<kL>(); else vm_wait<0>();
      __syncthreads();
      if (kt + kStages - 1 < nk) issue(kt + kStages - 1, smem + nxt);
      __builtin_amdgcn_sched_barrier(0);
      compute(smem + cur);
      cur = cur == (kStages - 1) * kStageBytes ? 0 : cur + kStageBytes;
      nxt = nxt == (kStages - 1) * kStageBytes ? 0 : nxt + kStageBytes;
    }
  }

  // Transposed C fragment: lane holds output row lane%16 of each 16-row block
  // and its output columns 4*(lane/16) .. +3 of each 16-column block, one
  // 8-byte word. Intermediate roundings skip the NaN canonicalization (a NaN
  // stays NaN through silu and the product, and the stored value is
  // canonicalized). The bf16 tile is staged in the (now idle) LDS stages and
  // written out row by row in 16-byte words, so that a store instruction
  // covers whole output rows (512 or 256 bytes each) instead of 32-byte
  // pieces of 16 rows. Staged row r's 16-byte chunk c sits at c ^ (r & kSw):
  // the 16 rows of one fragment store fall on different bank groups.
  constexpr int kChunks = kOB / 16, kSw = (kChunks < 16 ? kChunks : 16) - 1;
  auto staged = [&](int row) -> char * {
    if constexpr (kTM <= kHalfRows) return smem + row * kOB;
    else return row < kHalfRows ? smem + row * kOB : smem1 + (row - kHalfRows) * kOB;
  };
  __syncthreads();  // every wave has finished reading the stages
  if constexpr (kRouteList)
    if (threadIdx.x < kTM) route_of[threadIdx.x] = my_route;
#pragma unroll
  for (int rb = 0; rb < kRB; ++rb) {
    const int row = wr * kWaveRows + rb * 16 + fr;
    char *srow = staged(row);
    if constexpr (kGateUp) {
#pragma unroll
      for (int cb = 0; cb < kCB / 2; ++cb) {
        float h[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          h[i] = round_bf16_nc(silu(round_bf16_nc(acc[rb][cb][i]))) * round_bf16_nc(acc[rb][cb + kCB / 2][i]);
        const int byte = 2 * (wc * kGateCols + cb * 16 + 4 * fk);
        *reinterpret_cast<uint2 *>(srow + (((byte >> 4) ^ (row & kSw)) << 4) + (byte & 8)) =
            make_uint2(pack_bf16(h[0], h[1]), pack_bf16(h[2], h[3]));
      }
    } else {
#pragma unroll
      for (int cb = 0; cb < kCB; ++cb) {
        const int byte = 2 * (wc * kWaveCols + cb * 16 + 4 * fk);
        *reinterpret_cast<uint2 *>(srow + (((byte >> 4) ^ (row & kSw)) << 4) + (byte & 8)) =
            make_uint2(pack_bf16(acc[rb][cb][0], acc[rb][cb][1]), pack_bf16(acc[rb][cb][2], acc[rb][cb][3]));
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < (kTM * kChunks + kThreadsT - 1) / kThreadsT; ++i) {
    const int idx = i * kThreadsT + threadIdx.x;
    const int row = idx / kChunks, c = idx % kChunks;
    if (row >= n) continue;
    const int64_t orow = kGateUp && kSortedAct ? r0 + row : route_of[row];
    // Non-temporal: act and y are written once and read once by the next
    // launch, far more bytes (0.4 and 1.2 GB at cfg 4) than the caches hold
    // (the cfg 4 prefill 102.8 -> 100.1-100.5 ms, A/B on one box, three runs
    // each).
    __builtin_nontemporal_store(*reinterpret_cast<const u32x4 *>(staged(row) + ((c ^ (row & kSw)) << 4)),
                                reinterpret_cast<u32x4 *>(out + orow * out_cols + c0 + c * 8));
  }
}

}  // namespace

bool expert_gemm_ok(int64_t routes, int64_t hidden, int64_t inter, int64_t experts) {
  // 32-bit element offsets: the gathered rows and the weights stay below 2^31.
  const int64_t rows = std::max(routes, experts * std::max(2 * inter, hidden));
  return routes >= kExpertGemmMinRoutes && hidden % kBK == 0 && inter % kBK == 0 &&
         (2 * inter) % GateLow::N == 0 && hidden % DownLow::N == 0 &&
         rows * std::max(hidden, inter) < ((int64_t)1 << 31);
}

namespace {

template <bool kGateUp, class T>
int launch_tile(const bf16 *a, const bf16 *w, const int32_t *offsets,
                const int32_t *sorted, int64_t routes, int64_t topk, int64_t K, int64_t out_cols,
                int64_t inter, int64_t experts, bf16 *out, bool packed, bool sorted_act,
                hipStream_t stream) {
  const int64_t blocks = align_up(cdiv(routes, T::M) + experts, kXcds);
  if (blocks > 65535) return LM_EUNSUPPORTED;
  const int64_t cols = kGateUp ? 2 * inter : out_cols;
  const dim3 grid((unsigned)(cols / T::N), (unsigned)blocks);
  const int threads = 64 * T::WM * T::WN;
  auto go = [&](auto packed_c, auto sorted_c) {
    expert_gemm_kernel<kGateUp, T::M, T::N, T::WM, T::WN, T::Stages, decltype(packed_c)::value,
                       decltype(sorted_c)::value>
        <<<grid, threads, 0, stream>>>(a, w, offsets, sorted, (int)topk, (int)K, (int)out_cols,
                                       (int)inter, (int)experts, out);
  };
  using Y = std::true_type;
  using F = std::false_type;
  if (packed) {
    if (sorted_act) go(Y{}, Y{}); else go(Y{}, F{});
  } else {
    if (sorted_act) go(F{}, Y{}); else go(F{}, F{});
  }
  LM_CHECK_LAUNCH();
  return LM_OK;
}

// GateHigh from 1024 routes per expert where its rounds of 256 tiles cost no
// more than GateMid's of 512: a round of those takes three quarters of the time
// (a last one of 128 tiles half of it), an expert's last block counts half, and
// uneven experts add a thirty-second. From 2048 also where they cost a little
// more, unless GateMid needs one round only. lm_moe_routes, us, GateMid /
// GateHigh, fragment-order weights: hidden 1024, inter 128, 32 experts, 1600
// routes per expert 98 / 87, 1400 76 / 78, 2040 112 / 130; hidden 1536, inter
// 256, 1800 207 / 194, 1400 168 / 175; inter 512, 40 experts, 1600 380 / 370,
// 1200 300 / 295, 2040 454 / 467; hidden 384, inter 256, 4 experts, 2040 27 / 34.
bool gate_high(int64_t routes, int64_t cols, int64_t experts) {
  if (routes < kHighFrom * experts) return false;
  const int64_t mid = (routes / GateMid::M + experts / 2) * (cols / GateMid::N);
  const int64_t high = (routes / GateHigh::M + experts / 2) * (cols / GateHigh::N), last = mid % 512;
  const int64_t mid_time = 3 * (mid / 512) + (last > 128 ? 3 : last > 0 ? 2 : 0);  // quarters of a GateHigh round
  return mid > 512 && (routes >= kGateHighAlways * experts || 4 * cdiv(high + high / 32, 256) <= mid_time);
}

}  // namespace

int launch_expert_gemm_gate_up(const bf16 *x, const bf16 *w13, const int32_t *offsets,
                               const int32_t *sorted, int64_t routes, int64_t topk, int64_t hidden,
                               int64_t inter, int64_t experts, bf16 *act, bool packed,
                               bool sorted_act, hipStream_t stream) {
  auto launch = routes < kLowBelow * experts                    ? launch_tile<true, GateLow>
                : gate_high(routes, 2 * inter, experts)        ? launch_tile<true, GateHigh>
                                                               : launch_tile<true, GateMid>;
  return launch(x, w13, offsets, sorted, routes, topk, hidden, inter, inter, experts, act,
                packed, sorted_act, stream);
}

int launch_expert_gemm_down(const bf16 *act, const bf16 *w2, const int32_t *offsets,
                            const int32_t *sorted, int64_t routes, int64_t hidden, int64_t inter,
                            int64_t experts, bf16 *y, bool packed, bool sorted_act,
                            hipStream_t stream) {
  const bool wide = hidden % DownMid::N == 0;
  auto launch = routes < kLowBelow * experts       ? launch_tile<false, DownLow>
                : !wide                            ? launch_tile<false, DownMidNarrow>
                : routes < kHighFrom * experts ? launch_tile<false, DownMid>
                                                   : launch_tile<false, DownHigh>;
  return launch(act, w2, offsets, sorted, routes, 1, inter, hidden, inter, experts, y, packed,
                sorted_act, stream);
}

}  // namespace lm
