// A 128 x 128 tile of a bfloat16 product on the matrix cores whose rows are found through the caller's functions:
// gathered activation rows (a mixture of experts' tokens, sorted by expert), a weight per group (expert, head),
// outputs scattered or strided.  Used by the grouped products of moe.hip and latent.hip.
//
// Workgroup: 256 threads, four waves as 2 x 2, each 64 activation rows x 64 weight rows: sixteen
// v_mfma_f32_16x16x32_bf16 per 32 k, the weight as the first operand, so that a lane ends up with four
// consecutive weight rows (outputs) of one activation row.  K runs in steps of 64 through two LDS stages (rows
// padded to 144 bytes); the next step's 16-byte chunks are on their way into registers while a step is
// multiplied; one barrier a step.  K must be a multiple of 8 and every row 16-byte aligned; chunks past K and
// rows that do not exist are zeros.  An output element is summed in k order whatever else the tile holds.
#pragma once
#include <type_traits>

#include "common.h"

typedef __bf16 gt_bf16x8 __attribute__((ext_vector_type(8)));
typedef float gt_f32x4 __attribute__((ext_vector_type(4)));

constexpr int GT_TILE = 128;     // rows of activations and of weights per workgroup
constexpr int GT_BK = 64;        // k per step
constexpr int GT_ROW = GT_BK * 2 + 16;   // bytes per LDS row
constexpr int GT_STAGE = 2 * GT_TILE * GT_ROW;
constexpr int GT_LDS_BYTES = 2 * GT_STAGE;

// a_row(r): pointer to activation row r of the tile (r < 128) or nullptr; w_row(r): pointer to weight row r of the
// tile or nullptr.  After the call acc[tn][tm] holds, for this lane, weight rows wn * 64 + tn * 16 + (lane / 16) * 4
// + 0..3 of activation row wm * 64 + tm * 16 + lane % 16.
// Chunks that do not exist are not loaded (measured against reading them at a fixed address and masking: a tile of a
// decode step, which is mostly empty rows, took 40 % longer that way).
template <typename ARow, typename WRow>
__device__ __forceinline__ void group_tile_mma(ARow a_row, WRow w_row, int K, unsigned char* lds,
                                               gt_f32x4 (&acc)[4][4]) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = gt_f32x4{0.f, 0.f, 0.f, 0.f};
  // a thread's eight chunks of a step: four of activations, four of weights; chunk c: row c / 8, k (c % 8) * 8
  const __bf16* src[8];
  unsigned dst[8];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = tid + i * 256, row = c >> 3, kc = c & 7;
    const __bf16* pa = a_row(row);
    const __bf16* pw = w_row(row);
    src[i] = pa ? pa + kc * 8 : nullptr;
    src[4 + i] = pw ? pw + kc * 8 : nullptr;
    dst[i] = (unsigned)(row * GT_ROW + kc * 16);
    dst[4 + i] = (unsigned)((GT_TILE + row) * GT_ROW + kc * 16);
  }
  const int kc_of = tid & 7;      // the same for all of a thread's chunks (256 is a multiple of 8)
  gt_bf16x8 held[8];
  auto fetch = [&](int k0) {
    const bool in = k0 + kc_of * 8 < K;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      gt_bf16x8 zero = {};
      held[i] = (src[i] && in) ? *(const gt_bf16x8*)(src[i] + k0) : zero;
    }
  };
  auto stash = [&](int stage) {
#pragma unroll
    for (int i = 0; i < 8; ++i) *(gt_bf16x8*)(lds + stage * GT_STAGE + dst[i]) = held[i];
  };
  const int steps = (K + GT_BK - 1) / GT_BK;
  fetch(0);
  stash(0);
  __syncthreads();
  for (int s = 0; s < steps; ++s) {
    const int stage = s & 1;
    if (s + 1 < steps) fetch((s + 1) * GT_BK);
    const unsigned char* base = lds + stage * GT_STAGE;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      gt_bf16x8 fa[4], fw[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        fa[t] = *(const gt_bf16x8*)(base + (wm * 64 + t * 16 + lr) * GT_ROW + half * 64 + lg * 16);
        fw[t] = *(const gt_bf16x8*)(base + (GT_TILE + wn * 64 + t * 16 + lr) * GT_ROW + half * 64 + lg * 16);
      }
#pragma unroll
      for (int tn = 0; tn < 4; ++tn)
#pragma unroll
        for (int tm = 0; tm < 4; ++tm)
          acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[tn], fa[tm], acc[tn][tm], 0, 0, 0);
    }
    if (s + 1 < steps) stash(stage ^ 1);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------------------------
// A tile of BM activation rows x BN weight rows whose operands go straight from memory into LDS (buffer loads with the
// lds modifier: no staging registers, no LDS stores), for K in multiples of 64.  WM x WN waves, each BM / WM x BN / WN
// outputs; K in steps of 64 through STAGES stages, the loads of STAGES - 1 steps in flight.  LDS rows are 128 bytes, unpadded (a load
// instruction fills 1 KB: 8 rows, lane L the 16 bytes at 16 L); chunk c of row r sits in slot c ^ (r % 8), so that 16
// rows read the same chunk from different banks.  A wave reads the operands of a half step while it multiplies the other half.
//
// The main loop is that of gemm_tile_direct_kernel (gemm_bf16.hip), whose rows lie a stride apart; a change to one is to be
// weighed for the other.
//
// Every row's place is a byte offset of its own, so rows may be gathered; a row that does not exist has GT_NO_ROW and
// reads zero without touching memory.
constexpr int GT_MIDDLE = 192, GT_WIDE = 256;                    // rows of activations of its larger tiles
constexpr int GT_EITHER = 96;                                    // in a tile's place: 128 or 192, as the groups' sizes say
constexpr unsigned GT_NO_ROW = 0x80000000u;                      // past the end of every view; so are the steps behind it
constexpr long long GT_VIEW_BYTES = 0x7fffffffll;                // views are shorter than GT_NO_ROW

struct GtView {
  __amdgpu_buffer_rsrc_t rsrc;
};
__device__ __forceinline__ GtView gt_view(const void* base, long long bytes) {
  return GtView{__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000)};
}

// Until at most N of the wave's vector memory loads are in flight (they complete in the order of their issue).
template <int N>
__device__ __forceinline__ void gt_wait_loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

template <int BM, int BN, int STAGES>
constexpr int gt_direct_lds() {
  return STAGES * (BM + BN) * GT_BK * 2;
}

// a_off(r), w_off(r): byte offset of row r of the tile; w_second(r): whether weight row r lies in the second view (the
// same for eight rows from a multiple of eight on).  After the call acc[tn][tm] holds, for this lane, weight rows
// wn * (BN / WN) + tn * 16 + (lane / 16) * 4 + 0..3 of activation row wm * (BM / WM) + tm * 16 + lane % 16.
template <int BM, int BN, int WM, int WN, int STAGES, typename AOff, typename WOff, typename WSecond>
__device__ __forceinline__ void group_tile_direct(const GtView a_view, AOff a_off_of, const GtView w_view, const GtView w_view2,
                                                  WOff w_off_of, WSecond w_second, int K, int rows, unsigned char* lds,
                                                  gt_f32x4 (&acc)[BN / WN / 16][BM / WM / 16]) {
  typedef __attribute__((address_space(3))) void* lds_ptr;
  constexpr int WAVES = WM * WN, TM = BM / WM / 16, TN = BN / WN / 16, ROW = GT_BK * 2;
  constexpr int A_LOADS = BM / 8 / WAVES, W_LOADS = BN / 8 / WAVES, LOADS = A_LOADS + W_LOADS, STAGE = (BM + BN) * ROW;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "tile rows must divide among the waves' loads");
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, lr = lane & 15, lg = lane >> 4;
#pragma unroll
  for (int i = 0; i < TN; ++i)
#pragma unroll
    for (int j = 0; j < TM; ++j) acc[i][j] = gt_f32x4{0.f, 0.f, 0.f, 0.f};
  const int ld_row = lane >> 3, ld_chunk = (lane & 7) ^ (lane >> 3);
  unsigned a_off[A_LOADS], w_off[W_LOADS];
  bool second[W_LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i) a_off[i] = a_off_of((wave * A_LOADS + i) * 8 + ld_row) + ld_chunk * 16;
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) {
    w_off[i] = w_off_of((wave * W_LOADS + i) * 8 + ld_row) + ld_chunk * 16;
    second[i] = w_second((wave * W_LOADS + i) * 8);
  }
  auto issue = [&](int stage, int step) {
    unsigned char* to_a = lds + stage * STAGE + wave * A_LOADS * 1024;
    unsigned char* to_w = lds + stage * STAGE + BM * ROW + wave * W_LOADS * 1024;
    const unsigned kb = (unsigned)step * ROW;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_view.rsrc, (lds_ptr)(to_a + i * 1024), 16, (int)(a_off[i] + kb), 0, 0, 0);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(second[i] ? w_view2.rsrc : w_view.rsrc, (lds_ptr)(to_w + i * 1024), 16,
                                               (int)(w_off[i] + kb), 0, 0, 0);
  };
  // chunk lg (first half of a step) or lg + 4 (second half) of row lr of each 16-row tile: bit 6 of the byte offset
  const unsigned frag_a = (unsigned)((wm * TM * 16 + lr) * ROW + ((lg ^ (lr & 7)) * 16));
  const unsigned frag_w = (unsigned)(BM * ROW + (wn * TN * 16 + lr) * ROW + ((lg ^ (lr & 7)) * 16));
  auto read = [&](int stage, int half, gt_bf16x8 (&fa)[TM], gt_bf16x8 (&fw)[TN]) {
    const unsigned char* base = lds + stage * STAGE;
#pragma unroll
    for (int t = 0; t < TN; ++t) fw[t] = *(const gt_bf16x8*)(base + (frag_w ^ (half * 64)) + t * 16 * ROW);
#pragma unroll
    for (int t = 0; t < TM; ++t) fa[t] = *(const gt_bf16x8*)(base + (frag_a ^ (half * 64)) + t * 16 * ROW);
  };
  auto multiply = [&](const gt_bf16x8 (&fa)[TM], const gt_bf16x8 (&fw)[TN]) {
#pragma unroll
    for (int tn = 0; tn < TN; ++tn)
#pragma unroll
      for (int tm = 0; tm < TM; ++tm)
        acc[tn][tm] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[tn], fa[tm], acc[tn][tm], 0, 0, 0);
  };
  const int steps = K / GT_BK;
  gt_bf16x8 fa0[TM], fw0[TN], fa1[TM], fw1[TN];
  issue(0, 0);
#pragma unroll
  for (int i = 1; i < STAGES; ++i)
    if (i < steps) issue(i, i);
  if (steps >= STAGES) gt_wait_loads_but<(STAGES - 1) * LOADS>();
  else gt_wait_loads_but<0>();
  __syncthreads();
  read(0, 0, fa0, fw0);
  // with_loads: step s + STAGES exists; in_flight: how many steps' loads may stay in flight when step s + 1 has to be there
  // Hints for the order within a half step: LDS reads and loads go out one by one between products.
  auto interleave = [](auto lds_reads, auto loads) {
    constexpr int READS = decltype(lds_reads)::value, LOADS_NOW = decltype(loads)::value;
#pragma unroll
    for (int i = 0; i < LOADS_NOW; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one matrix instruction
      __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // one load
    }
#pragma unroll
    for (int i = 0; i < READS; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // one LDS read
    }
    __builtin_amdgcn_sched_group_barrier(0x008, TM * TN, 0);
  };
  auto step = [&](int s, int stage, int next, auto with_loads, auto with_next, auto in_flight) {
    read(stage, 1, fa1, fw1);
    multiply(fa0, fw0);
    interleave(std::integral_constant<int, TM + TN>{}, std::integral_constant<int, 0>{});
    __builtin_amdgcn_sched_barrier(0);             // the products stay on this side: they cover the reads above
    gt_wait_loads_but<decltype(in_flight)::value * LOADS>();
    __syncthreads();                               // step s + 1 is there, and nobody reads this step's stage any more
    if constexpr (decltype(with_loads)::value) issue(stage, s + STAGES);
    if constexpr (decltype(with_next)::value) read(next, 0, fa0, fw0);
    multiply(fa1, fw1);
    interleave(std::integral_constant<int, decltype(with_next)::value ? TM + TN : 0>{},
               std::integral_constant<int, decltype(with_loads)::value ? LOADS : 0>{});
    __builtin_amdgcn_sched_barrier(0);
  };
  typedef std::integral_constant<bool, true> yes;
  typedef std::integral_constant<bool, false> no;
  int s = 0, stage = 0;
  if (wm * (BM / WM) >= rows) {   // none of the wave's rows exist: it only loads for the others, at their pace
    for (; s < steps; ++s, stage = stage + 1 == STAGES ? 0 : stage + 1) {
      if (s + STAGES < steps) gt_wait_loads_but<(STAGES - 2) * LOADS>();
      else gt_wait_loads_but<0>();
      __syncthreads();
      if (s + STAGES < steps) issue(stage, s + STAGES);
    }
    return;
  }
  auto after = [](int at) { return at + 1 == STAGES ? 0 : at + 1; };
  for (; s + STAGES < steps; ++s, stage = after(stage))
    step(s, stage, after(stage), yes{}, yes{}, std::integral_constant<int, STAGES - 2>{});
  for (; s + 1 < steps; ++s, stage = after(stage)) step(s, stage, after(stage), no{}, yes{}, std::integral_constant<int, 0>{});
  step(s, stage, after(stage), no{}, no{}, std::integral_constant<int, 0>{});
}
