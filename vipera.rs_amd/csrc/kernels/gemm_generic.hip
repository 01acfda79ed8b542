// C[M,N] = A[M,K] * W[N,K]^T (+ bias[N]) with every product and sum in 32-bit FMA.
//
// This is the true 32-bit matrix product of the engine (no matrix-core mode of reduced
// precision) and the fallback for mixed storage types.
//
// The reference computes every linear layer as dot(row of W, activation) with the bias added
// after the product (crates/vipera-backend-cpu/src/model.rs:623-629, 1005-1031); weights are
// row-major [out, in] (crates/vipera-backend-cpu/src/quant.rs:1-4).
//
// One order of summation for every output element, whatever kernel computes it, whatever M is and
// whatever else is in the batch, so that a token's result is the same bit for bit however a step is
// cut or batched:
//   * K is cut into ranges of RANGE_K = 256 consecutive k; a range's sum is one chain
//     acc = fma(a[k], w[k], acc) over ascending k, started at +0;
//   * SLAB_RANGES = 4 consecutive ranges form a slab, whose sum is +0 + r0 + r1 + r2 + r3 in that
//     order (ranges past the end of K count as +0, which changes nothing: a chain that starts at +0
//     never ends at -0);
//   * the element is +0 + s0 + s1 + ... over its slabs in ascending order, then + bias, then,
//     when accumulating, old + that.
// Every kernel follows it. gemm_stream_kernel, for up to 8 rows of A in 32-bit operands, is a stream
// of the weights: the product of a few tokens is bound by the bytes of W. Everything else runs on the
// matrix cores, gemm_matrix_kernel for any types and rows, gemm_rows_kernel and gemm_slab_kernel for
// 32-bit operands whose rows start on 16 bytes: v_mfma_f32_32x32x2_f32 computes each of its outputs as
// fma(a[k + 1], w[k + 1], fma(a[k], w[k], c)), rounded after every product, and v_mfma_f32_16x16x4_f32 as
// four of these (compared with fmaf chains bit for bit, values of all magnitudes, denormal, infinite and
// NaN ones included), so a chain of either over ascending k is the range's chain above.

#include "common.h"

namespace {
constexpr int RANGE_K = 256, SLAB_RANGES = 4, SLAB_K = RANGE_K * SLAB_RANGES;
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------------------------
// The tiled product: any operand types, any M. A workgroup owns 64 x 64 outputs, its four waves 32 x 32 each; K in
// steps of 16 through two LDS stages, the next step's loads on their way into registers while a step is multiplied, one
// barrier a step.
//
// What bounds it: the matrix cores' 32-bit rate (64 cycles for 32 x 32 x 2, 157 TFLOP/s over the chip) where the
// tiles fill the chip, the number of workgroups where they do not, and the bytes of W below some 64 rows of A. A wave reads two
// LDS values per 64 cycles of the matrix core, so LDS is idle. Tiles of 128 x 64 and 128 x 128 ask the caches for less but
// hold two and four times the accumulators in three sets (the sums' levels), which leaves fewer waves to hide a step's
// barrier: 2,048 x 37,888 x 3,584 takes 5.23 ms (106 TFLOP/s) here, 5.56 and 6.71 ms with those.
//
// UNITS: 0: a workgroup walks all of K and stores C. 1 or 4: a workgroup (blockIdx.y) owns one range or one slab of
// K and stores its sum to `parts` [unit][M][N]; gemm_parts_finish_kernel adds them, in the order above.
constexpr int TILE = 64, BK = 16, TILE_ROW = BK + 4;   // a row's 16 k and 4 floats of padding: 8 lanes' 16 bytes lie in 32 different banks
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));

// Four consecutive k of a row as floats; VECTOR: K is a multiple of 4 and rows are aligned for one load (a row past
// the end and a k past the end are read at the last place and cleared by the caller where it matters).  whole: no k of
// the step lies past the end, the same for all lanes (a place of its own for every k costs an odd K a tenth of its rate).
template <typename T, bool VECTOR>
__device__ __forceinline__ f32x4_t fetch4(const T* __restrict__ row, int k, int K, bool whole) {
  f32x4_t v;
  if constexpr (VECTOR) {
    const int at = min(k, K - 4);
    if constexpr (sizeof(T) == 4) {
      v = *(const f32x4_t*)(row + at);
    } else {
      const bf16x4_t raw = *(const bf16x4_t*)(row + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = (float)raw[e];
    }
  } else if (whole) {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = to_float<T>(row[k + e]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = to_float<T>(row[min(k + e, K - 1)]);
  }
  return v;
}

template <typename TA, typename TW, typename TC, bool ACCUMULATE, int UNITS, bool VECTOR>
__global__ __launch_bounds__(256) void gemm_matrix_kernel(const TA* __restrict__ A, const TW* __restrict__ W,
                                                          const float* __restrict__ bias, TC* __restrict__ C,
                                                          float* __restrict__ parts, int M, int N, int K, long long lda,
                                                          long long ldc) {
  __shared__ __attribute__((aligned(16))) float As[2][TILE][TILE_ROW];
  __shared__ __attribute__((aligned(16))) float Ws[2][TILE][TILE_ROW];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // the tiles of one run of W's rows follow each other, so that they read it at about the same time
  const int m_tiles = (M + TILE - 1) / TILE;
  const int m0 = blockIdx.x % m_tiles * TILE, n0 = blockIdx.x / m_tiles * TILE;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int k_begin = UNITS ? blockIdx.y * (UNITS * RANGE_K) : 0;
  const int k_end = UNITS ? min(K, k_begin + UNITS * RANGE_K) : K;
  f32x16_t acc, slab, total;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = slab[r] = total[r] = 0.f;

  // A thread stages k 4 q .. 4 q + 3 of row tid / 4 of both operands. Instruction t of a step takes k 2 t from lanes
  // 0 to 31 and k 2 t + 1 from lanes 32 to 63, so a row lies in LDS as its eight even k, then its eight odd ones: a
  // lane's next four operands are one 16-byte read.
  const int lr = tid >> 2, q = tid & 3;
  const TA* a_row = A + (size_t)min(m0 + lr, M - 1) * lda;   // a row past the end is a copy of the last and is not stored
  const TW* w_row = W + (size_t)min(n0 + lr, N - 1) * K;
  f32x4_t ra, rw;
  auto fetch = [&](int k0) {
    const bool whole = k0 + BK <= K;
    ra = fetch4<TA, VECTOR>(a_row, k0 + 4 * q, K, whole);
    rw = fetch4<TW, VECTOR>(w_row, k0 + 4 * q, K, whole);
  };
  auto stage = [&](int buf, int k0) {
    const int left = k_end - (k0 + 4 * q);   // a k past the end adds 0 * 0, which changes no sum
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ra[e] = e < left ? ra[e] : 0.f;
      rw[e] = e < left ? rw[e] : 0.f;
    }
    *(f32x2_t*)(As[buf][lr] + 2 * q) = f32x2_t{ra[0], ra[2]};
    *(f32x2_t*)(As[buf][lr] + 8 + 2 * q) = f32x2_t{ra[1], ra[3]};
    *(f32x2_t*)(Ws[buf][lr] + 2 * q) = f32x2_t{rw[0], rw[2]};
    *(f32x2_t*)(Ws[buf][lr] + 8 + 2 * q) = f32x2_t{rw[1], rw[3]};
  };
  fetch(k_begin);
  stage(0, k_begin);
  __syncthreads();
  int buf = 0;
  const int in_tile = lane & 31, half = (lane >> 5) * 8;
  for (int k0 = k_begin; k0 < k_end;) {
    // a range's steps in a loop of their own, which touches no sum but acc: with the sums added up behind a branch of every
    // step the compiler moves all three sets between the two register files in each of them
    const int range_end = min(k_end, k0 + RANGE_K);
    for (; k0 < range_end; k0 += BK) {
      const bool more = k0 + BK < k_end;
      if (more) fetch(k0 + BK);
#pragma unroll
      for (int t4 = 0; t4 < 2; ++t4) {
        const f32x4_t a = *(const f32x4_t*)&As[buf][wm + in_tile][half + 4 * t4];
        const f32x4_t w = *(const f32x4_t*)&Ws[buf][wn + in_tile][half + 4 * t4];
#pragma unroll
        for (int t = 0; t < 4; ++t) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[t], w[t], acc, 0, 0, 0);
      }
      if (more) stage(buf ^ 1, k0 + BK);
      __syncthreads();
      buf ^= 1;
    }
    if constexpr (UNITS != 1) {
      slab += acc;
      acc = 0.f;
    }
    if constexpr (UNITS == 0) {
      if (k0 % SLAB_K == 0 || k0 >= k_end) {
        total += slab;
        slab = 0.f;
      }
    }
  }
  // a lane holds column lane % 32 of its tile, rows 8 (r / 4) + 4 (lane / 32) + r % 4
  const int n = n0 + wn + in_tile;
  if (n >= N) return;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int m = m0 + wm + 8 * (r / 4) + 4 * (lane >> 5) + r % 4;
    if (m >= M) continue;
    if constexpr (UNITS != 0) {
      parts[((size_t)blockIdx.y * M + m) * N + n] = UNITS == 1 ? acc[r] : slab[r];
    } else {
      float v = total[r];
      if (bias) v += bias[n];
      TC* dst = C + (size_t)m * ldc + n;
      if (ACCUMULATE)
        *dst = from_float<TC>(to_float<TC>(*dst) + v);
      else
        *dst = from_float<TC>(v);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The same product where A, W and C are 32-bit and every row starts on 16 bytes: operands go from memory straight into LDS
// (buffer loads with the lds modifier: no staging registers, no LDS stores) several steps ahead.  Lane group
// g = lane / 16 gives v_mfma_f32_16x16x4_f32 k 4 t + g of its row, which it reads from LDS as such, 4 bytes, two blocks of
// 16 rows with one instruction.  Two kernels:
//   gemm_rows_kernel   a workgroup walks all of K
//   gemm_slab_kernel   a workgroup owns one slab of K, wave w range w of it: the ranges' sums meet in LDS, and where K is one
//                      slab that is the output, with no second launch; else parts and gemm_parts_finish_kernel
// What bounds them: the matrix cores, and the cycles that each LDS read and load between two products takes of its wave.  Lanes
// that read 16 bytes of four k and exchange them took more of those (four exchanges for each such read): 333 x 1,152 x 896 in
// tiles of 48 x 32 15.4 us, 12.4 now; 333 x 9,728 x 896 in tiles of 64 x 128 74.1, 68.0 now.  Below a round of tiles a range's
// chain is what a call waits for: 64 instructions of 32 cycles for each 16 x 16 outputs of a wave.  Tiles of more outputs are
// faster at no size: those of 112 x 128 for 333 x 9,728 x 896 fit one round and take 64.4 us, 62.1 as 48 x 48 over one slab.
// A row past the end is a copy of the last one and is not stored; a k past the end reads as zero (an offset past the view).
constexpr unsigned NO_CHUNK = 0x80000000u;            // past the end of every view, and so are the steps behind it
constexpr long long VIEW_BYTES = 0x7fffffffll;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t row_view(const float* base) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, (int)VIEW_BYTES, 0x00020000);
}

// Until at most N of the wave's vector memory loads are in flight (they complete in the order of their issue).
template <int N>
__device__ __forceinline__ void loads_but() {
  static_assert(N >= 0 && N < 64, "vmcnt has six bits");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0F70);
}

// A block of 16 rows of an operand, 16 k: value t is the lane's k 4 t + lane / 16 of row lane % 16.
typedef f32x4_t Fragment;
__device__ __forceinline__ f32x4_t matrix_step(float w, float a, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(w, a, c, 0, 0, 0); }
// A lane's four sums of 16 x 16 outputs: row lane % 16 of A, columns 4 (lane / 16) and on.

// Four consecutive outputs of a row (as far as they exist): + bias, + old, in that order.  quads: every four lie on 16 bytes
// and exist together.
template <bool ACCUMULATE>
__device__ __forceinline__ void store_outputs(float* __restrict__ C, const float* __restrict__ bias, f32x4_t v, int m, int n, int M,
                                              int N, long long ldc, bool quads) {
  if (m >= M || n >= N) return;
  float* dst = C + (size_t)m * ldc + n;
  if (quads) {
    if (bias) v += *(const f32x4_t*)(bias + n);
    if (ACCUMULATE) v = *(const f32x4_t*)dst + v;
    *(f32x4_t*)dst = v;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (n + e >= N) break;
    float x = v[e];
    if (bias) x += bias[n + e];
    dst[e] = ACCUMULATE ? dst[e] + x : x;
  }
}

// Four outputs of a gated product: up * silu(gate).
__device__ __forceinline__ f32x4_t gated_outputs(f32x4_t gate, f32x4_t up) {
  f32x4_t v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = up[e] * (gate[e] / (1.0f + expf(-gate[e])));
  return v;
}

// Hints for the order of what was written since the last such line: LDS reads and loads go out one by one between the products.
// All of them ahead of the products made every wave wait for the others' at the LDS and address units: 112 TFLOP/s at
// 2,048 x 4,096 x 4,096.
template <int PRODUCTS, int READS, int LOADS>
__device__ __forceinline__ void between_products() {
  constexpr int MOST = READS > LOADS ? READS : LOADS;
  constexpr int EACH = MOST <= PRODUCTS ? 1 : (MOST + PRODUCTS - 1) / PRODUCTS;
#pragma unroll
  for (int i = 0; i < PRODUCTS; ++i) {
    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);     // one matrix instruction
    if (i * EACH < READS) __builtin_amdgcn_sched_group_barrier(0x100, EACH, 0);   // LDS reads
    if (i * EACH < LOADS) __builtin_amdgcn_sched_group_barrier(0x020, EACH, 0);   // loads
  }
  __builtin_amdgcn_sched_barrier(0);
}
// LDS reads of 16 k of TM + TN blocks: two blocks an instruction
template <int TM, int TN> constexpr int READS_OF = 4 * ((TM + 1) / 2 + (TN + 1) / 2);

// A workgroup's outputs over all of K: WM x WN waves, each TM x TN blocks of 16 x 16; steps of 32 k through STAGES stages, the
// loads of STAGES - 1 steps in flight.  LDS rows are 128 bytes, unpadded (a load instruction fills 1 KB: 8 rows, lane L the 16
// bytes at 16 L); chunk c of row r sits in slot c ^ (r / 2 % 8): the 64 values of a block's next four k lie in 64 banks.  A wave
// loads every WAVES-th 8 rows, so that its lanes' chunks are the same in all of them.  It reads the operands of a half step
// while it multiplies the first half of the other.  SLABS: K has several.
// GATED: W is [gate; up], N rows each, and C's N columns up * silu(gate); every second block of 16 rows of a tile is up's of the
// outputs whose gates the block before it has, so that a lane has both sums of an output.
template <int TM, int TN, int WM, int WN, int STAGES, bool SLABS, bool ACCUMULATE, bool GATED = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_rows_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                                 const float* __restrict__ bias, float* __restrict__ C, int M,
                                                                 int N, int K, long long lda, long long ldc, bool quads) {
  typedef __attribute__((address_space(3))) void* lds_at;
  constexpr int WAVES = WM * WN, BM = 16 * TM * WM, BN = 16 * TN * WN, STEP = 32, ROW = STEP * 4;
  constexpr int A_LOADS = BM / 8 / WAVES, W_LOADS = BN / 8 / WAVES, LOADS = A_LOADS + W_LOADS, STAGE = (BM + BN) * ROW;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0 && WAVES % 2 == 0, "tile rows must divide among the waves' loads");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN, lr = lane & 15;
  const int m_tiles = (M + BM - 1) / BM;
  const int m0 = blockIdx.x % m_tiles * BM, n0 = blockIdx.x / m_tiles * (GATED ? BN / 2 : BN);
  static_assert(!GATED || (TN % 2 == 0 && !ACCUMULATE), "blocks of gate and up in pairs");
  const __amdgpu_buffer_rsrc_t a_view = row_view(A + (size_t)m0 * lda), w_view = row_view(W + (size_t)n0 * K);
  const int ld_row = lane >> 3, ld_chunk = (lane & 7) ^ (lane >> 4) ^ (wave & 1) * 4;
  unsigned a_off[A_LOADS], w_off[W_LOADS];
#pragma unroll
  for (int i = 0; i < A_LOADS; ++i)
    a_off[i] = (unsigned)(min(m0 + (i * WAVES + wave) * 8 + ld_row, M - 1) - m0) * (unsigned)(lda * 4) + ld_chunk * 16;
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) {
    const int r = (i * WAVES + wave) * 8 + ld_row;
    if constexpr (GATED)
      w_off[i] = (unsigned)((r & 16 ? N : 0) + min(n0 + (r / 32 * 16 + r % 16), N - 1) - n0) * (unsigned)(K * 4) + ld_chunk * 16;
    else
      w_off[i] = (unsigned)(min(n0 + r, N - 1) - n0) * (unsigned)(K * 4) + ld_chunk * 16;
  }
  auto issue = [&](int stage, int step) {
    unsigned char* to_a = lds + stage * STAGE + wave * 1024;
    unsigned char* to_w = to_a + BM * ROW;
    const unsigned kb = step * STEP + ld_chunk * 4 < K ? (unsigned)step * ROW : NO_CHUNK;
#pragma unroll
    for (int i = 0; i < A_LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(a_view, (lds_at)(to_a + i * WAVES * 1024), 16, (int)(a_off[i] + kb), 0, 0, 0);
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(w_view, (lds_at)(to_w + i * WAVES * 1024), 16, (int)(w_off[i] + kb), 0, 0, 0);
  };
  unsigned at[4];                                      // the lane's four k of a block's first half step; bit 6 of the place: the second half
#pragma unroll
  for (int t = 0; t < 4; ++t) at[t] = (unsigned)(lr * ROW + ((t ^ (lr >> 1)) * 16) + (lane >> 4) * 4);
  const unsigned at_a = wm * TM * 16 * ROW, at_w = (BM + wn * TN * 16) * ROW;
  auto read = [&](int stage, int half, Fragment (&fa)[TM], Fragment (&fw)[TN]) {
    const unsigned char* base = lds + stage * STAGE;
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const unsigned char* from = base + (at[t] ^ (half * 64));
#pragma unroll
      for (int n = 0; n < TN; ++n) fw[n][t] = *(const float*)(from + at_w + n * 16 * ROW);
#pragma unroll
      for (int m = 0; m < TM; ++m) fa[m][t] = *(const float*)(from + at_a + m * 16 * ROW);
    }
  };
  f32x4_t acc[TN][TM], slab[TN][TM], total[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = slab[n][m] = total[n][m] = 0.f;
  auto multiply = [&](const Fragment (&fa)[TM], const Fragment (&fw)[TN], int half) {
#pragma unroll
    for (int t = 2 * half; t < 2 * half + 2; ++t)
#pragma unroll
      for (int n = 0; n < TN; ++n)
#pragma unroll
        for (int m = 0; m < TM; ++m) acc[n][m] = matrix_step(fw[n][t], fa[m][t], acc[n][m]);
  };
  const int steps = (K + STEP - 1) / STEP;
  Fragment fa0[TM], fw0[TN], fa1[TM], fw1[TN];
#pragma unroll
  for (int i = 0; i < STAGES; ++i) issue(i, i);        // a step past the end loads zeros
  loads_but<(STAGES - 1) * LOADS>();
  __syncthreads();
  read(0, 0, fa0, fw0);
  int stage = 0, s = 0;
  for (int slabs_done = 0; s < steps;) {
    // a range's steps in a loop of their own, which touches no sum but acc
    const int range_end = min(steps, s + RANGE_K / STEP);
    for (; s < range_end; ++s) {
      const int next = stage + 1 == STAGES ? 0 : stage + 1;
      read(stage, 1, fa1, fw1);
      multiply(fa0, fw0, 0);
      between_products<2 * TM * TN, READS_OF<TM, TN>, 0>();
      multiply(fa0, fw0, 1);
      __builtin_amdgcn_sched_barrier(0);
      loads_but<(STAGES - 2) * LOADS>();
      __syncthreads();                                 // step s + 1 is there, and nobody reads this step's stage any more
      read(next, 0, fa0, fw0);
      issue(stage, s + STAGES);
      multiply(fa1, fw1, 0);
      between_products<2 * TM * TN, READS_OF<TM, TN>, LOADS>();
      multiply(fa1, fw1, 1);
      __builtin_amdgcn_sched_barrier(0);
      stage = next;
    }
    const bool slab_ends = ++slabs_done % SLAB_RANGES == 0 || s == steps;
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m) {
        slab[n][m] += acc[n][m];
        acc[n][m] = 0.f;
        if constexpr (SLABS) {
          if (slab_ends) {
            total[n][m] += slab[n][m];
            slab[n][m] = 0.f;
          }
        }
      }
  }
  loads_but<0>();                                      // no load may write LDS that the next workgroup has
  if constexpr (GATED) {
#pragma unroll
    for (int n = 0; n < TN; n += 2)
#pragma unroll
      for (int m = 0; m < TM; ++m)
        store_outputs<false>(C, nullptr, SLABS ? gated_outputs(total[n][m], total[n + 1][m]) : gated_outputs(slab[n][m], slab[n + 1][m]),
                             m0 + (wm * TM + m) * 16 + lr, n0 + (wn * TN + n) * 8 + 4 * (lane >> 4), M, N, ldc, quads);
    return;
  }
  auto store = [&](bool in_quads) {
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m)
        store_outputs<ACCUMULATE>(C, bias, SLABS ? total[n][m] : slab[n][m], m0 + (wm * TM + m) * 16 + lr,
                                  n0 + (wn * TN + n) * 16 + 4 * (lane >> 4), M, N, ldc, in_quads);
  };
  if (quads) store(true);
  else store(false);
}

// A workgroup's 16 TM x 16 TN outputs over one slab (blockIdx.y), a range a wave.  A wave has stages of its own, of 16 k,
// and waits for no other before the ranges' sums meet.  LDS rows are 64 bytes (a load instruction: 16 rows); chunk c of row r
// sits in slot c ^ (r / 4 % 4): the 64 values of a block's next four k lie in 64 banks.
// GATED: as in gemm_rows_kernel, but a block's first eight rows are gate's and its others up's of the same eight outputs, as a
// tile may have an odd number of blocks: the sums of an output are 32 lanes apart.
template <int TM, int TN, int STAGES, bool PARTS, bool ACCUMULATE, bool GATED = false>
__global__ __launch_bounds__(256) void gemm_slab_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                        const float* __restrict__ bias, float* __restrict__ C,
                                                        float* __restrict__ parts, int M, int N, int K, long long lda,
                                                        long long ldc, bool quads) {
  typedef __attribute__((address_space(3))) void* lds_at;
  constexpr int STEP = 16, GROUPS = TM + TN, STAGE = GROUPS * 1024, SUM_QUADS = TM * TN;
  static_assert(SUM_QUADS * 1024 <= STAGES * STAGE, "the ranges' sums reuse the stages");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m_tiles = (M + 16 * TM - 1) / (16 * TM);
  const int m0 = blockIdx.x % m_tiles * (16 * TM), n0 = blockIdx.x / m_tiles * (GATED ? 8 * TN : 16 * TN);
  static_assert(!GATED || (!PARTS && !ACCUMULATE), "the gate needs whole sums");
  const int k_begin = blockIdx.y * SLAB_K + wave * RANGE_K, k_end = min(K, k_begin + RANGE_K);
  unsigned char* mine = lds + wave * (STAGES * STAGE);
  f32x4_t acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = 0.f;
  if (k_begin < k_end) {
    const __amdgpu_buffer_rsrc_t a_view = row_view(A + (size_t)m0 * lda + k_begin), w_view = row_view(W + (size_t)n0 * K + k_begin);
    const int ld_row = lane >> 2, ld_chunk = (lane & 3) ^ (lane >> 4), left = k_end - k_begin;
    unsigned off[GROUPS];
#pragma unroll
    for (int g = 0; g < GROUPS; ++g) {
      const int w_row = GATED ? (ld_row & 8 ? N : 0) + min(n0 + 8 * (g - TM) + (ld_row & 7), N - 1) : min(n0 + 16 * (g - TM) + ld_row, N - 1);
      off[g] = (g < TM ? (unsigned)(min(m0 + 16 * g + ld_row, M - 1) - m0) * (unsigned)(lda * 4)
                             : (unsigned)(w_row - n0) * (unsigned)(K * 4)) + ld_chunk * 16;
    }
    auto issue = [&](int stage, int step) {
      unsigned char* to = mine + stage * STAGE;
      const unsigned kb = step * STEP + ld_chunk * 4 < left ? (unsigned)(step * STEP * 4) : NO_CHUNK;
#pragma unroll
      for (int g = 0; g < GROUPS; ++g)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(g < TM ? a_view : w_view, (lds_at)(to + g * 1024), 16, (int)(off[g] + kb), 0, 0, 0);
    };
    const int lr = lane & 15;
    unsigned at[4];                                    // the lane's four k of a block
#pragma unroll
    for (int t = 0; t < 4; ++t) at[t] = (unsigned)(lr * 64 + ((t ^ (lr >> 2)) * 16) + (lane >> 4) * 4);
    auto read = [&](int stage, Fragment (&fa)[TM], Fragment (&fw)[TN]) {
      const unsigned char* base = mine + stage * STAGE;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
#pragma unroll
        for (int n = 0; n < TN; ++n) fw[n][t] = *(const float*)(base + (TM + n) * 1024 + at[t]);
#pragma unroll
        for (int m = 0; m < TM; ++m) fa[m][t] = *(const float*)(base + m * 1024 + at[t]);
      }
    };
    auto multiply = [&](const Fragment (&fa)[TM], const Fragment (&fw)[TN], int half) {
#pragma unroll
      for (int t = 2 * half; t < 2 * half + 2; ++t)
#pragma unroll
        for (int n = 0; n < TN; ++n)
#pragma unroll
          for (int m = 0; m < TM; ++m) acc[n][m] = matrix_step(fw[n][t], fa[m][t], acc[n][m]);
    };
    const int steps = (left + STEP - 1) / STEP;
    Fragment fa0[TM], fw0[TN], fa1[TM], fw1[TN];
#pragma unroll
    for (int i = 0; i < STAGES; ++i) issue(i, i);      // a step past the end loads zeros
    loads_but<(STAGES - 1) * GROUPS>();
    asm volatile("" ::: "memory");
    read(0, fa0, fw0);
    int stage = 0;
    // fa, fw: this step's operands; the next one's are read while their first half is multiplied
    auto step = [&](int s, Fragment (&fa)[TM], Fragment (&fw)[TN], Fragment (&na)[TM], Fragment (&nw)[TN]) {
      const int next = stage + 1 == STAGES ? 0 : stage + 1;
      __builtin_amdgcn_s_waitcnt(0xC07F);              // lgkmcnt(0): this step's operands are in registers, its stage is free
      asm volatile("" ::: "memory");
      issue(stage, s + STAGES);
      loads_but<(STAGES - 1) * GROUPS>();              // step s + 1 is there
      asm volatile("" ::: "memory");
      read(next, na, nw);
      multiply(fa, fw, 0);
      between_products<2 * TM * TN, READS_OF<TM, TN>, 0>();
      multiply(fa, fw, 1);
      __builtin_amdgcn_sched_barrier(0);
      stage = next;
    };
    int s = 0;
    for (; s + 2 <= steps; s += 2) {
      step(s, fa0, fw0, fa1, fw1);
      step(s + 1, fa1, fw1, fa0, fw0);
    }
    if (s < steps) step(s, fa0, fw0, fa1, fw1);
    loads_but<0>();
  }
  __syncthreads();                                     // every wave is done with its stages
  float* sums = (float*)lds;                           // [wave][four sums][lane][4]
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m)
      *(f32x4_t*)(sums + (((size_t)wave * SUM_QUADS + n * TM + m) * 64 + lane) * 4) = acc[n][m];
  __syncthreads();
#pragma unroll
  for (int b0 = 0; b0 < SUM_QUADS; b0 += 4) {
    const int b = b0 + wave;
    if (b >= SUM_QUADS) break;
    f32x4_t v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < SLAB_RANGES; ++w) v += *(const f32x4_t*)(sums + (((size_t)w * SUM_QUADS + b) * 64 + lane) * 4);
    if constexpr (GATED) {
      f32x4_t up;
#pragma unroll
      for (int e = 0; e < 4; ++e) up[e] = __shfl_xor(v[e], 32, 64);
      if (lane < 32)
        store_outputs<false>(C, nullptr, gated_outputs(v, up), m0 + 16 * (b % TM) + (lane & 15), n0 + 8 * (b / TM) + 4 * (lane >> 4), M, N,
                             ldc, quads);
      continue;
    }
    const int row = m0 + 16 * (b % TM) + (lane & 15), column = n0 + 16 * (b / TM) + 4 * (lane >> 4);
    if constexpr (PARTS) store_outputs<false>(parts + (size_t)blockIdx.y * M * N, nullptr, v, row, column, M, N, N, N % 4 == 0);
    else store_outputs<ACCUMULATE>(C, bias, v, row, column, M, N, ldc, quads);
  }
}

// C = the sum of the parts (+ bias) (+ old C): units of `per_slab` to a slab (4: ranges, 1: slabs), slabs in order.
// Four consecutive columns a thread where N allows, so that the parts are read 16 bytes at a time.
template <typename TC, bool ACCUMULATE, int COLUMNS>
__global__ __launch_bounds__(256) void gemm_parts_finish_kernel(const float* __restrict__ parts,
                                                                const float* __restrict__ bias, TC* __restrict__ C,
                                                                int M, int N, long long ldc, int units, int per_slab) {
  const long long at = ((long long)blockIdx.x * blockDim.x + threadIdx.x) * COLUMNS;
  if (at >= (long long)M * N) return;
  const int m = (int)(at / N), n = (int)(at % N);
  float total[COLUMNS];
#pragma unroll
  for (int e = 0; e < COLUMNS; ++e) total[e] = 0.f;
  const size_t stride = (size_t)M * N;
  for (int u = 0; u < units; u += per_slab) {
    float slab[COLUMNS];
#pragma unroll
    for (int e = 0; e < COLUMNS; ++e) slab[e] = 0.f;
#pragma unroll
    for (int r = 0; r < SLAB_RANGES; ++r) {
      if (r < per_slab && u + r < units) {
        const float* from = parts + (size_t)(u + r) * stride + at;
        if constexpr (COLUMNS == 4) {
          const f32x4_t v = *(const f32x4_t*)from;
#pragma unroll
          for (int e = 0; e < 4; ++e) slab[e] += v[e];
        } else {
          slab[0] += from[0];
        }
      }
    }
#pragma unroll
    for (int e = 0; e < COLUMNS; ++e) total[e] += slab[e];
  }
#pragma unroll
  for (int e = 0; e < COLUMNS; ++e) {
    float v = total[e];
    if (bias) v += bias[n + e];
    TC* dst = C + (size_t)m * ldc + n + e;
    if (ACCUMULATE)
      *dst = from_float<TC>(to_float<TC>(*dst) + v);
    else
      *dst = from_float<TC>(v);
  }
}

// How K is cut for a product of M x N: whole (0), in slabs (4) or in ranges (1), so that the workgroups fill the chip
// (256 CUs, four workgroups each). Measured on tiles x K, us whole / slabs / ranges, weights from memory:
//   many tiles need no cut, and the parts' way through memory costs: 2,432 x 896: 193 / - / 221; 912 x 896: 82 / - / 87;
//   2,240 x 1,536: 296 / 293 / 331; but 608 x 896: 64 / - / 64 and 1,120 x 1,536: 181 / 161 / 174;
//   slabs where those are enough: 384 x 8,960: 426 / 295 / 335; 56 x 18,944: 729 / 117 / 138; 512 x 1,536: 75 / 74 / 84;
//   ranges below: 112 x 4,864: 177 / 69 / 66; 256 x 1,536: 54 / 49 / 46; 84 x 896: 32 / - / 18; 14 x 4,864: 154 / 40 / 24.
int matrix_units(int M, int N, int K) {
  const long long tiles = (long long)((M + TILE - 1) / TILE) * ((N + TILE - 1) / TILE);
  const int ranges = (K + RANGE_K - 1) / RANGE_K, slabs = (K + SLAB_K - 1) / SLAB_K;
  if (ranges == 1 || ranges > 65535 || tiles >= (slabs == 1 ? 900 : 1200)) return 0;
  const int units = slabs > 1 && tiles * slabs >= 700 ? SLAB_RANGES : 1;
  // at most 256 MB of parts (2,048 x 2,048 outputs in 16 slabs)
  return (long long)(units == 1 ? ranges : slabs) * M * N <= 64ll * 1024 * 1024 ? units : 0;
}

template <typename TA, typename TW, typename TC, bool ACCUMULATE, int UNITS>
int launch_tiles(const TA* A, const TW* W, const float* bias, TC* C, float* parts, int M, int N, int K, long long lda,
                 long long ldc, hipStream_t s) {
  const long long m_tiles = (M + TILE - 1) / TILE, n_tiles = (N + TILE - 1) / TILE;
  // loads of four k where every row of both operands starts on a boundary of their size
  const bool vector = K % 4 == 0 && lda % 4 == 0 && (uintptr_t)A % (4 * sizeof(TA)) == 0 && (uintptr_t)W % (4 * sizeof(TW)) == 0;
  // A launch counts its threads in 32 bits, and past them leaves tiles out without an error: so many columns are several
  // launches (one is enough where K is cut, which takes few tiles)
  const long long slice = min(n_tiles, 0xffffffffll / 256 / m_tiles);
  for (long long n0 = 0; n0 < n_tiles; n0 += slice) {
    const long long first = n0 * TILE;
    dim3 grid((unsigned)(m_tiles * min(slice, n_tiles - n0)), UNITS ? (K + UNITS * RANGE_K - 1) / (UNITS * RANGE_K) : 1);
    const int columns = (int)min((long long)N - first, slice * TILE);
    const TW* w = W + first * K;
    const float* b = bias ? bias + first : nullptr;
    if (vector)
      gemm_matrix_kernel<TA, TW, TC, ACCUMULATE, UNITS, true><<<grid, 256, 0, s>>>(A, w, b, C + first, parts, M, columns, K, lda, ldc);
    else
      gemm_matrix_kernel<TA, TW, TC, ACCUMULATE, UNITS, false><<<grid, 256, 0, s>>>(A, w, b, C + first, parts, M, columns, K, lda, ldc);
    VK_LAUNCH_CHECK();
  }
  return 0;
}

template <typename TC, bool ACCUMULATE>
int launch_finish(const float* parts, const float* bias, TC* C, int M, int N, long long ldc, int units, int per_slab,
                  hipStream_t s) {
  const long long outputs = (long long)M * N;
  if (N % 4 == 0)
    gemm_parts_finish_kernel<TC, ACCUMULATE, 4><<<(unsigned)((outputs / 4 + 255) / 256), 256, 0, s>>>(parts, bias, C, M, N, ldc, units, per_slab);
  else
    gemm_parts_finish_kernel<TC, ACCUMULATE, 1><<<(unsigned)((outputs + 255) / 256), 256, 0, s>>>(parts, bias, C, M, N, ldc, units, per_slab);
  VK_LAUNCH_CHECK();
  return 0;
}

template <typename TA, typename TW, typename TC>
int launch(const void* A_, const void* W_, const float* bias, void* C_, int M, int N, int K, long long lda, long long ldc,
           int accumulate, int units, float* parts, hipStream_t s) {
  const TA* A = (const TA*)A_;
  const TW* W = (const TW*)W_;
  TC* C = (TC*)C_;
  if (units == 0)
    return accumulate ? launch_tiles<TA, TW, TC, true, 0>(A, W, bias, C, parts, M, N, K, lda, ldc, s)
                      : launch_tiles<TA, TW, TC, false, 0>(A, W, bias, C, parts, M, N, K, lda, ldc, s);
  const int status = units == 1 ? launch_tiles<TA, TW, float, false, 1>(A, W, nullptr, nullptr, parts, M, N, K, lda, ldc, s)
                                : launch_tiles<TA, TW, float, false, SLAB_RANGES>(A, W, nullptr, nullptr, parts, M, N, K, lda, ldc, s);
  if (status != 0) return status;
  const int count = (K + units * RANGE_K - 1) / (units * RANGE_K), per_slab = SLAB_RANGES / units;
  return accumulate ? launch_finish<TC, true>(parts, bias, C, M, N, ldc, count, per_slab, s)
                    : launch_finish<TC, false>(parts, bias, C, M, N, ldc, count, per_slab, s);
}

// Whether four outputs at a time lie on 16 bytes, in C and in the bias.
inline bool stores_quads(const float* C, const float* bias, int N, long long ldc) {
  return N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C & 15) == 0 && ((uintptr_t)bias & 15) == 0;
}

template <int TM, int TN, int WM, int WN, int STAGES>
int launch_rows(const float* A, const float* W, const float* bias, float* C, int M, int N, int K, long long lda, long long ldc,
                int accumulate, hipStream_t s) {
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, lds_bytes = STAGES * (BM + BN) * 128;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipSuccess;
    for (const void* f : {(const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, false, false>, (const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, false, true>,
                          (const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, true, false>, (const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, true, true>})
      if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN - 1) / BN));
  const bool quads = stores_quads(C, bias, N, ldc);
#define VK_ROWS(SLABS, ACC) gemm_rows_kernel<TM, TN, WM, WN, STAGES, SLABS, ACC><<<tiles, 64 * WM * WN, lds_bytes, s>>>(A, W, bias, C, M, N, K, lda, ldc, quads)
  if (K <= SLAB_K) { if (accumulate) VK_ROWS(false, true); else VK_ROWS(false, false); }
  else { if (accumulate) VK_ROWS(true, true); else VK_ROWS(true, false); }
#undef VK_ROWS
  VK_LAUNCH_CHECK();
  return 0;
}

template <int TM, int TN, int STAGES>
int launch_slabs(const float* A, const float* W, const float* bias, float* C, float* parts, int M, int N, int K, long long lda,
                 long long ldc, int accumulate, hipStream_t s) {
  constexpr int BM = 16 * TM, BN = 16 * TN, lds_bytes = 4 * STAGES * (BM + BN) * 64;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipSuccess;
    for (const void* f : {(const void*)gemm_slab_kernel<TM, TN, STAGES, false, false>, (const void*)gemm_slab_kernel<TM, TN, STAGES, false, true>,
                          (const void*)gemm_slab_kernel<TM, TN, STAGES, true, false>})
      if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const int slabs = (K + SLAB_K - 1) / SLAB_K;
  const bool quads = stores_quads(C, bias, N, ldc);
  const dim3 grid((unsigned)(((M + BM - 1) / BM) * ((N + BN - 1) / BN)), slabs);
  if (slabs > 1) gemm_slab_kernel<TM, TN, STAGES, true, false><<<grid, 256, lds_bytes, s>>>(A, W, nullptr, nullptr, parts, M, N, K, lda, 0, false);
  else if (accumulate) gemm_slab_kernel<TM, TN, STAGES, false, true><<<grid, 256, lds_bytes, s>>>(A, W, bias, C, nullptr, M, N, K, lda, ldc, quads);
  else gemm_slab_kernel<TM, TN, STAGES, false, false><<<grid, 256, lds_bytes, s>>>(A, W, bias, C, nullptr, M, N, K, lda, ldc, quads);
  VK_LAUNCH_CHECK();
  if (slabs == 1) return 0;
  return accumulate ? launch_finish<float, true>(parts, bias, C, M, N, ldc, slabs, 1, s)
                    : launch_finish<float, false>(parts, bias, C, M, N, ldc, slabs, 1, s);
}

// The gated forms: C [M, N] from W [2 N, K]; K is one slab where a workgroup owns a slab.
template <int TM, int TN, int WM, int WN, int STAGES>
int launch_rows_gated(const float* A, const float* W, float* C, int M, int N, int K, long long lda, long long ldc, hipStream_t s) {
  constexpr int BM = 16 * TM * WM, BN = 16 * TN * WN, lds_bytes = STAGES * (BM + BN) * 128;
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipSuccess;
    for (const void* f : {(const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, false, false, true>, (const void*)gemm_rows_kernel<TM, TN, WM, WN, STAGES, true, false, true>})
      if (e == hipSuccess) e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN / 2 - 1) / (BN / 2)));
  const bool quads = stores_quads(C, nullptr, N, ldc);
  if (K <= SLAB_K) gemm_rows_kernel<TM, TN, WM, WN, STAGES, false, false, true><<<tiles, 64 * WM * WN, lds_bytes, s>>>(A, W, nullptr, C, M, N, K, lda, ldc, quads);
  else gemm_rows_kernel<TM, TN, WM, WN, STAGES, true, false, true><<<tiles, 64 * WM * WN, lds_bytes, s>>>(A, W, nullptr, C, M, N, K, lda, ldc, quads);
  VK_LAUNCH_CHECK();
  return 0;
}

template <int TM, int TN, int STAGES>
int launch_slab_gated(const float* A, const float* W, float* C, int M, int N, int K, long long lda, long long ldc, hipStream_t s) {
  constexpr int BM = 16 * TM, BN = 16 * TN, lds_bytes = 4 * STAGES * (BM + BN) * 64;
  static bool configured = false;
  if (!configured) {
    const hipError_t e = hipFuncSetAttribute((const void*)gemm_slab_kernel<TM, TN, STAGES, false, false, true>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  const unsigned tiles = (unsigned)(((M + BM - 1) / BM) * ((N + BN / 2 - 1) / (BN / 2)));
  gemm_slab_kernel<TM, TN, STAGES, false, false, true><<<tiles, 256, lds_bytes, s>>>(A, W, nullptr, C, nullptr, M, N, K, lda, ldc,
                                                                                     stores_quads(C, nullptr, N, ldc));
  VK_LAUNCH_CHECK();
  return 0;
}

// Which kernel an all-32-bit product of aligned rows takes.  Both cut M x N into tiles, one a workgroup, and a call lasts as
// long as the CU with the most of them: us = beside + step (tiles of that CU), as measured (weights from memory):
//   slab, 16 x 32 outputs   4 + 3.3 (tiles x slabs)      12 x 1,152 x 896: 6.8 us (14.2 as 64 x 64 tiles cut over workgroups)
//         32 x 32           3.9 + 4.9                    200 x 1,152 x 896: 10.3 (18.4)
//         48 x 32           3.9 + 6.8                    333 x 1,152 x 896: 12.4 (21.2)
//         48 x 48           4.5 + 9.7                    333 x 9,728 x 896: 62.1 (80.7)
//         48 x 64           4.2 + 12.8                   333 x 896 x 4,864: 40.3 (54.2)
//         64 x 64           4.7 + 16.3                   333 x 2,048 x 11,008: 167 (191)
//     and, with several slabs, 3 for adding the parts and their way through memory; the smaller tiles fall behind by a fifth
//     where rows are longer than 8,192 (333 x 2,048 x 11,008: 190 as 48 x 48)
//   rows, 64 x 64           4.1 + 0.0164 K, and 0.0045 K for every three on a CU     256 x 9,728 x 896: 53.6 (65.0)
//         32 x 128          4.8 + 0.0159 K, 0.0038 K for every two                   65 x 17,920 x 1,536: 61.9 (91.7)
//         64 x 128          3.5 + 0.0313 K, 0.0055 K for every two                   333 x 9,728 x 896: 68.0 (80.7)
// Two or three stages leave room for a second or third workgroup on a CU, which hide a wave's own chain of loads better than a
// deeper queue of its own does (a slab's 64 x 64 with four stages took 1.10 of the time with two).  Over 233 sizes from 12 to
// 2,048 rows and K 700 or more the choice takes 0.885 of the time of kernels that exchanged lanes' values, with as many stages and
// without tiles of 48 x 48 (geometric mean), 1.006 of it at worst, and 1.012 of the best form's.  The 64 x 64 tiles cut over workgroups
// are the fastest at none of them; they keep any other type, and rows off 16 bytes.
// Below K 704 a slab's ranges are short or missing, while a walk over all of K has its first loads and its last stores to wait for:
//   slab   the first tile takes what a range of K takes (256 of k or less), each further one on the CU `range` of a step for a whole
//          range alone and all of it from K 704 on (the ranges share the CU's loads); `less` of `beside` falls away
//   rows   `first` more beside it, `each` more a tile, and K in whole steps of 32
//   the 64 x 64 tiles (two stages through registers, no slab to end), which pass both where K is a step or two
// us, as chosen without that and now: 500 x 130 x 132 7.1 / 4.6, 65 x 4,096 x 132 7.7 / 5.8, 257 x 1,152 x 64 5.0 / 4.1, 9 x 9,728 x
// 260 9.7 / 6.6, 2,500 x 9,728 x 16 36.4 / 26.9.  Over 1,430 sizes of K 4 to 1,000 the choice takes 0.89 of the time of kernels that
// exchanged lanes' values in three and four stages, one workgroup a CU (1.03 without it), and 1.026 of the best form's; at worst 1.12 of theirs,
// 1,396 x 9,728 x 24 as 64 x 128, and 2,500 x 1,024 x 1,000 as 48 x 32: rows that do not begin on 128 bytes cost the smaller slabs a
// fifth, which the choice does not tell apart.
enum Direct { NOT_DIRECT, SLAB_16_32, SLAB_32_32, SLAB_48_32, SLAB_64_64, ROWS_64_64, ROWS_32_128, ROWS_64_128, SLAB_48_48, SLAB_48_64 };

Direct direct_plan(int M, int N, int K, long long part_floats) {
  struct Slab { Direct form; int rows, columns, resident; double beside, step, less, range; };
  struct Rows { Direct form; int rows, columns, resident; double beside, step, together, over, first, each; };
  constexpr Slab slab_forms[] = {{SLAB_16_32, 16, 32, 4, 4.0, 3.3, 1.1, 0.41}, {SLAB_32_32, 32, 32, 5, 3.9, 4.9, 0.8, 0.41},
                                 {SLAB_48_32, 48, 32, 4, 3.9, 6.8, 0.5, 0.41}, {SLAB_48_48, 48, 48, 3, 4.5, 9.7, 0.8, 0.45},
                                 {SLAB_48_64, 48, 64, 2, 4.2, 12.8, 0.4, 0.55}, {SLAB_64_64, 64, 64, 2, 4.7, 16.3, 0.4, 0.55}};
  constexpr Rows row_forms[] = {{ROWS_64_64, 64, 64, 3, 4.1, 0.0164, 0.0045, 0.25, -0.7, 0.6},
                                {ROWS_32_128, 32, 128, 2, 4.8, 0.0159, 0.0038, 0.6, -1.3, 0.9},
                                {ROWS_64_128, 64, 128, 2, 3.5, 0.0313, 0.0055, 0.5, 2.0, 0.6}};
  constexpr int SHORT_K = 704, STEP_OR_TWO = 96;
  const long long slabs = (K + SLAB_K - 1) / SLAB_K;
  const double parts = slabs == 1 ? 0.0 : 3.0 + 1.1 * slabs * M * N * 8 / 6e6;
  const double pitch = K % 2048 == 0 ? 1.04 : 1.0;     // weights whose rows are a multiple of 8 KB apart
  const double shorter = K < SHORT_K ? 1.0 - (double)K / SHORT_K : 0.0;
  const int k16 = (K + 15) / 16 * 16, k32 = K < SHORT_K ? (K + 31) / 32 * 32 : K;
  double best = 1e300;
  Direct chosen = NOT_DIRECT;
  auto tiles_of = [&](int rows, int columns) { return (long long)((M + rows - 1) / rows) * ((N + columns - 1) / columns); };
  auto offer = [&](Direct form, long long tiles, double us) {
    if (tiles <= 0xffffffffll / 256 && us < best) best = us, chosen = form;
  };
  if (slabs == 1 || slabs * M * N <= part_floats)
    for (const Slab& f : slab_forms) {
      const long long tiles = tiles_of(f.rows, f.columns);
      const double each = tiles * slabs / 256.0;       // past what is resident a CU short of its share waits for none; past 8 they even out
      const double most = each > 8 ? each + 0.5 : each > f.resident ? ceil(each + 0.05) : ceil(each);
      const double ranges = (double)k16 / RANGE_K;
      const double first = fmin(ranges, 1.0) * (1.0 - 0.03 * shorter);
      const double further = ranges <= 1 ? 0.09 + (f.range - 0.09) * ranges
                                         : fmin(1.0, f.range + (1.0 - f.range) * (k16 - RANGE_K) / (SHORT_K - RANGE_K));
      const double us = (f.beside - f.less * shorter + f.step * (first + (most - 1) * further)) * pitch;
      offer(f.form, tiles, us * (K > 8192 && f.form != SLAB_64_64 ? 1.2 : 1.0) + parts);
    }
  for (const Rows& f : row_forms) {
    const long long tiles = tiles_of(f.rows, f.columns);
    const double each = tiles / 256.0, most = ceil(each) > 2 * f.resident ? each + f.over : ceil(each);
    offer(f.form, tiles, f.beside + (f.step * most + f.together * ceil(most / f.resident)) * k32 * pitch + shorter * (f.first + f.each * most));
  }
  if (K <= STEP_OR_TWO) {
    const double us = 3.3 + 0.0117 * k16 + (0.42 + 0.0203 * k16) * fmax(1.0, tiles_of(TILE, TILE) / 256.0 + 0.3);
    if (us < best) chosen = NOT_DIRECT;
  }
  return chosen;
}

int launch_direct(Direct form, const float* A, const float* W, const float* bias, float* C, float* parts, int M, int N, int K,
                  long long lda, long long ldc, int accumulate, hipStream_t s) {
  switch (form) {
    case SLAB_16_32: return launch_slabs<1, 2, 3>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case SLAB_32_32: return launch_slabs<2, 2, 2>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case SLAB_48_32: return launch_slabs<3, 2, 2>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case SLAB_48_48: return launch_slabs<3, 3, 2>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case SLAB_48_64: return launch_slabs<3, 4, 2>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case SLAB_64_64: return launch_slabs<4, 4, 2>(A, W, bias, C, parts, M, N, K, lda, ldc, accumulate, s);
    case ROWS_64_64: return launch_rows<2, 2, 2, 2, 3>(A, W, bias, C, M, N, K, lda, ldc, accumulate, s);
    case ROWS_32_128: return launch_rows<2, 2, 1, 4, 3>(A, W, bias, C, M, N, K, lda, ldc, accumulate, s);
    case ROWS_64_128: return launch_rows<2, 4, 2, 2, 3>(A, W, bias, C, M, N, K, lda, ldc, accumulate, s);
    case NOT_DIRECT: break;
  }
  return VK_BAD_ARGUMENT;
}

// Rows of 32-bit operands that start on 16 bytes, and tiles whose bytes lie within a view.
constexpr long long DIRECT_MAX_ROW = 4000000;
static_assert(128 * DIRECT_MAX_ROW * 4 < VIEW_BYTES, "a tile has up to 128 rows");
inline bool direct_takes(const void* A, int a_dtype, const void* W, int w_dtype, int c_dtype, int K, long long lda) {
  return a_dtype == DT_F32 && w_dtype == DT_F32 && c_dtype == DT_F32 && K % 4 == 0 && lda % 4 == 0 && lda <= DIRECT_MAX_ROW &&
         K <= DIRECT_MAX_ROW && ((uintptr_t)A & 15) == 0 && ((uintptr_t)W & 15) == 0;
}

// ---------------------------------------------------------------------------------------------
// The weight stream, for 32-bit A and W and up to 8 rows of A. A workgroup of four waves owns 64 rows
// of W and one slab of K; wave w owns range w of the slab, and each of its lanes one row of W, whose
// chain over the range's k it computes for all rows of A (MT accumulators). What a lane needs of W is
// consecutive in memory, which is the opposite of what 64 lanes should request together: so W goes
// through LDS, in stages of 32 k (8 KB per wave): a wave's load instruction fetches eight rows' 128 bytes
// each and writes them straight into LDS (no registers in between), the next stage's instructions in
// flight while this stage is multiplied. Rows are 128 bytes in LDS and cannot be padded (a load writes
// lane L's 16 bytes at 16 L), so chunk c of row r sits in slot c ^ (r / 2 % 8): the 16 lanes that read
// together then touch 16 different 16-byte bank groups. The stage's columns of A come the same way and
// are read by all lanes at one address (a broadcast). A wave has one stage of loads in flight while it
// multiplies the other, and the waves do not wait for one another until the end of the range.
constexpr int STREAM_ROWS = 64, SUB_K = 32, W_STAGE = STREAM_ROWS * SUB_K * 4, W_LOADS = W_STAGE / 1024;

typedef __attribute__((address_space(3))) void* lds_ptr;
typedef __attribute__((address_space(1))) const void* global_ptr;

// Until at most N of the wave's vector memory loads are in flight (they complete in the order of their issue).
// Also a barrier for the compiler: no LDS read may move above the wait for the load that fills what it reads,
// and none below the issue of the load that overwrites it.
template <int N>
__device__ __forceinline__ void wait_loads_but() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <int MT>
__global__ __launch_bounds__(256) void gemm_stream_kernel(const float* __restrict__ A, const float* __restrict__ W,
                                                          float* __restrict__ slabs, int M, int N, int K,
                                                          long long lda) {
  static_assert(MT <= 8, "a load instruction brings 32 k of eight rows of A");
  constexpr int STAGE = W_STAGE + 1024, LOADS = W_LOADS + 1;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * STREAM_ROWS, slab = blockIdx.y;
  const int k_begin = slab * SLAB_K + wave * RANGE_K;
  const int k_end = min(K, k_begin + RANGE_K);           // K is a multiple of 4
  unsigned char* mine = lds + wave * 2 * STAGE;
  float acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = 0.f;

  // what this lane fetches with each load instruction of a stage: of W, chunk (slot ^ swizzle) of row 8 i + sub_row;
  // of A, chunk `slot` of row sub_row. A row past the end is a copy of the last one and is not stored; a
  // chunk past the end of K is a copy of the last one and is never multiplied.
  const int sub_row = lane >> 3, slot = lane & 7;
  const float* w_from[W_LOADS];
  int w_chunk[W_LOADS];
#pragma unroll
  for (int i = 0; i < W_LOADS; ++i) {
    const int r = i * 8 + sub_row;
    w_from[i] = W + (size_t)min(n0 + r, N - 1) * K;
    w_chunk[i] = (slot ^ ((r >> 1) & 7)) << 2;
  }
  auto issue = [&](int k_sub, int stage) {
    unsigned char* to = mine + stage * STAGE;
#pragma unroll
    for (int i = 0; i < W_LOADS; ++i)
      __builtin_amdgcn_global_load_lds((global_ptr)(w_from[i] + min(k_sub + w_chunk[i], K - 4)),
                                       (lds_ptr)(to + i * 1024), 16, 0, 0);
    __builtin_amdgcn_global_load_lds((global_ptr)(A + (size_t)min(sub_row, M - 1) * lda + min(k_sub + (slot << 2), K - 4)),
                                     (lds_ptr)(to + W_STAGE), 16, 0, 0);
  };
  const unsigned my_row = (unsigned)(lane * (SUB_K * 4)), my_swizzle = (unsigned)((lane >> 1) & 7);
  if (k_begin < k_end) {
    const int subs = (k_end - k_begin + SUB_K - 1) / SUB_K;
    issue(k_begin, 0);
    for (int s = 0; s < subs; ++s) {
      const int k_sub = k_begin + s * SUB_K;
      if (s + 1 < subs) {
        issue(k_sub + SUB_K, (s + 1) & 1);   // that stage was multiplied in the step before this one
        wait_loads_but<LOADS>();
      } else {
        wait_loads_but<0>();
      }
      const unsigned char* stage = mine + (s & 1) * STAGE;
      const int chunks = (min(k_end, k_sub + SUB_K) - k_sub) >> 2;
      if (chunks == SUB_K / 4) {
#pragma unroll
        for (int j = 0; j < SUB_K / 4; ++j) {
          const f32x4_t w = *(const f32x4_t*)(stage + my_row + ((j ^ my_swizzle) << 4));
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const f32x4_t a = *(const f32x4_t*)(stage + W_STAGE + m * (SUB_K * 4) + (j << 4));   // the same for every lane
            acc[m] = fmaf(a[0], w[0], acc[m]);
            acc[m] = fmaf(a[1], w[1], acc[m]);
            acc[m] = fmaf(a[2], w[2], acc[m]);
            acc[m] = fmaf(a[3], w[3], acc[m]);
          }
        }
      } else {
        for (int j = 0; j < chunks; ++j) {
          const f32x4_t w = *(const f32x4_t*)(stage + my_row + ((j ^ my_swizzle) << 4));
#pragma unroll
          for (int m = 0; m < MT; ++m) {
            const f32x4_t a = *(const f32x4_t*)(stage + W_STAGE + m * (SUB_K * 4) + (j << 4));
            acc[m] = fmaf(a[0], w[0], acc[m]);
            acc[m] = fmaf(a[1], w[1], acc[m]);
            acc[m] = fmaf(a[2], w[2], acc[m]);
            acc[m] = fmaf(a[3], w[3], acc[m]);
          }
        }
      }
      // the next step's loads overwrite the other stage, which the step before this one read: its reads are done,
      // since their values went into the chains above; nothing of this step may move below the next issue
      asm volatile("" ::: "memory");
    }
  }
  // the slab's sum: the four ranges in ascending order, through LDS (every wave is done with its stages)
  __syncthreads();
  float* sums = (float*)lds;   // [wave][m][row]
#pragma unroll
  for (int m = 0; m < MT; ++m) sums[(wave * MT + m) * STREAM_ROWS + lane] = acc[m];
  __syncthreads();
  for (int at = threadIdx.x; at < MT * STREAM_ROWS; at += 256) {
    const int m = at / STREAM_ROWS, r = at % STREAM_ROWS;
    if (m >= M || n0 + r >= N) continue;
    float total = 0.f;
#pragma unroll
    for (int w = 0; w < SLAB_RANGES; ++w) total += sums[(w * MT + m) * STREAM_ROWS + r];
    slabs[((size_t)slab * M + m) * N + n0 + r] = total;
  }
}

// C = +0 + slab 0 + slab 1 + ... (+ bias) (+ old C): the last level of the sum.
template <typename TC, bool ACCUMULATE>
__global__ __launch_bounds__(256) void gemm_stream_finish_kernel(const float* __restrict__ slabs,
                                                                 const float* __restrict__ bias, TC* __restrict__ C,
                                                                 int M, int N, long long ldc, int num_slabs) {
  const long long at = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (at >= (long long)M * N) return;
  const int m = (int)(at / N), n = (int)(at % N);
  float total = 0.f;
  for (int s = 0; s < num_slabs; ++s) total += slabs[(size_t)s * M * N + at];
  if (bias) total += bias[n];
  TC* dst = C + (size_t)m * ldc + n;
  if (ACCUMULATE)
    *dst = from_float<TC>(to_float<TC>(*dst) + total);
  else
    *dst = from_float<TC>(total);
}

template <int MT>
int launch_stream_as(const float* A, const float* W, float* slabs, int M, int N, int K, long long lda, int num_slabs,
                     hipStream_t s) {
  constexpr int lds_bytes = 4 * 2 * (W_STAGE + 1024);
  static_assert(4 * MT * STREAM_ROWS * 4 <= lds_bytes, "the ranges' sums reuse the stages");
  static bool configured = false;
  if (!configured) {
    hipError_t e = hipFuncSetAttribute((const void*)gemm_stream_kernel<MT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       lds_bytes);
    if (e != hipSuccess) return (int)e;
    configured = true;
  }
  dim3 grid((N + STREAM_ROWS - 1) / STREAM_ROWS, num_slabs);
  gemm_stream_kernel<MT><<<grid, 256, lds_bytes, s>>>(A, W, slabs, M, N, K, lda);
  VK_LAUNCH_CHECK();
  return 0;
}
}  // namespace

// The weight stream: float A (row stride lda, a multiple of 4) and W, M <= 8, K a multiple of 4, 16-byte aligned
// operands; C float or bfloat16. `slabs`: workspace of ceil(K / 1024) M N floats.
extern "C" int vk_gemm_stream(const float* A, const float* W, const float* bias, void* C, int c_dtype, int M, int N,
                              int K, long long lda, long long ldc, int accumulate, float* slabs,
                              long long slab_floats, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (M > 8) return VK_UNSUPPORTED_SIZE;
  if (K < 4 || (K & 3) || (lda & 3) || lda < K || ldc < N || !slabs) return VK_BAD_ARGUMENT;
  if (((uintptr_t)A & 15) || ((uintptr_t)W & 15)) return VK_BAD_ARGUMENT;
  if (accumulate && c_dtype != DT_F32) return VK_BAD_ARGUMENT;
  const int num_slabs = (K + SLAB_K - 1) / SLAB_K;
  if ((long long)num_slabs * M * N > slab_floats || num_slabs > 65535) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  int status;
  if (M <= 1) status = launch_stream_as<1>(A, W, slabs, M, N, K, lda, num_slabs, s);
  else if (M <= 2) status = launch_stream_as<2>(A, W, slabs, M, N, K, lda, num_slabs, s);
  else if (M <= 4) status = launch_stream_as<4>(A, W, slabs, M, N, K, lda, num_slabs, s);
  else status = launch_stream_as<8>(A, W, slabs, M, N, K, lda, num_slabs, s);
  if (status != 0) return status;
  const long long outputs = (long long)M * N;
  const unsigned blocks = (unsigned)((outputs + 255) / 256);
  if (c_dtype == DT_F32) {
    if (accumulate)
      gemm_stream_finish_kernel<float, true><<<blocks, 256, 0, s>>>(slabs, bias, (float*)C, M, N, ldc, num_slabs);
    else
      gemm_stream_finish_kernel<float, false><<<blocks, 256, 0, s>>>(slabs, bias, (float*)C, M, N, ldc, num_slabs);
  } else if (c_dtype == DT_BF16) {
    gemm_stream_finish_kernel<bf16_t, false><<<blocks, 256, 0, s>>>(slabs, bias, (bf16_t*)C, M, N, ldc, num_slabs);
  } else {
    return VK_BAD_ARGUMENT;
  }
  VK_LAUNCH_CHECK();
  return 0;
}

namespace {
int dispatch(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C, int c_dtype, int M, int N,
             int K, long long lda, long long ldc, int accumulate, float* parts, long long part_floats, hipStream_t s) {
  if (direct_takes(A, a_dtype, W, w_dtype, c_dtype, K, lda))
    if (const Direct form = direct_plan(M, N, K, part_floats); form != NOT_DIRECT)
      return launch_direct(form, (const float*)A, (const float*)W, bias, (float*)C, parts, M, N, K, lda, ldc, accumulate, s);
  const int units = parts ? matrix_units(M, N, K) : 0;
  switch (a_dtype * 4 + w_dtype * 2 + c_dtype) {
    case 0: return launch<float, float, float>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 1: return launch<float, float, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 2: return launch<float, bf16_t, float>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 3: return launch<float, bf16_t, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 4: return launch<bf16_t, float, float>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 5: return launch<bf16_t, float, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 6: return launch<bf16_t, bf16_t, float>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
    case 7: return launch<bf16_t, bf16_t, bf16_t>(A, W, bias, C, M, N, K, lda, ldc, accumulate, units, parts, s);
  }
  return VK_BAD_ARGUMENT;
}
}  // namespace

extern "C" long long vk_gemm_generic_workspace(int M, int N, int K);

// The kernel that an all-32-bit product of aligned rows takes with a workspace of part_floats (direct_plan); 0: the 64 x 64 tiles.
extern "C" int vk_gemm_generic_form(int M, int N, int K, long long part_floats) {
  return M <= 0 || N <= 0 || K <= 0 || (K & 3) || K > DIRECT_MAX_ROW ? 0 : (int)direct_plan(M, N, K, part_floats);
}

// A gated product, C [M, N] = up * silu(gate) with W = [gate; up], N rows each, all 32-bit and rows on 16 bytes, in the form and the bits
// of the product of 2 N rows.  Whether it is taken: where that form leaves no parts in memory and W lies within a view.  The gate as a
// launch of its own waits for the product and passes its sums through memory.  us, product and gate in two launches and here: 333 x (2 x
// 4,864) x 896 78.2 / 69.2, of 64 rows 25.8 / 23.8, of 17 17.6 / 16.0; 65 x (2 x 8,960) x 1,536 72.0 / 65.0, of 400 rows 235 / 222.
static Direct gated_plan(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0 || (K & 3) || K > DIRECT_MAX_ROW || 2ll * N * K * 4 >= VIEW_BYTES) return NOT_DIRECT;
  const Direct form = direct_plan(M, 2 * N, K, vk_gemm_generic_workspace(M, 2 * N, K));
  const bool slab = form != ROWS_64_64 && form != ROWS_32_128 && form != ROWS_64_128;
  return slab && K > SLAB_K ? NOT_DIRECT : form;
}
extern "C" int vk_gemm_generic_gated_takes(int M, int N, int K) { return gated_plan(M, N, K) != NOT_DIRECT; }

// Whether it is the faster way there too. Past one round the larger slabs' workgroups end in step with the others of their CU when they apply the
// gate, and the next ones come to a CU in twos (48 x 48: threes): where the last round has fewer for a CU than its places, some CUs get a
// tile more than the product's launch gives any. us, product and gate in two launches and here: 400 x (2 x 4,096) x 1,024, 4.5 tiles of 48 x 64 a CU, 75 / 83;
// 494 x (2 x 2,148) x 948, 2.9, 51 / 61; 441 x (2 x 3,396) x 932, 2.9 of 64 x 64, 67 / 75; 231 x (2 x 6,056) x 956, 4.9 of 48 x 48, 74 / 76. Of 209 such sizes of the
// four larger slabs 83 stay here, in 0.96 of the time, 1.03 at worst, and 126 would take 1.03, 1.2 at worst; of 530 others none takes longer here.
extern "C" int vk_gemm_generic_gated_pays(int M, int N, int K) {
  const Direct form = gated_plan(M, N, K);
  auto most = [&](int rows, int columns) {
    const long long tiles = (long long)((M + rows - 1) / rows) * ((2ll * N + columns - 1) / columns);
    return (tiles + 255) / 256;
  };
  switch (form) {
    case NOT_DIRECT: return 0;
    case SLAB_48_48: return most(48, 48) <= 3 || most(48, 48) % 3 != 2;
    case SLAB_48_64: return most(48, 64) <= 2 || most(48, 64) == 4;
    case SLAB_64_64: return most(64, 64) <= 8 && (most(64, 64) == 1 || most(64, 64) % 2 == 0);
    default: return 1;
  }
}

extern "C" int vk_gemm_generic_gated(const float* A, const float* W, float* C, int M, int N, int K, long long lda, long long ldc,
                                     void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N || lda % 4 || lda > DIRECT_MAX_ROW || (((uintptr_t)A | (uintptr_t)W) & 15)) return VK_BAD_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  switch (gated_plan(M, N, K)) {
    case SLAB_16_32: return launch_slab_gated<1, 2, 3>(A, W, C, M, N, K, lda, ldc, s);
    case SLAB_32_32: return launch_slab_gated<2, 2, 2>(A, W, C, M, N, K, lda, ldc, s);
    case SLAB_48_32: return launch_slab_gated<3, 2, 2>(A, W, C, M, N, K, lda, ldc, s);
    case SLAB_48_48: return launch_slab_gated<3, 3, 2>(A, W, C, M, N, K, lda, ldc, s);
    case SLAB_48_64: return launch_slab_gated<3, 4, 2>(A, W, C, M, N, K, lda, ldc, s);
    case SLAB_64_64: return launch_slab_gated<4, 4, 2>(A, W, C, M, N, K, lda, ldc, s);
    case ROWS_64_64: return launch_rows_gated<2, 2, 2, 2, 3>(A, W, C, M, N, K, lda, ldc, s);
    case ROWS_32_128: return launch_rows_gated<2, 2, 1, 4, 3>(A, W, C, M, N, K, lda, ldc, s);
    case ROWS_64_128: return launch_rows_gated<2, 4, 2, 2, 3>(A, W, C, M, N, K, lda, ldc, s);
    case NOT_DIRECT: break;
  }
  return VK_UNSUPPORTED_SIZE;
}

// Without a workspace: no sums go through memory. dtypes: 0 = float, 1 = bfloat16. lda / ldc are row strides in elements.
extern "C" int vk_gemm_generic(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C,
                               int c_dtype, int M, int N, int K, long long lda, long long ldc, int accumulate,
                               void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N) return VK_BAD_ARGUMENT;
  if ((M + TILE - 1) / TILE > 65535) return VK_UNSUPPORTED_SIZE;
  return dispatch(A, a_dtype, W, w_dtype, bias, C, c_dtype, M, N, K, lda, ldc, accumulate, nullptr, 0, (hipStream_t)stream);
}

// Floats of workspace that vk_gemm_generic_split wants for an M x N product over K (0: it is not split).
extern "C" long long vk_gemm_generic_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int units = matrix_units(M, N, K);
  return units ? (long long)((K + units * RANGE_K - 1) / (units * RANGE_K)) * M * N : 0;
}

// Those of them that the product leaves in memory where its operands are all 32-bit and aligned (direct_takes): one sum a slab in
// the forms over slabs, none where K is one slab or a workgroup walks it. The form is the one that takes all of them into account.
extern "C" long long vk_gemm_generic_direct_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= SLAB_K || K > DIRECT_MAX_ROW) return 0;
  switch (direct_plan(M, N, K, vk_gemm_generic_workspace(M, N, K))) {
    case NOT_DIRECT: case ROWS_64_64: case ROWS_32_128: case ROWS_64_128: return 0;
    default: return (long long)((K + SLAB_K - 1) / SLAB_K) * M * N;
  }
}

// The same product, with K split over workgroups where the tiles alone are too few. `parts`: a workspace of
// vk_gemm_generic_workspace(M, N, K) floats, or of vk_gemm_generic_direct_workspace(M, N, K) where that covers the operands, aligned
// to 16 bytes.
extern "C" int vk_gemm_generic_split(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C,
                                     int c_dtype, int M, int N, int K, long long lda, long long ldc, int accumulate,
                                     float* parts, long long part_floats, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N) return VK_BAD_ARGUMENT;
  if ((M + TILE - 1) / TILE > 65535) return VK_UNSUPPORTED_SIZE;
  const bool direct = direct_takes(A, a_dtype, W, w_dtype, c_dtype, K, lda);
  const long long floats = direct ? vk_gemm_generic_direct_workspace(M, N, K) : vk_gemm_generic_workspace(M, N, K);
  if (floats > part_floats || ((uintptr_t)parts & 15)) return VK_BAD_ARGUMENT;
  return dispatch(A, a_dtype, W, w_dtype, bias, C, c_dtype, M, N, K, lda, ldc, accumulate, parts, part_floats,
                  (hipStream_t)stream);
}
