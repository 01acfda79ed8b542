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
// Two kernels follow it. gemm_stream_kernel, for up to 8 rows of A in 32-bit operands, is a stream
// of the weights: the product of a few tokens is bound by the bytes of W. gemm_matrix_kernel, for
// everything else, runs on the matrix cores: v_mfma_f32_32x32x2_f32 computes each of its outputs as
// fma(a[k + 1], w[k + 1], fma(a[k], w[k], c)), rounded after every product (compared with fmaf chains bit
// for bit, values of all magnitudes, denormal, infinite and NaN ones included), so a chain of these
// instructions over ascending k is the range's chain above.
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
             int K, long long lda, long long ldc, int accumulate, int units, float* parts, hipStream_t s) {
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

// K whole in every workgroup, which needs no workspace. dtypes: 0 = float, 1 = bfloat16. lda / ldc are row strides in elements.
extern "C" int vk_gemm_generic(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C,
                               int c_dtype, int M, int N, int K, long long lda, long long ldc, int accumulate,
                               void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N) return VK_BAD_ARGUMENT;
  if ((M + TILE - 1) / TILE > 65535) return VK_UNSUPPORTED_SIZE;
  return dispatch(A, a_dtype, W, w_dtype, bias, C, c_dtype, M, N, K, lda, ldc, accumulate, 0, nullptr, (hipStream_t)stream);
}

// Floats of workspace that vk_gemm_generic_split wants for an M x N product over K (0: it is not split).
extern "C" long long vk_gemm_generic_workspace(int M, int N, int K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int units = matrix_units(M, N, K);
  return units ? (long long)((K + units * RANGE_K - 1) / (units * RANGE_K)) * M * N : 0;
}

// The same product, with K split over workgroups where the tiles alone are too few. `parts`: a workspace of
// vk_gemm_generic_workspace(M, N, K) floats, aligned to 16 bytes.
extern "C" int vk_gemm_generic_split(const void* A, int a_dtype, const void* W, int w_dtype, const float* bias, void* C,
                                     int c_dtype, int M, int N, int K, long long lda, long long ldc, int accumulate,
                                     float* parts, long long part_floats, void* stream) {
  if (M <= 0 || N <= 0) return 0;
  if (K <= 0 || lda < K || ldc < N) return VK_BAD_ARGUMENT;
  if ((M + TILE - 1) / TILE > 65535) return VK_UNSUPPORTED_SIZE;
  if (vk_gemm_generic_workspace(M, N, K) > part_floats || ((uintptr_t)parts & 15)) return VK_BAD_ARGUMENT;
  return dispatch(A, a_dtype, W, w_dtype, bias, C, c_dtype, M, N, K, lda, ldc, accumulate, matrix_units(M, N, K), parts,
                  (hipStream_t)stream);
}
