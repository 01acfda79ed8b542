// Causal grouped-query attention over the paged cache, one workgroup per (token, query head),
// all arithmetic in 32-bit. It serves prompts and decoded tokens alike: a token at position
// `pos` reads the keys at [lo, pos], lo = 0 or pos + 1 - window, from its own request's pages.
// The cache already holds the keys and values of every token of the step.
//
// Formula of the reference (crates/vipera-backend-cpu/src/model.rs:1811-1857): head h uses key
// head h / (heads / kv_heads); score = dot(q, k) * scale with the scale applied after the dot;
// softmax over the visible positions; output = sum of weight * v. The window keeps the last
// `window` positions, the current one included (model.rs:2509). Here the softmax is computed
// online over tiles of 256 keys that start at lo, so the arithmetic of a token depends only on
// its position and the cache contents, not on how the step was cut or batched.
//
// Cache layout: K [page, kv_head, slot, head_dim], V transposed [page, kv_head, head_dim, slot];
// page of position p = table[entry, p / block_size].
#include <type_traits>

#include "attn_extras.h"

namespace {
constexpr int THREADS = 256;
constexpr int MAX_HD = 256;

template <typename T>
__global__ __launch_bounds__(THREADS) void attn_generic_kernel(
    const T* __restrict__ q, long long q_stride, const T* __restrict__ k_cache, const T* __restrict__ v_cache,
    T* __restrict__ out, const int* __restrict__ positions, const int* __restrict__ entry_of_token,
    const int* __restrict__ block_table, int table_width, int block_size, int heads, int kv_heads, int hd,
    float scale, int window, float softcap, const int* __restrict__ skip_single_of, AttnExtras ex) {
  // skip_single_of (entry_start, or null): tokens of entries that hold one token are left to the decode kernel
  if (skip_single_of) {
    const int e = entry_of_token[blockIdx.x];
    if (skip_single_of[e + 1] - skip_single_of[e] == 1) return;
  }
  __shared__ float q_s[MAX_HD];
  __shared__ float p_s[THREADS];
  __shared__ int page_s[THREADS];
  __shared__ float red[16];
  __shared__ float part_s[THREADS];

  const int t = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int kvh = h / (heads / kv_heads);
  const int pos = positions[t];
  const int hi = pos + 1;
  const int lo = first_visible(pos, window);
  const int* table = block_table + (size_t)entry_of_token[t] * table_width;

  for (int d = tid; d < hd; d += THREADS) q_s[d] = to_float<T>(q[(size_t)t * q_stride + (size_t)h * hd + d]);

  // value phase mapping: thread -> (part, d); part p takes keys j with j % parts == p
  const int parts = THREADS / hd > 0 ? THREADS / hd : 1;
  const int vd = tid % hd, vpart = tid / hd;
  const bool v_active = vpart < parts;
  float acc = 0.f, m = -INFINITY, l = 0.f;
  __syncthreads();

  // the positions that a window keeps beside its own (the first `keep_first`) are walked first: index v of the walk
  // is position v below `kept`, and position lo + (v - kept) from there on
  const int kept = min(ex.keep_first, lo);
  const int hi_v = kept + (hi - lo);
  for (int base = 0; base < hi_v; base += THREADS) {
    const int v = base + tid;
    const int p = v < kept ? v : lo + (v - kept);
    float s = -INFINITY;
    int page = -1;
    if (v < hi_v) {
      page = table[p / block_size];
      const T* k_row = k_cache + (((size_t)page * kv_heads + kvh) * block_size + (p % block_size)) * hd;
      float dot = 0.f;
      for (int d = 0; d < hd; ++d) dot = fmaf(q_s[d], to_float<T>(k_row[d]), dot);
      s = capped(dot * scale, softcap);
      if (ex.rel) s += distance_bias(ex, h, pos - p);
    }
    const float tile_max = block_max(s, red);
    const float m_new = fmaxf(m, tile_max);
    const float w = (v < hi_v) ? expf(s - m_new) : 0.f;
    const float tile_sum = block_sum(w, red);
    const float rescale = (m == -INFINITY) ? 0.f : expf(m - m_new);
    l = l * rescale + tile_sum;
    m = m_new;
    p_s[tid] = w;
    page_s[tid] = page;
    __syncthreads();
    if (v_active) {
      acc *= rescale;
      const int count = min(THREADS, hi_v - base);
      for (int j = vpart; j < count; j += parts) {
        const int vj = base + j;
        const int pj = vj < kept ? vj : lo + (vj - kept);
        const T* v_at = v_cache + (((size_t)page_s[j] * kv_heads + kvh) * hd + vd) * block_size + (pj % block_size);
        acc = fmaf(p_s[j], to_float<T>(*v_at), acc);
      }
    }
    __syncthreads();
  }
  // sum the parts in a fixed order
  part_s[tid] = v_active ? acc : 0.f;
  __syncthreads();
  if (tid < hd) {
    float total = 0.f;
    for (int pidx = 0; pidx < parts; ++pidx) total += part_s[pidx * hd + tid];
    out[(size_t)t * heads * hd + (size_t)h * hd + tid] = from_float<T>(total / (l + sink_term(ex, h, m)) * output_gate(ex, t, h));
  }
}

// ---------------------------------------------------------------------------------------------
// Decoding in 32-bit: entries that hold one token. The kernel above gives such a token one workgroup per query
// head, which walks all of its positions alone and reads every key and value once per query head; with a few
// requests of thousands of positions that is a handful of workgroups reading the cache seven times over. Here a
// workgroup owns (entry, key head, chunk of 256 positions) and up to HB query heads of the key head share every
// read; the chunks' (max, sum, weighted sum) are merged by a second kernel in ascending order, as the
// reference's split kernels do (crates/vipera-backend-gpu/src/layer.cu:307-467). A wave owns 64 positions:
//   scores   16 lanes per position, each 4 dims of every 64 (a wave's load is four whole K rows, which lie
//            one after another in a page), the dot products summed over the 16 lanes in a fixed tree;
//   softmax  a lane per position: maximum, exp (library grade), sum over the wave in a fixed tree;
//   output   a lane owns dims dg, dg + 16, ... and every fourth quad of positions (V pages are stored
//            transposed, so four positions of a dim are 16 bytes); a position that the token does not see
//            counts as zero whatever its slot holds, not as its weight of zero times that.
// Which positions a chunk and a wave hold depends on the position alone, so a token's arithmetic does not
// depend on its company. Needs a head width that is a multiple of 4 and pages of a multiple of 4 positions.
constexpr int DEC_CHUNK = 256, DEC_WAVE = 64;

template <int HB, int QC>   // HB query heads together; QC chunks of 64 dims cover the head width
__global__ __launch_bounds__(256) void attn_decode_f32_kernel(
    const float* __restrict__ q, long long q_stride, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, float* __restrict__ partial, const int* __restrict__ entries,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first_pos,
    const int* __restrict__ block_table, int table_width, int block_size, int heads, int kv_heads, int hd,
    float scale, int window, float softcap, int head_blocks, AttnExtras ex) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  __shared__ float sw[4][HB][DEC_WAVE];                 // a wave's scores, then its weights
  __shared__ float merge_o[4][HB][MAX_HD];              // the waves' weighted sums
  __shared__ float merge_ml[4][HB][2];                  // and their (max, sum)
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int slot_index = blockIdx.x, entry = entries[slot_index];
  const int kvh = blockIdx.y / head_blocks, hb = blockIdx.y % head_blocks;
  const int group = heads / kv_heads;
  const int token = entry_start[entry], pos = entry_first_pos[entry];
  const int lo = first_visible(pos, window);
  const int chunk_begin = blockIdx.z * DEC_CHUNK;
  const int first_head = kvh * group + hb * HB;                       // of this block of heads
  const int block_heads = min(HB, group - hb * HB);
  const size_t stride = hd + 2;
  float* dst = partial + (((size_t)slot_index * heads + first_head) * gridDim.z + blockIdx.z) * stride;
  const size_t head_stride = (size_t)gridDim.z * stride;
  const int keep = ex.keep_first;                                     // positions below it stay visible
  if (chunk_begin > pos || (chunk_begin + DEC_CHUNK <= lo && chunk_begin >= keep)) {   // nothing of this chunk is visible
    if ((int)threadIdx.x < block_heads) {
      dst[threadIdx.x * head_stride + hd] = -INFINITY;
      dst[threadIdx.x * head_stride + hd + 1] = 0.f;
    }
    return;
  }
  const int* table = block_table + (size_t)entry * table_width;
  const int wave_begin = chunk_begin + wave * DEC_WAVE;
  const bool wave_sees = wave_begin <= pos && (wave_begin + DEC_WAVE > lo || wave_begin < keep);

  // ---- scores
  const int ps = lane >> 4, c = lane & 15;
  f32x4 qr[HB][QC];
#pragma unroll
  for (int h = 0; h < HB; ++h)
#pragma unroll
    for (int i = 0; i < QC; ++i) {
      const int d = c * 4 + 64 * i;
      qr[h][i] = (h < block_heads && d < hd) ? *(const f32x4*)(q + (size_t)token * q_stride + (size_t)(first_head + h) * hd + d)
                                             : f32x4{0.f, 0.f, 0.f, 0.f};
    }
  if (wave_sees) {
    // Eight steps of four positions at a time: their page ids are requested together, then their K rows, and only
    // then is anything multiplied. A step at a time (look up the page, wait, fetch the row, wait, multiply) made
    // the kernel sixteen pairs of round trips long: 96 us a layer for 134 MB at the 7B shape. No load sits behind
    // a condition: a dim past the head width reads the last four dims again (its q is zero).
    constexpr int AHEAD = 8;
    for (int it0 = 0; it0 < DEC_WAVE / 4; it0 += AHEAD) {
      int at[AHEAD], page[AHEAD];
#pragma unroll
      for (int b = 0; b < AHEAD; ++b) {
        const int p = wave_begin + (it0 + b) * 4 + ps;
        at[b] = p < keep ? min(p, pos) : min(max(p, lo), pos);   // a position outside the range reads one inside it; its score is masked
        page[b] = table[at[b] / block_size];
      }
      f32x4 k4[AHEAD][QC];
#pragma unroll
      for (int b = 0; b < AHEAD; ++b) {
        const float* row = k_cache + (((size_t)page[b] * kv_heads + kvh) * block_size + at[b] % block_size) * hd;
#pragma unroll
        for (int i = 0; i < QC; ++i) k4[b][i] = *(const f32x4*)(row + min(c * 4 + 64 * i, hd - 4));
      }
#pragma unroll
      for (int b = 0; b < AHEAD; ++b) {
        const int p = wave_begin + (it0 + b) * 4 + ps;
        float dot[HB];
#pragma unroll
        for (int h = 0; h < HB; ++h) dot[h] = 0.f;
#pragma unroll
        for (int i = 0; i < QC; ++i)
#pragma unroll
          for (int h = 0; h < HB; ++h) {
            dot[h] = fmaf(qr[h][i][0], k4[b][i][0], dot[h]);
            dot[h] = fmaf(qr[h][i][1], k4[b][i][1], dot[h]);
            dot[h] = fmaf(qr[h][i][2], k4[b][i][2], dot[h]);
            dot[h] = fmaf(qr[h][i][3], k4[b][i][3], dot[h]);
          }
#pragma unroll
        for (int h = 0; h < HB; ++h) {
#pragma unroll
          for (int off = 1; off < 16; off <<= 1) dot[h] += __shfl_xor(dot[h], off, WAVE);
          if (c == 0) {
            float sc = ((p >= lo || p < keep) && p <= pos) ? capped(dot[h] * scale, softcap) : -INFINITY;
            if (ex.rel && h < block_heads) sc += distance_bias(ex, first_head + h, max(pos - p, 0));
            sw[wave][h][(it0 + b) * 4 + ps] = sc;
          }
        }
      }
    }
  }
  __syncthreads();
  // ---- softmax over the wave's 64 positions, a lane per position
  float m[HB], l[HB];
#pragma unroll
  for (int h = 0; h < HB; ++h) {
    const float sc = wave_sees ? sw[wave][h][lane] : -INFINITY;
    m[h] = wave_max(sc);
    const float w = m[h] > -INFINITY ? expf(sc - m[h]) : 0.f;
    l[h] = wave_sum(w);
    sw[wave][h][lane] = w;
  }
  __syncthreads();
  // ---- output: lane (dg, qs) owns dims dg + 16 i and the quads of positions qs, qs + 4, qs + 8, qs + 12
  constexpr int OD = QC * 4;                  // 16-dim steps that cover the head width
  const int dg = lane >> 2, qs = lane & 3;
  float o[HB][OD];
#pragma unroll
  for (int h = 0; h < HB; ++h)
#pragma unroll
    for (int i = 0; i < OD; ++i) o[h][i] = 0.f;
  if (wave_sees) {
    // the four quads' pages first, then their values, no load behind a condition: a quad of which the token sees
    // nothing reads the quad of its own position instead (whose page is held) and counts as zeros
    const float* quad[4];
    bool sees[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int p0 = wave_begin + (qs + 4 * j) * 4;             // four positions of one page
      const bool any = p0 <= pos && (p0 + 3 >= lo || p0 < keep);
      const int from = any ? p0 : (pos & ~3);
#pragma unroll
      for (int e = 0; e < 4; ++e) sees[j][e] = any && (p0 + e >= lo || p0 + e < keep) && p0 + e <= pos;
      quad[j] = v_cache + ((size_t)table[from / block_size] * kv_heads + kvh) * hd * block_size + from % block_size;
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      f32x4 v4[OD];
#pragma unroll
      for (int i = 0; i < OD; ++i) v4[i] = *(const f32x4*)(quad[j] + (size_t)min(dg + 16 * i, hd - 1) * block_size);
      f32x4 w4[HB];
#pragma unroll
      for (int h = 0; h < HB; ++h) w4[h] = *(const f32x4*)&sw[wave][h][(qs + 4 * j) * 4];
#pragma unroll
      for (int i = 0; i < OD; ++i) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v4[i][e] = sees[j][e] ? v4[i][e] : 0.f;
#pragma unroll
        for (int h = 0; h < HB; ++h) {   // a dim past the head width adds into a sum that is never stored
          o[h][i] = fmaf(w4[h][0], v4[i][0], o[h][i]);
          o[h][i] = fmaf(w4[h][1], v4[i][1], o[h][i]);
          o[h][i] = fmaf(w4[h][2], v4[i][2], o[h][i]);
          o[h][i] = fmaf(w4[h][3], v4[i][3], o[h][i]);
        }
      }
    }
  }
#pragma unroll
  for (int h = 0; h < HB; ++h) {
#pragma unroll
    for (int i = 0; i < OD; ++i) {
      float v = o[h][i];
      v += __shfl_xor(v, 1, WAVE);
      v += __shfl_xor(v, 2, WAVE);
      if (qs == 0 && dg + 16 * i < hd) merge_o[wave][h][dg + 16 * i] = v;
    }
    if (lane == 0) {
      merge_ml[wave][h][0] = m[h];
      merge_ml[wave][h][1] = l[h];
    }
  }
  __syncthreads();
  // ---- the four waves' results merged in ascending order
  for (int at = threadIdx.x; at < block_heads * hd; at += 256) {
    const int h = at / hd, d = at % hd;
    float best = -INFINITY;
#pragma unroll
    for (int w = 0; w < 4; ++w) best = fmaxf(best, merge_ml[w][h][0]);
    float total = 0.f, sum = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float mw = merge_ml[w][h][0];
      if (mw > -INFINITY) {
        const float factor = expf(mw - best);
        total = fmaf(merge_o[w][h][d], factor, total);
        sum = fmaf(merge_ml[w][h][1], factor, sum);
      }
    }
    dst[h * head_stride + d] = total;
    if (d == 0) {
      dst[h * head_stride + hd] = best;
      dst[h * head_stride + hd + 1] = sum;
    }
  }
}

// out = sum_c acc_c e^(m_c - M) / sum_c l_c e^(m_c - M) over the chunks in ascending order, M their largest maximum.
template <typename T>
__global__ __launch_bounds__(64) void attn_combine_f32_kernel(const float* __restrict__ partial, T* __restrict__ out,
                                                              const int* __restrict__ entries,
                                                              const int* __restrict__ entry_start, int heads, int hd,
                                                              int chunks, AttnExtras ex) {
  const int slot_index = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
  const size_t stride = hd + 2;
  const float* src = partial + ((size_t)slot_index * heads + h) * chunks * stride;
  float best = -INFINITY;
  for (int ch = lane; ch < chunks; ch += 64) best = fmaxf(best, src[(size_t)ch * stride + hd]);
  best = wave_max(best);
  const int token = entry_start[entries[slot_index]];
  for (int d = lane; d < hd; d += 64) {
    float total = 0.f, sum = 0.f;
    for (int ch = 0; ch < chunks; ++ch) {
      const float mc = src[(size_t)ch * stride + hd];
      if (mc > -INFINITY) {      // an empty chunk's sums hold nothing
        const float factor = expf(mc - best);
        total = fmaf(src[(size_t)ch * stride + d], factor, total);
        sum = fmaf(src[(size_t)ch * stride + hd + 1], factor, sum);
      }
    }
    out[(size_t)token * heads * hd + (size_t)h * hd + d] = from_float<T>(total / (sum + sink_term(ex, h, best)) * output_gate(ex, token, h));
  }
}

// ---------------------------------------------------------------------------------------------
// Prompt portions in 32-bit. The general kernel gives every (token, query head) a workgroup that walks all of the
// token's positions alone: 2,048 tokens x 28 heads read the cache 58 GB over per layer. Here a workgroup owns 16 RB
// consecutive tokens of one entry and one query head and walks the positions in tiles of 64 that begin at
// multiples of 64 (so which positions share a tile, and with it a token's arithmetic, depends on the position alone,
// not on how the prompt was cut).  Both products run on the matrix cores: v_mfma_f32_16x16x4_f32 computes each of its
// outputs as four FMAs in ascending k on top of c (compared with fmaf chains bit for bit), so the sums are those of
// FMA chains:
//   scores   wave w owns the tile's positions 16 w .. 16 w + 15 for all of the workgroup's tokens: an FMA chain over the
//            head width in ascending order;
//   softmax  online over the tiles (crates/vipera-backend-cpu/src/model.rs:1840-1857 is the plain form): thread (ty, tx) of
//            16 x 16 owns positions tx, tx + 16, tx + 32, tx + 48 of tokens ty, ty + 16, ...; a row's
//            maximum and sum over the sixteen lanes that share it in a fixed tree, library-grade exp;
//   output   wave w owns dims 16 w .. 16 w + 15 (and 64 further on): an FMA chain over the tile's positions in ascending order.
// No two waves read the same of K or V, so both go from memory into registers, sixteen bytes a lane, K of the next tile
// while this one's softmax runs; what the matrix instruction wants of a lane (one k of four) comes out of two lane
// exchanges a register pair. Only scores and weights go through LDS, in two buffers, two barriers a tile. Positions past the
// tokens' last one and those before the first one that the first token sees (a window has passed them, their page may have
// been given back and its id in the table is then -1) are read at a place of the tile that is held (stand_in: the first one that
// is seen, the last first position that stays visible, or the tokens' last one); their scores are masked and their values
// count as zeros (a weight of zero times whatever a free slot holds must stay zero).
//
// What bounds it: a few hundred tokens have little to multiply (333 tokens of 14 heads of 64: 0.2 GFLOP a layer, 1.3 us of
// the chip), and their last tokens' walk takes some 2.6 us a tile, one wave a SIMD issuing some 600 instructions; long prompts
// run at 80 TFLOP/s (their matrix instructions wait for the softmax between the products). us, with both products on
// vector FMAs in LDS tiles of 64 tokens (the same sums) and so: 333 tokens of 14 heads of 64 66 and 19; 2,048 of them 378 and
// 182; 4,096 tokens of 28 heads of 128 7,570 and 1,970. Asking for a tile's keys and pages a whole tile ahead gained nothing.
// Head widths that are multiples of 16 up to 128 and pages of a multiple of 4 positions; anything else stays with the
// general kernel.
constexpr int PF_TILE = 64, PF_ROW = PF_TILE + 4;   // a row of scores: eight lanes' 16 bytes of consecutive rows lie in 32 different banks
typedef float pf_f32x4 __attribute__((ext_vector_type(4)));

// r[e] holds k 4 g + e in lane group g = lane / 16; afterwards r[t] holds k 4 t + g.
__device__ __forceinline__ void transpose_lane_groups(float (&r)[4]) {
  auto swap = [](float& x, float& y, auto wide) {
    const unsigned a = __builtin_bit_cast(unsigned, x), b = __builtin_bit_cast(unsigned, y);
    if constexpr (decltype(wide)::value) {
      const auto s = __builtin_amdgcn_permlane32_swap(a, b, false, false);   // the upper half of x and the lower half of y
      x = __builtin_bit_cast(float, (unsigned)s[0]);
      y = __builtin_bit_cast(float, (unsigned)s[1]);
    } else {
      const auto s = __builtin_amdgcn_permlane16_swap(a, b, false, false);   // x's odd groups and y's even ones
      x = __builtin_bit_cast(float, (unsigned)s[0]);
      y = __builtin_bit_cast(float, (unsigned)s[1]);
    }
  };
  swap(r[0], r[1], std::false_type{});
  swap(r[2], r[3], std::false_type{});
  swap(r[0], r[2], std::true_type{});
  swap(r[1], r[3], std::true_type{});
}

// The maximum and the sum over 16 neighbouring lanes, as a tree over lanes 1, 2, 4 and 8 apart, without LDS: once a quad
// holds one value, a mirrored half row brings that of the lane 4 apart, and a mirrored row that of the lane 8 apart.
template <int CTRL>
__device__ __forceinline__ float lane_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
__device__ __forceinline__ float max16(float v) {
  v = fmaxf(v, lane_move<0xB1>(v));
  v = fmaxf(v, lane_move<0x4E>(v));
  v = fmaxf(v, lane_move<0x141>(v));
  return fmaxf(v, lane_move<0x140>(v));
}
__device__ __forceinline__ float sum16(float v) {
  v += lane_move<0xB1>(v);
  v += lane_move<0x4E>(v);
  v += lane_move<0x141>(v);
  return v + lane_move<0x140>(v);
}

template <int DPT, int RB>   // the head width is 16 * DPT, the workgroup's tokens 16 * RB
__global__ __launch_bounds__(256) void attn_prefill_f32_kernel(
    const float* __restrict__ q, long long q_stride, const float* __restrict__ k_cache,
    const float* __restrict__ v_cache, float* __restrict__ out, const int* __restrict__ tiles,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first_pos, const int* __restrict__ block_table,
    int table_width, int block_size, int heads, int kv_heads, float scale, int window, float softcap, int tile_tokens,
    AttnExtras ex) {
  constexpr int HD = 16 * DPT, ROWS = 16 * RB, OB = (DPT + 3) / 4;
  __shared__ __attribute__((aligned(16))) float sw_s[2][ROWS][PF_ROW];   // scores, then weights
  __shared__ float rescale_s[2][ROWS];
  const int parts = tile_tokens / ROWS;                    // workgroups per tile of the step's list
  // the list comes with the tiles that see most positions last; workgroups start in the order of their index, and the
  // long ones should start first, so that the short ones fill the gaps at the end
  const int index = gridDim.x - 1 - blockIdx.x;
  const int tile = index / parts, part = index % parts, h = blockIdx.y;
  const int entry = tiles[2 * tile], offset = tiles[2 * tile + 1] + part * ROWS;
  const int count = entry_start[entry + 1] - entry_start[entry];
  if (offset >= count) return;
  const int rows = min(ROWS, count - offset);
  const int tok0 = entry_start[entry] + offset, pos0 = entry_first_pos[entry] + offset;
  const int last_pos = pos0 + rows - 1;
  const int kvh = h / (heads / kv_heads);
  const int* table = block_table + (size_t)entry * table_width;
  const int tid = threadIdx.x, ty = tid >> 4, tx = tid & 15;
  const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;

  float qf[RB][DPT * 4];   // a row past the end is a copy of the last and is not stored
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const float* row = q + (size_t)(tok0 + min(16 * b + lr, rows - 1)) * q_stride + (size_t)h * HD + 4 * lg;
#pragma unroll
    for (int u = 0; u < DPT; ++u) {
      const pf_f32x4 v = *(const pf_f32x4*)(row + 16 * u);
      float r[4] = {v[0], v[1], v[2], v[3]};
      transpose_lane_groups(r);
#pragma unroll
      for (int t = 0; t < 4; ++t) qf[b][4 * u + t] = r[t];
    }
  }
  float m[RB], l[RB];
  pf_f32x4 o[OB][RB];
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    m[b] = -INFINITY;
    l[b] = 0.f;
#pragma unroll
    for (int d = 0; d < OB; ++d) o[d][b] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  const int lowest = first_visible(pos0, window);   // the first token's first position
  // the tiles of the first positions that stay visible whatever the window has passed come first (those that the
  // window's own tiles do not hold anyway), then the tiles from the window's first position on
  const int keep = ex.keep_first;
  const int first_tile = lowest / PF_TILE, kept_tiles = min((keep + PF_TILE - 1) / PF_TILE, first_tile);
  auto tile_begin = [&](int it) { return (it < kept_tiles ? it : first_tile + (it - kept_tiles)) * PF_TILE; };
  // a tile that every token sees whole needs no masks
  const int lowest_of_last = first_visible(last_pos, window);
  auto whole = [&](int kv0) { return kv0 >= lowest_of_last && kv0 + PF_TILE - 1 <= pos0; };
  // Where a tile's positions lie: its first position's page index is the same for all lanes; a lane's position is at most 63
  // further on, which a 16-bit reciprocal divides exactly (pages of 64 positions and more: a comparison).
  const int reciprocal = block_size < PF_TILE ? 65536 / block_size + 1 : 0;
  const int long_page = block_size < PF_TILE ? 0x7fffffff : block_size;
  auto pages_in = [&](int rem) { return (int)(((unsigned)rem * (unsigned)reciprocal) >> 16) + (rem >= long_page ? 1 : 0); };
  const size_t page_floats = (size_t)kv_heads * block_size * HD;
  const float* k_head = k_cache + (size_t)kvh * block_size * HD + 4 * lg;
  const float* v_head = v_cache + (size_t)kvh * block_size * HD;
  int v_row[OB];   // the lane's dims; past the head width the last one, which is not stored
#pragma unroll
  for (int d = 0; d < OB; ++d) v_row[d] = min(16 * (wave + 4 * d) + lr, HD - 1) * block_size;
  auto held = [&](int p) { return (p >= lowest || p < keep) && p <= last_pos; };
  // a held place of a tile for the lanes whose own is not
  auto stand_in = [&](int it, int kv0) {
    return it < kept_tiles ? min(PF_TILE - 1, keep - 1 - kv0) : kv0 < lowest ? lowest - kv0 : min(PF_TILE - 1, last_pos - kv0);
  };
  pf_f32x4 k_raw[DPT];
  auto fetch_k = [&](int it, int kv0, int index0, auto is_whole) {
    int off = 16 * wave + lr;
    if constexpr (!decltype(is_whole)::value) off = held(kv0 + off) ? off : stand_in(it, kv0);
    const int rem = kv0 - index0 * block_size + off, pages = pages_in(rem);
    const float* row = k_head + (size_t)table[index0 + pages] * page_floats + (rem - pages * block_size) * HD;
#pragma unroll
    for (int u = 0; u < DPT; ++u) k_raw[u] = *(const pf_f32x4*)(row + 16 * u);
  };
  auto walk_tile = [&](int it, int kv0, int& index0, int buf, auto is_whole) {
    constexpr bool WHOLE = decltype(is_whole)::value;
    // the values of four positions of a page and one dim per lane and load
    pf_f32x4 v_raw[OB][4];
    const float* v_at[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      int off = 16 * u + 4 * lg;
      if constexpr (!WHOLE) {
        const int p = kv0 + off;
        off = (p + 3 >= lowest || p < keep) && p <= last_pos ? off : stand_in(it, kv0) & ~3;
      }
      const int rem = kv0 - index0 * block_size + off, pages = pages_in(rem);
      v_at[u] = v_head + (size_t)table[index0 + pages] * page_floats + (rem - pages * block_size);
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int d = 0; d < OB; ++d) v_raw[d][u] = *(const pf_f32x4*)(v_at[u] + v_row[d]);
    // ---- scores
    pf_f32x4 s[RB];
#pragma unroll
    for (int b = 0; b < RB; ++b) s[b] = pf_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < DPT; ++u) {
      float kf[4] = {k_raw[u][0], k_raw[u][1], k_raw[u][2], k_raw[u][3]};
      transpose_lane_groups(kf);
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int b = 0; b < RB; ++b) s[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[t], qf[b][4 * u + t], s[b], 0, 0, 0);
    }
    // the next tile's keys
    if (const int next = tile_begin(it + 1); next <= last_pos) {
      if (it + 1 == kept_tiles) index0 = next / block_size;
      else index0 += pages_in(kv0 - index0 * block_size + PF_TILE % block_size) + PF_TILE / block_size;
      if (whole(next)) fetch_k(it + 1, next, index0, std::true_type{});
      else fetch_k(it + 1, next, index0, std::false_type{});
    }
    // a lane holds token lr's scores of positions 16 wave + 4 lg .. + 3
#pragma unroll
    for (int b = 0; b < RB; ++b) *(pf_f32x4*)&sw_s[buf][16 * b + lr][16 * wave + 4 * lg] = s[b];
    __syncthreads();
    // ---- softmax; weights go back where the scores were, as k 4 t + g of every 16 at 4 g + t (a row stays with its wave)
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int row = 16 * b + ty;
      float sc[4], best = -INFINITY;
#pragma unroll
      for (int j = 0; j < 4; ++j) sc[j] = sw_s[buf][row][tx + 16 * j] * scale;
      const int qpos = pos0 + row;
      if (softcap > 0.f || ex.rel) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sc[j] = capped(sc[j], softcap);
          if (ex.rel) sc[j] += distance_bias(ex, h, max(qpos - (kv0 + tx + 16 * j), 0));
        }
      }
      if constexpr (!WHOLE) {
        const int first = first_visible(qpos, window);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int p = kv0 + tx + 16 * j;
          sc[j] = p <= qpos && (p >= first || p < keep) ? sc[j] : -INFINITY;
        }
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) best = fmaxf(best, sc[j]);
      const float m_new = fmaxf(m[b], max16(best));
      float sum = 0.f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float w = sc[j] > -INFINITY ? expf(sc[j] - m_new) : 0.f;
        sw_s[buf][row][16 * j + 4 * (tx & 3) + (tx >> 2)] = w;
        sum += w;
      }
      sum = sum16(sum);
      const float rescale = m[b] > -INFINITY ? expf(m[b] - m_new) : 0.f;   // nothing seen so far: the sums are zero
      l[b] = l[b] * rescale + sum;
      m[b] = m_new;
      if (tx == 0) rescale_s[buf][row] = rescale;
    }
    __syncthreads();
    // ---- output: a lane holds token lr's dims 16 (wave + 4 d) + 4 lg .. + 3
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const float rescale = rescale_s[buf][16 * b + lr];
#pragma unroll
      for (int d = 0; d < OB; ++d) o[d][b] *= rescale;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      pf_f32x4 w[RB];
#pragma unroll
      for (int b = 0; b < RB; ++b) w[b] = *(const pf_f32x4*)&sw_s[buf][16 * b + lr][16 * u + 4 * lg];
#pragma unroll
      for (int d = 0; d < OB; ++d) {
        float vf[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[e] = WHOLE || held(kv0 + 16 * u + 4 * lg + e) ? v_raw[d][u][e] : 0.f;
        transpose_lane_groups(vf);
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
          for (int b = 0; b < RB; ++b) o[d][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[t], w[b][t], o[d][b], 0, 0, 0);
      }
    }
  };
  int index0 = tile_begin(0) / block_size;
  fetch_k(0, tile_begin(0), index0, std::false_type{});
  for (int it = 0;; ++it) {
    const int kv0 = tile_begin(it);
    if (kv0 > last_pos) break;
    if (whole(kv0)) walk_tile(it, kv0, index0, it & 1, std::true_type{});
    else walk_tile(it, kv0, index0, it & 1, std::false_type{});
  }
  __syncthreads();
#pragma unroll
  for (int b = 0; b < RB; ++b)
    if (tx == 0) rescale_s[0][16 * b + ty] = l[b] + sink_term(ex, h, m[b]);
  __syncthreads();
#pragma unroll
  for (int b = 0; b < RB; ++b) {
    const int row = 16 * b + lr;
    if (row >= rows) continue;
    float* dst = out + (size_t)(tok0 + row) * heads * HD + (size_t)h * HD + 4 * lg;
    const float sum = rescale_s[0][row], gate = output_gate(ex, tok0 + row, h);
#pragma unroll
    for (int d = 0; d < OB; ++d) {
      if (wave + 4 * d >= DPT) continue;
#pragma unroll
      for (int r = 0; r < 4; ++r) dst[16 * (wave + 4 * d) + r] = o[d][b][r] / sum * gate;
    }
  }
}

// 16-token blocks of a workgroup for a step of `items` pairs (64 tokens, head): one while those are about one workgroup a CU,
// two above, which read the keys and values half as often. us with one / two (and with four, slower at every size), from
// position 0: 12 heads of 128 16.3 / 22.7 (48 items), 34.3 / 35.5 (84), 41.2 / 39.2 (96), 28 of them 2,231 / 1,971 (1,792); behind
// 1,000 positions 61.5 / 88.4, 104.5 / 101.7, 111.6 / 105.2. One line for all widths: heads of 96 cross at the same place, narrower
// ones later (14 of 64 behind 1,000 60.0 / 62.5 at 84 items, 62.8 / 65.2 at 98, 67.0 / 67.6 at 112; 8 of 32 58.9 / 64.8 at 96).
inline int prefill_f32_row_blocks(long long items) { return items <= 90 ? 1 : 2; }

template <int DPT>
int launch_prefill_f32(int num_tiles, hipStream_t s, const float* q, long long q_stride, const float* k_cache,
                       const float* v_cache, float* out, const int* tiles, const int* entry_start,
                       const int* entry_first_pos, const int* block_table, int table_width, int block_size, int heads,
                       int kv_heads, float scale, int window, float softcap, int tile_tokens, int row_blocks, AttnExtras ex) {
  dim3 grid((unsigned)((long long)num_tiles * (tile_tokens / (16 * row_blocks))), heads);
#define VK_PF(RBV)                                                                                                    \
  attn_prefill_f32_kernel<DPT, RBV><<<grid, 256, 0, s>>>(q, q_stride, k_cache, v_cache, out, tiles, entry_start,       \
                                                         entry_first_pos, block_table, table_width, block_size, heads, \
                                                         kv_heads, scale, window, softcap, tile_tokens, ex)
  if (row_blocks == 1) VK_PF(1); else VK_PF(2);
#undef VK_PF
  return 0;
}

template <int HB, int QC>
void launch_decode_f32(dim3 grid, hipStream_t s, const float* q, long long q_stride, const float* k_cache,
                       const float* v_cache, float* partial, const int* entries, const int* entry_start,
                       const int* entry_first_pos, const int* block_table, int table_width, int block_size, int heads,
                       int kv_heads, int hd, float scale, int window, float softcap, int head_blocks, AttnExtras ex) {
  attn_decode_f32_kernel<HB, QC><<<grid, 256, 0, s>>>(q, q_stride, k_cache, v_cache, partial, entries, entry_start,
                                                      entry_first_pos, block_table, table_width, block_size, heads,
                                                      kv_heads, hd, scale, window, softcap, head_blocks, ex);
}
}  // namespace

static bool extras_ok(const AttnExtras& ex, int window) {
  return ex.rel_far >= 0 && ex.keep_first >= 0 && (ex.keep_first == 0 || window > 0);
}

extern "C" int vk_attn_generic_ext(const void* q, long long q_stride, const void* k_cache, const void* v_cache,
                               void* out, int dtype, const int* positions, const int* entry_of_token,
                               const int* block_table, int table_width, int block_size, int num_tokens, int heads,
                               int kv_heads, int hd, float scale, int window, float softcap, const int* skip_single_of,
                               const float* sink, const float* rel, int rel_far, int keep_first, const float* gate, long long gate_ld,
                               void* stream) {
  const AttnExtras ex{sink, rel, rel_far, keep_first, gate, gate_ld};
  if (!extras_ok(ex, window)) return VK_BAD_ARGUMENT;
  if (num_tokens <= 0) return 0;
  if (hd <= 0 || hd > MAX_HD) return VK_UNSUPPORTED_SIZE;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || heads > 65535 || block_size <= 0 || table_width <= 0)
    return VK_BAD_ARGUMENT;
  dim3 grid(num_tokens, heads);
  hipStream_t s = (hipStream_t)stream;
  if (dtype == DT_F32)
    attn_generic_kernel<float><<<grid, THREADS, 0, s>>>((const float*)q, q_stride, (const float*)k_cache,
                                                        (const float*)v_cache, (float*)out, positions,
                                                        entry_of_token, block_table, table_width, block_size,
                                                        heads, kv_heads, hd, scale, window, softcap, skip_single_of, ex);
  else if (dtype == DT_BF16)
    attn_generic_kernel<bf16_t><<<grid, THREADS, 0, s>>>((const bf16_t*)q, q_stride, (const bf16_t*)k_cache,
                                                         (const bf16_t*)v_cache, (bf16_t*)out, positions,
                                                         entry_of_token, block_table, table_width, block_size,
                                                         heads, kv_heads, hd, scale, window, softcap, skip_single_of, ex);
  else
    return VK_BAD_ARGUMENT;
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_attn_generic_capped(const void* q, long long q_stride, const void* k_cache, const void* v_cache,
                               void* out, int dtype, const int* positions, const int* entry_of_token,
                               const int* block_table, int table_width, int block_size, int num_tokens, int heads,
                               int kv_heads, int hd, float scale, int window, float softcap, const int* skip_single_of,
                               void* stream) {
  return vk_attn_generic_ext(q, q_stride, k_cache, v_cache, out, dtype, positions, entry_of_token, block_table,
                             table_width, block_size, num_tokens, heads, kv_heads, hd, scale, window, softcap,
                             skip_single_of, nullptr, nullptr, 0, 0, nullptr, 0, stream);
}


// Positions per chunk of vk_attn_decode_f32: `chunks` must cover the longest visible range.
extern "C" int vk_attn_decode_f32_chunk() { return DEC_CHUNK; }

// Attention of the single-token entries listed in `entries` in 32-bit: float q, cache and out. partial: at least
// num_entries * heads * chunks * (hd + 2) floats; chunks * 256 >= longest position + 1.
extern "C" int vk_attn_decode_f32_ext(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                  float* out, float* partial, const int* entries, int num_entries,
                                  const int* entry_start, const int* entry_first_pos, const int* block_table,
                                  int table_width, int block_size, int heads, int kv_heads, int hd, float scale,
                                  int window, float softcap, int chunks, const float* sink, const float* rel, int rel_far,
                                  int keep_first, const float* gate, long long gate_ld,
                               void* stream) {
  const AttnExtras ex{sink, rel, rel_far, keep_first, gate, gate_ld};
  if (!extras_ok(ex, window)) return VK_BAD_ARGUMENT;
  if (num_entries <= 0) return 0;
  if (hd <= 0 || hd > MAX_HD || (hd & 3) || block_size <= 0 || (block_size & 3) || (q_stride & 3)) return VK_UNSUPPORTED_SIZE;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || table_width <= 0 || chunks <= 0 ||
      chunks > 65535)
    return VK_BAD_ARGUMENT;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15)) return VK_BAD_ARGUMENT;
  const int group = heads / kv_heads;
  // heads that share the reads: as many as the registers hold beside hd / 16 sums each
  const int qc = (hd + 63) / 64;
  const int most = qc <= 2 ? 8 : 4;
  int hb = 1;
  while (hb < group && hb < most) hb *= 2;
  const int head_blocks = (group + hb - 1) / hb;
  if (kv_heads * head_blocks > 65535 || heads > 65535) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  dim3 grid(num_entries, kv_heads * head_blocks, chunks);
#define VK_DEC(HBV, QCV)                                                                                          \
  launch_decode_f32<HBV, QCV>(grid, s, q, q_stride, k_cache, v_cache, partial, entries, entry_start, entry_first_pos, \
                              block_table, table_width, block_size, heads, kv_heads, hd, scale, window, softcap, head_blocks, ex)
  if (qc == 1) {
    switch (hb) { case 1: VK_DEC(1, 1); break; case 2: VK_DEC(2, 1); break; case 4: VK_DEC(4, 1); break; default: VK_DEC(8, 1); }
  } else if (qc == 2) {
    switch (hb) { case 1: VK_DEC(1, 2); break; case 2: VK_DEC(2, 2); break; case 4: VK_DEC(4, 2); break; default: VK_DEC(8, 2); }
  } else {
    switch (hb) { case 1: VK_DEC(1, 4); break; case 2: VK_DEC(2, 4); break; default: VK_DEC(4, 4); }
  }
#undef VK_DEC
  VK_LAUNCH_CHECK();
  attn_combine_f32_kernel<float><<<dim3(num_entries, heads), 64, 0, s>>>(partial, out, entries, entry_start, heads, hd, chunks, ex);
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_attn_decode_f32_capped(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                  float* out, float* partial, const int* entries, int num_entries,
                                  const int* entry_start, const int* entry_first_pos, const int* block_table,
                                  int table_width, int block_size, int heads, int kv_heads, int hd, float scale,
                                  int window, float softcap, int chunks, void* stream) {
  return vk_attn_decode_f32_ext(q, q_stride, k_cache, v_cache, out, partial, entries, num_entries, entry_start,
                                entry_first_pos, block_table, table_width, block_size, heads, kv_heads, hd, scale, window,
                                softcap, chunks, nullptr, nullptr, 0, 0, nullptr, 0, stream);
}

// Attention of the step's prompt portions in 32-bit: float q, cache and out. tiles: pairs (entry, first token of the
// tile within the entry), `tile_tokens` tokens a tile (a multiple of 64), as vk_attn_bf16_prefill takes them. Head
// widths that are multiples of 16 up to 128, pages of a multiple of 4 positions.
extern "C" int vk_attn_prefill_f32_ext(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                   float* out, const int* tiles, int num_tiles, int tile_tokens, const int* entry_start,
                                   const int* entry_first_pos, const int* block_table, int table_width, int block_size,
                                   int heads, int kv_heads, int hd, float scale, int window, float softcap,
                                   const float* sink, const float* rel, int rel_far, int keep_first, const float* gate, long long gate_ld,
                               void* stream) {
  const AttnExtras ex{sink, rel, rel_far, keep_first, gate, gate_ld};
  if (!extras_ok(ex, window)) return VK_BAD_ARGUMENT;
  if (num_tiles <= 0) return 0;
  if (hd <= 0 || hd > 128 || (hd & 15) || block_size <= 0 || (block_size & 3) || (q_stride & 3)) return VK_UNSUPPORTED_SIZE;
  if (heads <= 0 || kv_heads <= 0 || heads % kv_heads != 0 || heads > 65535 || table_width <= 0 ||
      tile_tokens <= 0 || tile_tokens % PF_TILE)
    return VK_BAD_ARGUMENT;
  if (((uintptr_t)q & 15) || ((uintptr_t)k_cache & 15) || ((uintptr_t)v_cache & 15)) return VK_BAD_ARGUMENT;
  const long long groups = (long long)num_tiles * (tile_tokens / PF_TILE);
  if (groups > 0x7fffffffLL) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  const int row_blocks = prefill_f32_row_blocks(groups * heads);
  int status = 0;
#define VK_PF(DPTV)                                                                                                  \
  case DPTV:                                                                                                         \
    status = launch_prefill_f32<DPTV>(num_tiles, s, q, q_stride, k_cache, v_cache, out, tiles, entry_start, entry_first_pos, \
                                      block_table, table_width, block_size, heads, kv_heads, scale, window, softcap, tile_tokens, row_blocks, ex); \
    break;
  switch (hd / 16) { VK_PF(1) VK_PF(2) VK_PF(3) VK_PF(4) VK_PF(5) VK_PF(6) VK_PF(7) VK_PF(8) }
#undef VK_PF
  if (status != 0) return status;
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_attn_prefill_f32_capped(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                   float* out, const int* tiles, int num_tiles, int tile_tokens, const int* entry_start,
                                   const int* entry_first_pos, const int* block_table, int table_width, int block_size,
                                   int heads, int kv_heads, int hd, float scale, int window, float softcap, void* stream) {
  return vk_attn_prefill_f32_ext(q, q_stride, k_cache, v_cache, out, tiles, num_tiles, tile_tokens, entry_start,
                                 entry_first_pos, block_table, table_width, block_size, heads, kv_heads, hd, scale, window,
                                 softcap, nullptr, nullptr, 0, 0, nullptr, 0, stream);
}

// The same three without a cap on the scores.
extern "C" int vk_attn_generic(const void* q, long long q_stride, const void* k_cache, const void* v_cache,
                               void* out, int dtype, const int* positions, const int* entry_of_token,
                               const int* block_table, int table_width, int block_size, int num_tokens, int heads,
                               int kv_heads, int hd, float scale, int window, const int* skip_single_of,
                               void* stream) {
  return vk_attn_generic_capped(q, q_stride, k_cache, v_cache, out, dtype, positions, entry_of_token, block_table,
                                table_width, block_size, num_tokens, heads, kv_heads, hd, scale, window, 0.f,
                                skip_single_of, stream);
}

extern "C" int vk_attn_decode_f32(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                  float* out, float* partial, const int* entries, int num_entries,
                                  const int* entry_start, const int* entry_first_pos, const int* block_table,
                                  int table_width, int block_size, int heads, int kv_heads, int hd, float scale,
                                  int window, int chunks, void* stream) {
  return vk_attn_decode_f32_capped(q, q_stride, k_cache, v_cache, out, partial, entries, num_entries, entry_start,
                                   entry_first_pos, block_table, table_width, block_size, heads, kv_heads, hd, scale,
                                   window, 0.f, chunks, stream);
}

extern "C" int vk_attn_prefill_f32(const float* q, long long q_stride, const float* k_cache, const float* v_cache,
                                   float* out, const int* tiles, int num_tiles, int tile_tokens, const int* entry_start,
                                   const int* entry_first_pos, const int* block_table, int table_width, int block_size,
                                   int heads, int kv_heads, int hd, float scale, int window, void* stream) {
  return vk_attn_prefill_f32_capped(q, q_stride, k_cache, v_cache, out, tiles, num_tiles, tile_tokens, entry_start,
                                    entry_first_pos, block_table, table_width, block_size, heads, kv_heads, hd, scale,
                                    window, 0.f, stream);
}
