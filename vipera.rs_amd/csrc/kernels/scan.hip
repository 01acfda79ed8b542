// Recurrences with a diagonal decay: linear attention whose heads forget at a fixed rate each, and the selective
// scan (a state per channel whose step size depends on the token), with the short causal convolution in front of it.
//
// Everything that enters a recurrence is 32-bit: the state, step sizes, decays and their exponentials.  A request's
// state is one row of a `[slots + 1, floats]` tensor; an entry that starts at position 0 treats its row as zeros, so
// a slot that is used again needs no clearing.  The tokens of a step lie flat, entry after entry; `entry_start[e]`
// is the first token of entry e, `entry_first[e]` its position in the request, `slots[e]` the state row.
//
// Both recurrences give the sixteen lanes of a quarter of a wave one output channel: each lane keeps R of the
// channel's state numbers in registers, a sum over the state is R terms in a lane in ascending order and then four
// DPP exchanges inside the sixteen lanes.  That order depends on the sizes alone, so a token's result does not depend
// on how its prompt was cut or on what else is in the step.  A workgroup is one wave: four channels of one entry,
// whose tokens it walks in order, a few tokens' operands on their way while the few before them are worked on; no
// load sits behind a branch (a token past the entry's end reads the last one again).  What does not depend on the
// state (activations of the inputs, the step sizes' softplus) is taken inside for steps of single tokens and once,
// by a kernel ahead, for a prompt's portion, where every wave would pay for it token behind token.
#include "common.h"
#include "conv_state.h"
#include "scan_parts.h"

__device__ __forceinline__ float scan_silu(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float scan_sigmoid(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float scan_softplus(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

template <int CTRL>
__device__ __forceinline__ float scan_dpp_add(float v) {
  const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false);
  return v + __int_as_float(moved);
}

// The sum over the 16 lanes of a row, in every lane, without LDS: neighbours, pairs of neighbours, the other quad of
// the eight, the other eight.
__device__ __forceinline__ float row16_sum(float v) {
  v = scan_dpp_add<0xB1>(v);     // quad_perm [1, 0, 3, 2]
  v = scan_dpp_add<0x4E>(v);     // quad_perm [2, 3, 0, 1]
  v = scan_dpp_add<0x141>(v);    // row_half_mirror
  v = scan_dpp_add<0x140>(v);    // row_mirror
  return v;
}

constexpr int SCAN_THREADS = 64;      // a workgroup is one wave: four channels of sixteen lanes
constexpr int SCAN_CHANNELS = 4;

static inline int lanes_share(int n) { return n <= 16 ? 1 : n <= 32 ? 2 : n <= 64 ? 4 : n <= 128 ? 8 : 16; }

// ---------------------------------------------------------------------------------------------
// Linear attention with a fixed decay per head:  S <- decay_h S + k v^T,  o = S^T q   (S is dim x vdim).
//   q, k  [T, ldqk] 32-bit, head h at columns h * dim;  v [T, ldv], head h at columns h * vdim
//   act   1: q, k and v pass through silu as they are read
//   state per head `vdim * 16 R` floats: value channel c holds its key channels, padded to 16 R, one after another
// Grid (entries, heads, ceil(vdim / 4)).  VEC: dim = 16 R with R a multiple of 4 and 16-byte rows, so a lane's run of
// key channels is read four at a time.
template <int R, bool VEC>
__global__ __launch_bounds__(SCAN_THREADS) void decay_rule_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                         long long ldqk, const float* __restrict__ v, long long ldv,
                                                         int act, const float* __restrict__ decay,
                                                         float* __restrict__ state, long long state_stride,
                                                         const int* __restrict__ entry_start,
                                                         const int* __restrict__ entry_first,
                                                         const int* __restrict__ slots, int heads, int dim, int vdim,
                                                         float* __restrict__ o) {
  const int e = blockIdx.x, h = blockIdx.y;
  const int lane = threadIdx.x & 63;
  const int part = lane & 15;
  const int vch = blockIdx.z * SCAN_CHANNELS + (lane >> 4);
  const bool live = vch < vdim;
  const int vcol = h * vdim + min(vch, vdim - 1);
  const int t0 = entry_start[e], t1 = entry_start[e + 1];
  const bool fresh = entry_first[e] == 0;
  const float rate = decay[h];
  float* row = state + (long long)slots[e] * state_stride + ((long long)h * vdim + min(vch, vdim - 1)) * (16 * R) + part * R;
  float s[R];
  int col[R];
  bool in[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int c = part * R + r;
    in[r] = c < dim;
    col[r] = h * dim + min(c, dim - 1);
    const float old = row[r];
    s[r] = (fresh || !in[r]) ? 0.f : old;
  }
  if (t1 <= t0) return;
  // D tokens' operands are on their way while the D before them are worked on: a token's step is a few dozen
  // instructions, a load's way through the caches several hundred cycles
  constexpr int D = R >= 16 ? 2 : 4;
  float nk[D][R], nq[D][R], nv[D];
  auto fetch = [&](int first) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int t = min(first + j, t1 - 1);
      const float* kr = k + (long long)t * ldqk;
      const float* qr = q + (long long)t * ldqk;
      if constexpr (VEC) {
        typedef float f32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
        for (int r = 0; r < R; r += 4) {
          const f32x4 k4 = *(const f32x4*)(kr + col[r]), q4 = *(const f32x4*)(qr + col[r]);
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            nk[j][r + i] = k4[i];
            nq[j][r + i] = q4[i];
          }
        }
      } else {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          nk[j][r] = kr[col[r]];
          nq[j][r] = qr[col[r]];
        }
      }
      nv[j] = v[(long long)t * ldv + vcol];
    }
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += D) {
    float ck[D][R], cq[D][R], cv[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        ck[j][r] = nk[j][r];
        cq[j][r] = nq[j][r];
      }
      cv[j] = nv[j];
    }
    fetch(tb + D);
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int t = tb + j;
      if (t >= t1) break;
      if (act) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
          ck[j][r] = scan_silu(ck[j][r]);
          cq[j][r] = scan_silu(cq[j][r]);
        }
        cv[j] = scan_silu(cv[j]);
      }
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float kk = in[r] ? ck[j][r] : 0.f;
        s[r] = fmaf(rate, s[r], kk * cv[j]);
        sum = fmaf(s[r], in[r] ? cq[j][r] : 0.f, sum);
      }
      sum = row16_sum(sum);
      if (part == 0 && live) o[(long long)t * heads * vdim + vcol] = sum;
    }
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = s[r];
  }
}

// The same for prompts' portions, with every token's sum and state formed exactly as above.  A workgroup of two waves takes the
// tokens in blocks through two LDS stages, a block's numbers on their way into registers while the block before is worked on;
// a whole block is unrolled without a branch, two tokens side by side and the next two's LDS reads before them, so that neither
// a read nor a sum, which nothing waits for, is waited for alone; lane j of a channel's sixteen keeps token j's sum, so that a block is stored at once.  Above, a token's eight
// dependent FMAs, four exchanges and a store behind a branch stand in a row on less than a wave a SIMD.  Now the vector
// instructions of a token bound it (about 33 for 8 key channels a lane).  ALL: dim = 16 R; VEC: and 16-byte rows.
// Grid (entries, heads, ceil(vdim / 8)).  16 heads of 128 x 128, against that walk: one portion of 2,048 tokens 549 -> 214 us, portions of 1,000 and
// 834 269 -> 147 us, of 512 138 -> 55 us (without the reads ahead 291, 160 and 75 us).  Short entries stay above: the stages cost
// a single token more than they save.
constexpr int RUN_WAVES = 2, RUN_THREADS = RUN_WAVES * 64, RUN_COLS = 4 * RUN_WAVES;
template <int R, bool ALL, bool VEC>
__global__ __launch_bounds__(RUN_THREADS) void decay_run_kernel(const float* __restrict__ q, const float* __restrict__ k,
                                                                long long ldqk, const float* __restrict__ v, long long ldv,
                                                                const float* __restrict__ decay, float* __restrict__ state,
                                                                long long state_stride, const int* __restrict__ entry_start,
                                                                const int* __restrict__ entry_first,
                                                                const int* __restrict__ slots, int heads, int dim, int vdim,
                                                                float* __restrict__ o) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int KEYS = 16 * R, BLOCK = R <= 8 ? 16 : 8, QUADS = 8 * R;     // QUADS: 16-byte pieces of a token's k and q
  constexpr int LOADS = BLOCK * QUADS / RUN_THREADS, STEP = RUN_THREADS / QUADS;
  static_assert(RUN_THREADS % QUADS == 0 && BLOCK * RUN_COLS <= RUN_THREADS, "a thread's pieces lie in one column");
  __shared__ __attribute__((aligned(16))) float kq[2][BLOCK][2 * KEYS];
  __shared__ float vals[2][BLOCK][RUN_COLS];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int lane = tid & 63, part = lane & 15;
  const int v0 = blockIdx.z * RUN_COLS, mine = (tid >> 6) * 4 + (lane >> 4), vch = v0 + mine;
  const bool live = vch < vdim;
  const int vcol = h * vdim + min(vch, vdim - 1);
  const int t0 = entry_start[e], t1 = entry_start[e + 1];
  if (t1 <= t0) return;       // the whole workgroup
  const bool fresh = entry_first[e] == 0;
  const float rate = decay[h];
  float* row = state + (long long)slots[e] * state_stride + ((long long)h * vdim + min(vch, vdim - 1)) * KEYS + part * R;
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float old = row[r];
    s[r] = (fresh || (!ALL && part * R + r >= dim)) ? 0.f : old;
  }
  // this thread's pieces of a block: keys (or queries) key .. key + 3 of tokens tid / QUADS + i STEP; a token past the end is
  // the last one again, a key channel past dim zero
  const int piece = tid % QUADS, key = piece % (4 * R) * 4, of = tid / QUADS;
  const float* from = (piece < 4 * R ? k : q) + (long long)h * dim;
  // in LDS a lane's n-th pieces lie side by side over the sixteen lanes, so that these read them without bank conflicts
  constexpr int FLOATS = R < 4 ? R : 4;
  const int place = R <= 4 ? key : (key / 4 % (R / 4) * 16 + key / R) * 4;
  f32x4 held[LOADS];
  float held_v = 0.f;
  const float* v_from = v + h * vdim + min(v0 + tid % RUN_COLS, vdim - 1);
  auto fetch = [&](int first) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const float* src = from + (long long)min(first + of + i * STEP, t1 - 1) * ldqk;
      if constexpr (VEC) {
        held[i] = *(const f32x4*)(src + key);
      } else {
#pragma unroll
        for (int n = 0; n < 4; ++n) held[i][n] = src[ALL ? key + n : min(key + n, dim - 1)];
      }
    }
    held_v = v_from[(long long)min(first + tid / RUN_COLS, t1 - 1) * ldv];
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      if constexpr (!ALL) {
#pragma unroll
        for (int n = 0; n < 4; ++n) held[i][n] = key + n < dim ? held[i][n] : 0.f;
      }
      *(f32x4*)&kq[buf][of + i * STEP][piece < 4 * R ? place : KEYS + place] = held[i];
    }
    if (tid < BLOCK * RUN_COLS) vals[buf][tid / RUN_COLS][tid % RUN_COLS] = held_v;
  };
  fetch(t0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int tb = t0; tb < t1; tb += BLOCK, buf ^= 1) {
    const bool more = tb + BLOCK < t1;
    if (more) fetch(tb + BLOCK);
    float sums = 0.f;    // lane j of a channel's sixteen: token j's sum
    auto token = [&](int j, const float (&kj)[R], const float (&qj)[R], float value) {
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[r] = fmaf(rate, s[r], kj[r] * value);
        sum = fmaf(s[r], qj[r], sum);
      }
      sum = row16_sum(sum);
      sums = part == j ? sum : sums;
    };
    auto read = [&](int j, float (&kj)[R], float (&qj)[R], float& value) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const int at = r / FLOATS * 16 * FLOATS + part * FLOATS + r % FLOATS;
        kj[r] = kq[buf][j][at];
        qj[r] = kq[buf][j][KEYS + at];
      }
      value = vals[buf][j][mine];
    };
    const int count = min(BLOCK, t1 - tb);
    if (count == BLOCK) {
      float kp[2][2][R], qp[2][2][R], vp[2][2];     // two tokens at a time, the next two's reads before them
      read(0, kp[0][0], qp[0][0], vp[0][0]);
      read(1, kp[0][1], qp[0][1], vp[0][1]);
#pragma unroll
      for (int j = 0; j < BLOCK; j += 2) {
        const int now = j / 2 & 1;
        if (j + 2 < BLOCK) {
          read(j + 2, kp[now ^ 1][0], qp[now ^ 1][0], vp[now ^ 1][0]);
          read(j + 3, kp[now ^ 1][1], qp[now ^ 1][1], vp[now ^ 1][1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        token(j, kp[now][0], qp[now][0], vp[now][0]);
        token(j + 1, kp[now][1], qp[now][1], vp[now][1]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int j = 0; j < count; ++j) {
        float kj[R], qj[R], value;
        read(j, kj, qj, value);
        token(j, kj, qj, value);
      }
    }
    if (live && part < count) o[(long long)(tb + part) * heads * vdim + vcol] = sums;
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = s[r];
  }
}

// The same for 64 or 128 key channels in rows of whole 16 bytes, with every number formed as above: a block goes straight from memory
// into LDS, in the order in which the lanes read it, from places that are worked out once; two tokens' products, states and sums are
// three runs of instructions none of which waits for the one before it; and sixteen tokens' sums go through the lanes together.
// What bounds it is a token's instructions (32 for 8 key channels a lane, of which one goes out every 1.95 ns on a wave alone on
// its SIMD) and a block's branches and barrier.  us, above and here, launches behind one another in a graph: 16 heads of 128 x 128, one entry of 2,048
// tokens 210 / 171, of 512 55 / 45, of 1,000 and 834 139 / 103, of 512, 456 and 399 72 / 54, eight of 250 84 / 74, of 31 7.0 / 6.5.
template <int R>
__global__ __launch_bounds__(RUN_THREADS) void decay_run_direct_kernel(
    const float* __restrict__ q, const float* __restrict__ k, long long ldqk, const float* __restrict__ v, long long ldv,
    const float* __restrict__ decay, float* __restrict__ state, long long state_stride, const int* __restrict__ entry_start,
    const int* __restrict__ entry_first, const int* __restrict__ slots, int heads, int vdim, float* __restrict__ o) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int KEYS = 16 * R, BLOCK = 16, QUADS = KEYS / 4;      // QUADS: 16-byte pieces of a row
  constexpr int ROWS = 64 / QUADS, LOADS = BLOCK / ROWS / RUN_WAVES;     // rows a load, a wave's loads of a block's keys
  __shared__ __attribute__((aligned(16))) float kq[2][2][BLOCK][KEYS];
  __shared__ float vals[2][BLOCK][RUN_COLS];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, part = lane & 15;
  const int v0 = blockIdx.z * RUN_COLS, mine = (tid >> 6) * 4 + (lane >> 4), vch = v0 + mine;
  const bool live = vch < vdim;
  const int vcol = h * vdim + min(vch, vdim - 1);
  const int t0 = entry_start[e], t1 = entry_start[e + 1];
  if (t1 <= t0) return;       // the whole workgroup
  const bool fresh = entry_first[e] == 0;
  const float rate = decay[h];
  float* row = state + (long long)slots[e] * state_stride + ((long long)h * vdim + min(vch, vdim - 1)) * KEYS + part * R;
  float s[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const float old = row[r];
    s[r] = fresh ? 0.f : old;
  }
  // in LDS a row's pieces stand as the sixteen lanes' first, then their second ones, so that these read them without bank conflicts
  const int slot = lane % QUADS, piece = slot % 16 * (R / 4) + slot / 16, first_row = wave * LOADS * ROWS + lane / QUADS;
  const int row_bytes = (int)ldqk * 4, value_bytes = (int)ldv * 4;
  const int piece_at = (h * KEYS + piece * 4) * 4, value_at = (h * vdim + min(v0 + tid % RUN_COLS, vdim - 1)) * 4;
  int off[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) off[i] = (first_row + i * ROWS) * row_bytes + piece_at;
  const int value_off = tid / RUN_COLS * value_bytes + value_at;
  // where the block that is fetched next begins; a row past the entry's end is its last one, which nobody works on
  const float *next_k = k + t0 * ldqk, *next_q = q + t0 * ldqk, *next_v = v + t0 * ldv;
  auto fetch = [&](int first, int buf) {
    const ScanView keys = scan_view(next_k, 0x7fffffff), queries = scan_view(next_q, 0x7fffffff), values = scan_view(next_v, 0x7fffffff);
    float *to_k = &kq[buf][0][wave * LOADS * ROWS][0], *to_q = &kq[buf][1][wave * LOADS * ROWS][0], *to_v = &vals[buf][wave * 64 / RUN_COLS][0];
    if (first + BLOCK <= t1) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        scan_load_lds<true>(keys, to_k + i * 256, off[i]);
        scan_load_lds<true>(queries, to_q + i * 256, off[i]);
      }
      scan_load_lds<false>(values, to_v, value_off);
    } else {
      const int last = t1 - 1 - first;
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        const int at = min(first_row + i * ROWS, last) * row_bytes + piece_at;
        scan_load_lds<true>(keys, to_k + i * 256, at);
        scan_load_lds<true>(queries, to_q + i * 256, at);
      }
      scan_load_lds<false>(values, to_v, min(tid / RUN_COLS, last) * value_bytes + value_at);
    }
    next_k += BLOCK * ldqk;
    next_q += BLOCK * ldqk;
    next_v += BLOCK * ldv;
  };
  const RowMerge merge(lane);
  float sums = 0.f;    // lane j of a channel's sixteen: token j's sum
  float* to = o + (long long)(t0 + part) * heads * vdim + vcol;
  auto store = [&](int first) {
    if (live && part < t1 - first) *to = sums;
    to += (long long)BLOCK * heads * vdim;
  };
  fetch(t0, 0);
  for (int tb = t0, buf = 0; tb < t1; tb += BLOCK, buf ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0F70);     // the wave's loads of this block, asked for a block ago
    __syncthreads();                        // everybody's; and nobody reads the block before any more
    if (tb > t0) store(tb - BLOCK);
    if (tb + BLOCK < t1) fetch(tb + BLOCK, buf ^ 1);
    auto token = [&](const float (&kj)[R], const float (&qj)[R], float value) {
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        s[r] = fmaf(rate, s[r], kj[r] * value);
        sum = fmaf(s[r], qj[r], sum);
      }
      return sum;
    };
    auto read = [&](int j, float (&kj)[R], float (&qj)[R], float& value) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        kj[r] = kq[buf][0][j][r / 4 * 64 + part * 4 + r % 4];
        qj[r] = kq[buf][1][j][r / 4 * 64 + part * 4 + r % 4];
      }
      value = vals[buf][j][mine];
    };
    const int count = min(BLOCK, t1 - tb);
    if (count == BLOCK) {
      float kp[2][2][R], qp[2][2][R], vp[2][2], sum[4], quads[4];     // two tokens at a time, the next two's reads before them
      read(0, kp[0][0], qp[0][0], vp[0][0]);
      read(1, kp[0][1], qp[0][1], vp[0][1]);
#pragma unroll
      for (int j = 0; j < BLOCK; j += 2) {
        const int now = j / 2 & 1;
        if (j + 2 < BLOCK) {
          read(j + 2, kp[now ^ 1][0], qp[now ^ 1][0], vp[now ^ 1][0]);
          read(j + 3, kp[now ^ 1][1], qp[now ^ 1][1], vp[now ^ 1][1]);
        }
        __builtin_amdgcn_sched_barrier(0);
        float first[R], chain[2] = {0.f, 0.f};      // the state after the first of the two tokens; their sums, in turn
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
          for (int r = 0; r < R; ++r) kp[now][n][r] *= vp[now][n];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; ++r) first[r] = fmaf(rate, s[r], kp[now][0][r]);
#pragma unroll
        for (int r = 0; r < R; ++r) s[r] = fmaf(rate, first[r], kp[now][1][r]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < R; ++r) {
          chain[0] = fmaf(first[r], qp[now][0][r], chain[0]);
          chain[1] = fmaf(s[r], qp[now][1][r], chain[1]);
        }
        sum[j % 4] = chain[0];
        sum[j % 4 + 1] = chain[1];
        if (j % 4 == 2) quads[j / 4] = merge.quads(sum[0], sum[1], sum[2], sum[3]);
        __builtin_amdgcn_sched_barrier(0);
      }
      sums = merge.rows(quads);
    } else {
      for (int j = 0; j < count; ++j) {
        float kj[R], qj[R], value;
        read(j, kj, qj, value);
        const float sum = row16_sum(token(kj, qj, value));
        sums = part == j ? sum : sums;
      }
    }
  }
  store(t0 + (t1 - t0 - 1) / BLOCK * BLOCK);
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = s[r];
  }
}

extern "C" long long vk_decay_rule_head_floats(int dim, int vdim) { return (long long)vdim * 16 * lanes_share(dim); }

static int launch_decay_rule(const float* q, const float* k, long long ldqk, const float* v, long long ldv, int act,
                             const float* decay, float* state, long long state_stride, const int* entry_start,
                             const int* entry_first, const int* slots, int num_entries, int heads, int dim, int vdim,
                             int runs, float* o, void* stream) {
  if (num_entries <= 0) return 0;
  if (heads < 1 || dim < 1 || vdim < 1 || heads > 65535) return VK_BAD_ARGUMENT;
  if (dim > 256) return VK_UNSUPPORTED_SIZE;
  if (state_stride < heads * vk_decay_rule_head_floats(dim, vdim)) return VK_BAD_ARGUMENT;
  dim3 grid(num_entries, heads, (vdim + SCAN_CHANNELS - 1) / SCAN_CHANNELS);
  if (grid.z > 65535) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  const int share = lanes_share(dim);
  if (runs) {
    const dim3 run_grid(num_entries, heads, (vdim + RUN_COLS - 1) / RUN_COLS);
    const bool quads = dim == 16 * share && ldqk % 4 == 0 && (((uintptr_t)q | (uintptr_t)k) & 15) == 0;
#define VK_RUN_AS(RR, ALL, VEC)                                                                                              \
  decay_run_kernel<RR, ALL, VEC><<<run_grid, RUN_THREADS, 0, s>>>(q, k, ldqk, v, ldv, decay, state, state_stride, entry_start, \
                                                                  entry_first, slots, heads, dim, vdim, o)
#define VK_RUN_EACH(RR)                                \
  if (dim == 16 * RR) VK_RUN_AS(RR, true, false);      \
  else VK_RUN_AS(RR, false, false)
#define VK_RUN(RR)                              \
  if (quads) VK_RUN_AS(RR, true, true);         \
  else VK_RUN_EACH(RR)
#define VK_RUN_DIRECT(RR)                                                                                                     \
  decay_run_direct_kernel<RR><<<run_grid, RUN_THREADS, 0, s>>>(q, k, ldqk, v, ldv, decay, state, state_stride, entry_start,     \
                                                               entry_first, slots, heads, vdim, o)
    const bool direct = quads && ldqk < (1 << 24) && ldv < (1 << 24);
    switch (share) {
      case 1: VK_RUN(1); break;
      case 2: VK_RUN(2); break;
      case 4: if (direct) VK_RUN_DIRECT(4); else VK_RUN_EACH(4); break;
      case 8: if (direct) VK_RUN_DIRECT(8); else VK_RUN_EACH(8); break;
      default: VK_RUN(16); break;
    }
#undef VK_RUN
#undef VK_RUN_EACH
#undef VK_RUN_AS
#undef VK_RUN_DIRECT
    VK_LAUNCH_CHECK();
    return 0;
  }
  const bool vec = share >= 4 && dim == 16 * share && ldqk % 4 == 0 && (((uintptr_t)q | (uintptr_t)k) & 15) == 0;
#define VK_DR(RR, VV)                                                                                                 \
  decay_rule_kernel<RR, VV><<<grid, SCAN_THREADS, 0, s>>>(q, k, ldqk, v, ldv, act, decay, state, state_stride,        \
                                                          entry_start, entry_first, slots, heads, dim, vdim, o)
  switch (share) {
    case 1: VK_DR(1, false); break;
    case 2: VK_DR(2, false); break;
    case 4: if (vec) VK_DR(4, true); else VK_DR(4, false); break;
    case 8: if (vec) VK_DR(8, true); else VK_DR(8, false); break;
    default: if (vec) VK_DR(16, true); else VK_DR(16, false); break;
  }
#undef VK_DR
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_decay_rule(const float* q, const float* k, long long ldqk, const float* v, long long ldv, int act,
                             const float* decay, float* state, long long state_stride, const int* entry_start,
                             const int* entry_first, const int* slots, int num_entries, int heads, int dim, int vdim,
                             float* o, void* stream) {
  return launch_decay_rule(q, k, ldqk, v, ldv, act, decay, state, state_stride, entry_start, entry_first, slots, num_entries,
                           heads, dim, vdim, 0, o, stream);
}

// For steps that hold portions of prompts; the inputs' activation is the caller's.
extern "C" int vk_decay_rule_runs(const float* q, const float* k, long long ldqk, const float* v, long long ldv,
                                  const float* decay, float* state, long long state_stride, const int* entry_start,
                                  const int* entry_first, const int* slots, int num_entries, int heads, int dim, int vdim,
                                  float* o, void* stream) {
  return launch_decay_rule(q, k, ldqk, v, ldv, 0, decay, state, state_stride, entry_start, entry_first, slots, num_entries,
                           heads, dim, vdim, 1, o, stream);
}

// ---------------------------------------------------------------------------------------------
// out[t, c] = x[t, c] / rms(x[t, :]) * weight[c] * gate(g[t, c]) over the whole row; gate_act 0: g as it is,
// 1: silu, 2: sigmoid.  One workgroup per token.
template <typename TO>
__global__ __launch_bounds__(256) void gated_norm_kernel(const float* __restrict__ x, const float* __restrict__ weight,
                                                         const float* __restrict__ gate, long long ldg, int gate_act,
                                                         float eps, int width, TO* __restrict__ out) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  const float* src = x + (long long)t * width;
  float ss = 0.f;
  for (int c = threadIdx.x; c < width; c += 256) ss += src[c] * src[c];
  ss = block_sum(ss, scratch);
  const float inv = 1.0f / sqrtf(ss / (float)width + eps);
  for (int c = threadIdx.x; c < width; c += 256) {
    float g = gate[(long long)t * ldg + c];
    g = gate_act == 1 ? scan_silu(g) : gate_act == 2 ? scan_sigmoid(g) : g;
    out[(long long)t * width + c] = from_float<TO>(src[c] * inv * weight[c] * g);
  }
}

extern "C" int vk_gated_norm(const float* x, const float* weight, const float* gate, long long ldg, int gate_act,
                             float eps, int num_tokens, int width, void* out, int out_dtype, void* stream) {
  if (num_tokens <= 0) return 0;
  if (width < 1 || gate_act < 0 || gate_act > 2) return VK_BAD_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  if (out_dtype == DT_F32)
    gated_norm_kernel<float><<<num_tokens, 256, 0, s>>>(x, weight, gate, ldg, gate_act, eps, width, (float*)out);
  else if (out_dtype == DT_BF16)
    gated_norm_kernel<bf16_t><<<num_tokens, 256, 0, s>>>(x, weight, gate, ldg, gate_act, eps, width, (bf16_t*)out);
  else
    return VK_BAD_ARGUMENT;
  VK_LAUNCH_CHECK();
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Short causal convolution over time per channel, a bias, then silu:
//   y[t, c] = silu(bias[c] + sum_j conv[c, j] * in[t - (taps - 1 - j), c])
//   in    [T, ldi] 32-bit, channel c at column c; inputs before the entry's first token come from the state row
//         (`(taps - 1) * C` floats from `conv_offset` on, oldest first), or are zero for an entry at position 0
//   conv  [C, taps], the last column is the current token's
// Outputs: y32 [T, C] 32-bit and, if given, the same rounded to TO.  Grid (tokens, ceil(C / 256)).
template <typename TO>
__global__ __launch_bounds__(256) void causal_conv_kernel(const float* __restrict__ in, long long ldi,
                                                          const float* __restrict__ conv,
                                                          const float* __restrict__ bias, int taps, int C,
                                                          const float* __restrict__ state, long long state_stride,
                                                          long long conv_offset, const int* __restrict__ entry_of,
                                                          const int* __restrict__ entry_start,
                                                          const int* __restrict__ entry_first,
                                                          const int* __restrict__ slots, float* __restrict__ y32,
                                                          TO* __restrict__ yrun) {
  const int t = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int e = entry_of[t];
  const int offset = t - entry_start[e];
  const bool fresh = entry_first[e] == 0;
  const float* old = state + (long long)slots[e] * state_stride + conv_offset;
  float sum = bias ? bias[c] : 0.f;
  for (int j = 0; j < taps; ++j) {
    const int back = taps - 1 - j;
    const bool in_step = back <= offset, in_state = !in_step && !fresh;
    const float* from = in_step ? in + (long long)(t - back) * ldi + c
                                : in_state ? old + (long long)(taps - 1 - (back - offset)) * C + c : in + (long long)t * ldi + c;
    const float x = *from;
    sum = fmaf(conv[(long long)c * taps + j], (in_step || in_state) ? x : 0.f, sum);
  }
  const float y = scan_silu(sum);
  y32[(long long)t * C + c] = y;
  if (yrun) yrun[(long long)t * C + c] = from_float<TO>(y);
}

// The same for up to four taps over longer portions: a thread takes CONV_TOKENS consecutive tokens of its channel and
// keeps the last inputs in registers, so an input is read once (and the K - 1 before the first).  The sum's order is
// causal_conv_kernel's.  Grid (ceil(tokens / CONV_TOKENS), ceil(C / 256)).
constexpr int CONV_TOKENS = 16;
template <int K, typename TO>
__global__ __launch_bounds__(256) void causal_conv_run_kernel(const float* __restrict__ in, long long ldi,
                                                              const float* __restrict__ conv,
                                                              const float* __restrict__ bias, int C,
                                                              const float* __restrict__ state, long long state_stride,
                                                              long long conv_offset, const int* __restrict__ entry_of,
                                                              const int* __restrict__ entry_start,
                                                              const int* __restrict__ entry_first,
                                                              const int* __restrict__ slots, int num_tokens,
                                                              float* __restrict__ y32, TO* __restrict__ yrun) {
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int t0 = blockIdx.x * CONV_TOKENS, t1 = min(t0 + CONV_TOKENS, num_tokens);
  float weight[K], past[K - 1];
#pragma unroll
  for (int j = 0; j < K; ++j) weight[j] = conv[(long long)c * K + j];
  const float b = bias ? bias[c] : 0.f;
  // all inputs of the run are on their way before the first is used
  float x[CONV_TOKENS];
#pragma unroll
  for (int i = 0; i < CONV_TOKENS; ++i) x[i] = in[(long long)min(t0 + i, num_tokens - 1) * ldi + c];
  int of = -1;
#pragma unroll
  for (int i = 0; i < CONV_TOKENS; ++i) {
    const int t = t0 + i;
    if (t >= t1) break;
    const int e = entry_of[t];
    if (e != of) {                       // the run's first token, or another entry's
      of = e;
      const int offset = t - entry_start[e];
      const bool fresh = entry_first[e] == 0;
      const float* old = state + (long long)slots[e] * state_stride + conv_offset + c;
#pragma unroll
      for (int j = 0; j < K - 1; ++j) {
        const int back = K - 1 - j;      // tokens before t
        past[j] = back <= offset ? in[(long long)(t - back) * ldi + c] : fresh ? 0.f : old[(long long)(j + offset) * C];
      }
    }
    float sum = b;
#pragma unroll
    for (int j = 0; j < K - 1; ++j) sum = fmaf(weight[j], past[j], sum);
    sum = fmaf(weight[K - 1], x[i], sum);
#pragma unroll
    for (int j = 0; j + 1 < K - 1; ++j) past[j] = past[j + 1];
    past[K - 2] = x[i];
    const float y = scan_silu(sum);
    y32[(long long)t * C + c] = y;
    if (yrun) yrun[(long long)t * C + c] = from_float<TO>(y);
  }
}

// Both at once where every entry is a single token (one token per entry, so entry e is token entry_start[e]): a thread
// owns a channel, takes its old inputs in order and moves each one place down as it has used it.  The sum's order is
// causal_conv_kernel's.
template <typename TO>
__global__ __launch_bounds__(256) void causal_conv_single_kernel(const float* __restrict__ in, long long ldi,
                                                                 const float* __restrict__ conv,
                                                                 const float* __restrict__ bias, int taps, int C,
                                                                 float* __restrict__ state, long long state_stride,
                                                                 long long conv_offset,
                                                                 const int* __restrict__ entry_start,
                                                                 const int* __restrict__ entry_first,
                                                                 const int* __restrict__ slots, float* __restrict__ y32,
                                                                 TO* __restrict__ yrun) {
  const int e = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int t = entry_start[e];
  const bool fresh = entry_first[e] == 0;
  float* rows = state + (long long)slots[e] * state_stride + conv_offset + c;
  const float now = in[(long long)t * ldi + c];
  float sum = bias ? bias[c] : 0.f;
  for (int j = 0; j + 1 < taps; ++j) {
    const float old = rows[(long long)j * C];
    const float x = fresh ? 0.f : old;
    sum = fmaf(conv[(long long)c * taps + j], x, sum);
    if (j > 0) rows[(long long)(j - 1) * C] = x;
  }
  sum = fmaf(conv[(long long)c * taps + taps - 1], now, sum);
  if (taps > 1) rows[(long long)(taps - 2) * C] = now;
  const float y = scan_silu(sum);
  y32[(long long)t * C + c] = y;
  if (yrun) yrun[(long long)t * C + c] = from_float<TO>(y);
}

extern "C" int vk_causal_conv(const float* in, long long ldi, const float* conv, const float* bias, int taps, int C,
                              float* state, long long state_stride, long long conv_offset, const int* entry_of,
                              const int* entry_start, const int* entry_first, const int* slots, int num_tokens,
                              int num_entries, float* y32, void* yrun, int run_dtype, void* stream) {
  if (num_tokens <= 0) return 0;
  if (taps < 1 || C < 1 || num_entries < 1) return VK_BAD_ARGUMENT;
  dim3 grid(num_tokens, (C + 255) / 256);
  if (grid.y > 65535) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  if (num_tokens == num_entries) {
    dim3 singles(num_entries, grid.y);
    if (yrun == nullptr || run_dtype == DT_F32)
      causal_conv_single_kernel<float><<<singles, 256, 0, s>>>(in, ldi, conv, bias, taps, C, state, state_stride, conv_offset,
                                                               entry_start, entry_first, slots, y32, (float*)yrun);
    else if (run_dtype == DT_BF16)
      causal_conv_single_kernel<bf16_t><<<singles, 256, 0, s>>>(in, ldi, conv, bias, taps, C, state, state_stride, conv_offset,
                                                                entry_start, entry_first, slots, y32, (bf16_t*)yrun);
    else
      return VK_BAD_ARGUMENT;
    VK_LAUNCH_CHECK();
    return 0;
  }
  if (yrun != nullptr && run_dtype != DT_F32 && run_dtype != DT_BF16) return VK_BAD_ARGUMENT;
  const bool wide = yrun == nullptr || run_dtype == DT_F32;
  if (taps >= 2 && taps <= 4 && num_tokens >= 256) {
    dim3 runs((num_tokens + CONV_TOKENS - 1) / CONV_TOKENS, grid.y);
#define VK_CONV_RUN(K)                                                                                               \
  if (wide)                                                                                                          \
    causal_conv_run_kernel<K, float><<<runs, 256, 0, s>>>(in, ldi, conv, bias, C, state, state_stride, conv_offset,  \
                                                          entry_of, entry_start, entry_first, slots, num_tokens, y32, \
                                                          (float*)yrun);                                             \
  else                                                                                                               \
    causal_conv_run_kernel<K, bf16_t><<<runs, 256, 0, s>>>(in, ldi, conv, bias, C, state, state_stride, conv_offset, \
                                                           entry_of, entry_start, entry_first, slots, num_tokens, y32, \
                                                           (bf16_t*)yrun)
    switch (taps) {
      case 2: VK_CONV_RUN(2); break;
      case 3: VK_CONV_RUN(3); break;
      default: VK_CONV_RUN(4); break;
    }
#undef VK_CONV_RUN
  } else if (wide)
    causal_conv_kernel<float><<<grid, 256, 0, s>>>(in, ldi, conv, bias, taps, C, state, state_stride, conv_offset,
                                                   entry_of, entry_start, entry_first, slots, y32, (float*)yrun);
  else
    causal_conv_kernel<bf16_t><<<grid, 256, 0, s>>>(in, ldi, conv, bias, taps, C, state, state_stride, conv_offset,
                                                    entry_of, entry_start, entry_first, slots, y32, (bf16_t*)yrun);
  VK_LAUNCH_CHECK();
  if (taps > 1) {
    conv_keep_kernel<<<dim3(num_entries, grid.y), 256, 0, s>>>(in, ldi, taps, C, state, state_stride, conv_offset,
                                                               entry_start, entry_first, slots);
    VK_LAUNCH_CHECK();
  }
  return 0;
}

// ---------------------------------------------------------------------------------------------
// Selective scan.  Per channel c and state n:
//   dt = softplus(dtraw[t, c] + dt_bias[c]);  S[c, n] <- exp(dt A[c, n]) S[c, n] + dt x[t, c] B[t, n]
//   y = sum_n S[c, n] C[t, n] + D[c] x[t, c];  out[t, c] = y * silu(z[t, c])
//   A = -exp(a_log) [C, N];  B and C are column ranges of one [T, ldbc] buffer;  z a column range of [T, ldz]
//   state per channel 16 R floats (N padded), channel after channel
//   prepared: dtraw already holds softplus(dt + dt_bias) and z already silu(z) (scan_prepare below; a prompt's tokens
//   would each pay for them behind one another here)
// Grid (entries, ceil(C / 4)).
template <int R, typename TO>
__global__ __launch_bounds__(SCAN_THREADS) void selective_scan_kernel(
    const float* __restrict__ x, const float* __restrict__ dtraw, long long lddt, const float* __restrict__ dt_bias,
    const float* __restrict__ bmat, const float* __restrict__ cmat, long long ldbc, const float* __restrict__ a_log,
    const float* __restrict__ skip, const float* __restrict__ z, long long ldz, float* __restrict__ state,
    long long state_stride, const int* __restrict__ entry_start, const int* __restrict__ entry_first,
    const int* __restrict__ slots, int C, int N, int prepared, TO* __restrict__ out) {
  const int e = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int part = lane & 15;
  const int ch_raw = blockIdx.y * SCAN_CHANNELS + (lane >> 4);
  const bool live = ch_raw < C;
  const int ch = min(ch_raw, C - 1);
  const int t0 = entry_start[e], t1 = entry_start[e + 1];
  const bool fresh = entry_first[e] == 0;
  float* row = state + (long long)slots[e] * state_stride + (long long)ch * (16 * R) + part * R;
  float s[R], a[R];
  int col[R];
  bool in[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = part * R + r;
    in[r] = n < N;
    col[r] = min(n, N - 1);
    const float old = row[r];
    s[r] = (fresh || !in[r]) ? 0.f : old;
    a[r] = -expf(a_log[(long long)ch * N + col[r]]);
  }
  if (t1 <= t0) return;
  const float bias = dt_bias[ch], d = skip[ch];
  // D tokens' operands are on their way while the D before them are worked on (see decay_rule_kernel)
  constexpr int D = R >= 8 ? 2 : R >= 4 ? 4 : 8;
  float nb[D][R], nc[D][R], nx[D], ndt[D], nz[D];
  auto fetch = [&](int first) {
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int t = min(first + j, t1 - 1);
#pragma unroll
      for (int r = 0; r < R; ++r) {
        nb[j][r] = bmat[(long long)t * ldbc + col[r]];
        nc[j][r] = cmat[(long long)t * ldbc + col[r]];
      }
      nx[j] = x[(long long)t * C + ch];
      ndt[j] = dtraw[(long long)t * lddt + ch];
      nz[j] = z[(long long)t * ldz + ch];
    }
  };
  fetch(t0);
  for (int tb = t0; tb < t1; tb += D) {
    float cb[D][R], cc[D][R], cx[D], cdt[D], cz[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        cb[j][r] = nb[j][r];
        cc[j][r] = nc[j][r];
      }
      cx[j] = nx[j];
      cdt[j] = ndt[j];
      cz[j] = nz[j];
    }
    fetch(tb + D);
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const int t = tb + j;
      if (t >= t1) break;
      const float dt = prepared ? cdt[j] : scan_softplus(cdt[j] + bias);
      const float dtx = dt * cx[j];
      float sum = 0.f;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        const float keep = expf(dt * a[r]);
        s[r] = fmaf(keep, s[r], in[r] ? dtx * cb[j][r] : 0.f);
        sum = fmaf(s[r], in[r] ? cc[j][r] : 0.f, sum);
      }
      sum = row16_sum(sum);
      if (part == 0 && live)
        out[(long long)t * C + ch] = from_float<TO>(fmaf(d, cx[j], sum) * (prepared ? cz[j] : scan_silu(cz[j])));
    }
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = s[r];
  }
}

// The same for prompts' portions (`prepared`) and up to 64 states, with every token's sum and state formed exactly as above.  A
// workgroup of four waves (sixteen channels) takes the tokens in blocks (of 32 for a state a lane and 32 tokens an entry, else of 16) through two LDS stages, where a
// state's (a channel's) numbers of neighbouring tokens lie side by side, so that a lane reads four tokens' at once; a block's numbers
// are on their way into registers while the block before is worked on.  A whole block is unrolled without a branch: the exponentials,
// products and exchanges of neighbouring tokens, which wait for nothing but the state's one FMA a token, fill each other's
// latencies, and sixteen tokens' sums go through the lanes together.  Lane j of a channel's sixteen ends up with token j's sum and
// finishes that token's output.  What bounds it is the instructions (about 23 a token for a state a lane, fourteen of them the
// exponential).  ALL: N = 16 R.  4,096 channels of 16 states, with blocks of 16 and every token's sum by itself, and so: portions of
// 1,000 and 834 tokens 108 -> 95 us, one of 2,048 165 -> 144, of 512 44 -> 39, eight of 250 85 -> 74.  Short entries have no block of 32 and pay for
// its stages: in blocks of 32 and of 16, 64 of 20 tokens 72 -> 62 us, 30 of 5 16.4 -> 13.5, one of 16 5.1 -> 4.0.  Beyond 64 states a lane's registers and the stages grow past what the chip holds at once, and the walk above stays.
template <int R, int BLOCK, bool ALL, typename TO>
__global__ __launch_bounds__(256) void selective_run_kernel(
    const float* __restrict__ x, const float* __restrict__ dt, long long lddt, const float* __restrict__ bmat,
    const float* __restrict__ cmat, long long ldbc, const float* __restrict__ a_log, const float* __restrict__ skip,
    const float* __restrict__ z, long long ldz, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int C, int N,
    TO* __restrict__ out) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int HALVES = BLOCK / 16, ROW = BLOCK + 4, STATES = 16 * R;
  constexpr int BC_TOKENS = 256 / STATES, BC_LOADS = BLOCK / BC_TOKENS;
  __shared__ __attribute__((aligned(16))) float bc[2][2][STATES][ROW];     // B and C: [state][token]
  __shared__ __attribute__((aligned(16))) float xdz[2][3][16][ROW];        // x, dt and the gate: [channel][token]
  const int e = blockIdx.x, tid = threadIdx.x;
  const int lane = tid & 63, part = lane & 15, mine = (tid >> 6) * 4 + (lane >> 4);
  const int ch_raw = blockIdx.y * 16 + mine, ch = min(ch_raw, C - 1);
  const bool live = ch_raw < C;
  const int t0 = entry_start[e], t1 = entry_start[e + 1];
  if (t1 <= t0) return;       // the whole workgroup
  const bool fresh = entry_first[e] == 0;
  float* row = state + (long long)slots[e] * state_stride + (long long)ch * STATES + part * R;
  float s[R], a[R];
  bool in[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const int n = part * R + r;
    in[r] = ALL || n < N;
    const float old = row[r];
    s[r] = (fresh || !in[r]) ? 0.f : old;
    a[r] = -expf(a_log[(long long)ch * N + (ALL ? n : min(n, N - 1))]);
  }
  const float d = skip[ch];
  // this thread's numbers of a block: state tid % STATES of tokens tid / STATES + i (256 / STATES), channel tid % 16 of tokens
  // tid / 16 + 16 i; a token past the end is the last one again
  const int state_of = tid % STATES, bc_token = tid / STATES, ch_token = tid / 16;
  const int bc_col = ALL ? state_of : min(state_of, N - 1);
  const long long ch_col = min((int)blockIdx.y * 16 + tid % 16, C - 1);
  float held_b[BC_LOADS] = {}, held_c[BC_LOADS] = {}, held_x[HALVES] = {}, held_dt[HALVES] = {}, held_z[HALVES] = {};
  auto fetch = [&](int first) {
    if constexpr (HALVES == 1) {
#pragma unroll
      for (int i = 0; i < BC_LOADS; ++i) {
        const long long at = (long long)min(first + bc_token + i * BC_TOKENS, t1 - 1) * ldbc + bc_col;
        held_b[i] = bmat[at];
        held_c[i] = cmat[at];
      }
      const long long t = min(first + ch_token, t1 - 1);
      held_x[0] = x[t * C + ch_col];
      held_dt[0] = dt[t * lddt + ch_col];
      held_z[0] = z[t * ldz + ch_col];
    } else {
      const bool whole = first + BLOCK <= t1;
      const float *bs = bmat + first * ldbc + bc_col, *cs = cmat + first * ldbc + bc_col;
      const float *xs = x + (long long)first * C + ch_col, *dts = dt + first * lddt + ch_col, *zs = z + first * ldz + ch_col;
      const int last = t1 - 1 - first;
#pragma unroll
      for (int i = 0; i < BC_LOADS; ++i) {
        if (HALVES == 2 && i > 0 && last < 16) break;      // nobody reads what would be there
        const int j = bc_token + i * BC_TOKENS, at = (whole ? j : min(j, last)) * (int)ldbc;
        held_b[i] = bs[at];
        held_c[i] = cs[at];
      }
#pragma unroll
      for (int i = 0; i < HALVES; ++i) {
        if (i > 0 && last < 16) break;
        const int j = ch_token + i * 16, at = whole ? j : min(j, last);
        held_x[i] = xs[at * C];
        held_dt[i] = dts[at * (int)lddt];
        held_z[i] = zs[at * (int)ldz];
      }
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < BC_LOADS; ++i) {
      bc[buf][0][state_of][bc_token + i * BC_TOKENS] = held_b[i];
      bc[buf][1][state_of][bc_token + i * BC_TOKENS] = held_c[i];
    }
#pragma unroll
    for (int i = 0; i < HALVES; ++i) {
      xdz[buf][0][tid % 16][ch_token + i * 16] = held_x[i];
      xdz[buf][1][tid % 16][ch_token + i * 16] = held_dt[i];
      xdz[buf][2][tid % 16][ch_token + i * 16] = held_z[i];
    }
  };
  const RowMerge merge(lane);
  fetch(t0);
  stage(0);
  __syncthreads();
  int buf = 0;
  for (int tb = t0; tb < t1; tb += BLOCK, buf ^= 1) {
    const bool more = tb + BLOCK < t1;
    if (more) fetch(tb + BLOCK);
    float sums[HALVES] = {};
    const int count = min(BLOCK, t1 - tb);
    auto walk = [&](auto tokens) {      // the block's first ones
      constexpr int TOKENS = decltype(tokens)::value;
      float quads[4];
      f32x4 x4[2], dt4[2], b4[2][R], c4[2][R];     // four tokens at a time, the next four's reads before them
      auto read = [&](int j4, int to) {
        x4[to] = *(const f32x4*)&xdz[buf][0][mine][j4];
        dt4[to] = *(const f32x4*)&xdz[buf][1][mine][j4];
#pragma unroll
        for (int r = 0; r < R; ++r) {
          b4[to][r] = *(const f32x4*)&bc[buf][0][part * R + r][j4];
          c4[to][r] = *(const f32x4*)&bc[buf][1][part * R + r][j4];
        }
      };
      read(0, 0);
#pragma unroll
      for (int j4 = 0; j4 < TOKENS; j4 += 4) {
        const int now = j4 / 4 & 1;
        if (j4 + 4 < TOKENS) read(j4 + 4, now ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        // in phases, each of them over the four tokens, so that none of their chains is waited for alone
        float keep[4][R], add[4][R], sum[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
#pragma unroll
          for (int r = 0; r < R; ++r) {
            keep[j][r] = expf(dt4[now][j] * a[r]);
            add[j][r] = in[r] ? dt4[now][j] * x4[now][j] * b4[now][r][j] : 0.f;
          }
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          sum[j] = 0.f;
#pragma unroll
          for (int r = 0; r < R; ++r) {
            s[r] = fmaf(keep[j][r], s[r], add[j][r]);
            sum[j] = fmaf(s[r], in[r] ? c4[now][r][j] : 0.f, sum[j]);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        quads[j4 / 4 % 4] = merge.quads(sum[0], sum[1], sum[2], sum[3]);
        if (j4 % 16 == 12) sums[j4 / 16] = merge.rows(quads);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if (count == BLOCK) {
      walk(std::integral_constant<int, BLOCK>{});
    } else {
      const int walked = HALVES == 2 && count >= 16 ? 16 : 0;
      if (HALVES == 2 && walked) walk(std::integral_constant<int, 16>{});
      for (int j = walked; j < count; ++j) {
        const float step = xdz[buf][1][mine][j], dtx = step * xdz[buf][0][mine][j];
        float sum = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r) {
          s[r] = fmaf(expf(step * a[r]), s[r], in[r] ? dtx * bc[buf][0][part * R + r][j] : 0.f);
          sum = fmaf(s[r], in[r] ? bc[buf][1][part * R + r][j] : 0.f, sum);
        }
        sum = row16_sum(sum);
#pragma unroll
        for (int half = 0; half < HALVES; ++half) sums[half] = part + half * 16 == j ? sum : sums[half];
      }
    }
#pragma unroll
    for (int half = 0; half < HALVES; ++half) {
      const int j = part + half * 16;
      if (live && j < count)
        out[(long long)(tb + j) * C + ch] = from_float<TO>(fmaf(d, xdz[buf][0][mine][j], sums[half]) * xdz[buf][2][mine][j]);
    }
    if (more) stage(buf ^ 1);
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int r = 0; r < R; ++r) row[r] = s[r];
  }
}

// dt[t, c] <- softplus(dt[t, c] + dt_bias[c]) in place and gate[t, c] = silu(z[t, c]): what the scan of a prompt's
// portion would otherwise compute token behind token.  Grid (tokens, parts of 1,024 channels), four channels a thread: neighbours
// (VEC: rows in 16 bytes) or 256 apart.  Many numbers are bound by memory: 1,834 tokens of 4,096 channels take 26.1 us in fours, 28.4
// 256 apart and 32.2 a thread a number (scan_prepare_each_kernel).  Few numbers are bound by a thread's own chain, four
// exponentials and logarithms behind one another instead of one, and rows of few channels leave most of a workgroup idle: us, a thread
// a number, in fours and 256 apart, 333 tokens of 64 channels 2.8 / 4.9 / 2.8, 128 of 2,048 3.5 / 3.9 / 4.7, 333 of 1,000 4.1 / 4.7 / 5.5, 128 of 4,096
// 4.7 / 4.6 / 5.3, 4,096 of 256 7.2 / 7.2 / 6.6, 333 of 4,097 8.6 / - / 9.6, 1,834 of 4,097 31.9 / - / 28.6.
template <bool VEC>
__global__ __launch_bounds__(256) void scan_prepare_kernel(float* __restrict__ dt, long long lddt, const float* __restrict__ dt_bias,
                                                           const float* __restrict__ z, long long ldz, float* __restrict__ gate,
                                                           int C) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const long long t = blockIdx.x;
  float* step = dt + t * lddt;
  const float* from = z + t * ldz;
  float* to = gate + t * C;
  for (long long first = blockIdx.y * 1024LL; first < C; first += gridDim.y * 1024LL) {
    if constexpr (VEC) {
      const long long c = first + threadIdx.x * 4;
      if (c >= C) return;
      f32x4 d = *(const f32x4*)(step + c), g = *(const f32x4*)(from + c);
      const f32x4 bias = *(const f32x4*)(dt_bias + c);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d[i] = scan_softplus(d[i] + bias[i]);
        g[i] = scan_silu(g[i]);
      }
      *(f32x4*)(step + c) = d;
      *(f32x4*)(to + c) = g;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const long long c = first + i * 256 + threadIdx.x;
        if (c >= C) return;
        step[c] = scan_softplus(step[c] + dt_bias[c]);
        to[c] = scan_silu(from[c]);
      }
    }
  }
}

// The same, a thread a number; at most 2^32 - 256 of them, which is what a launch counts.
__global__ __launch_bounds__(256) void scan_prepare_each_kernel(float* __restrict__ dt, long long lddt, const float* __restrict__ dt_bias,
                                                                const float* __restrict__ z, long long ldz,
                                                                float* __restrict__ gate, int C, unsigned total) {
  const unsigned idx = blockIdx.x * 256u + threadIdx.x;
  if (idx >= total) return;
  const unsigned t = idx / (unsigned)C, c = idx - t * (unsigned)C;
  float* step = dt + t * lddt;
  const float d = step[c], bias = dt_bias[c], g = z[t * ldz + c];
  step[c] = scan_softplus(d + bias);
  gate[idx] = scan_silu(g);
}
constexpr int SCAN_ROW = 512;                                        // channels from which a row is worth a workgroup,
constexpr long long SCAN_FOURS = 1 << 19, SCAN_APART = 1 << 22;      // and numbers from which a thread takes four of it

extern "C" int vk_scan_prepare(float* dt, long long lddt, const float* dt_bias, const float* z, long long ldz,
                               float* gate, int num_tokens, int C, void* stream) {
  if (num_tokens <= 0) return 0;
  if (C < 1) return VK_BAD_ARGUMENT;
  const dim3 grid(num_tokens, (unsigned)min((C + 1023LL) / 1024, 65535LL));
  const bool vec = C % 4 == 0 && lddt % 4 == 0 && ldz % 4 == 0 &&
                   (((uintptr_t)dt | (uintptr_t)dt_bias | (uintptr_t)z | (uintptr_t)gate) & 15) == 0;
  const long long total = (long long)num_tokens * C;
  if ((C < SCAN_ROW || total < (vec ? SCAN_FOURS : SCAN_APART)) && total <= 0xffffff00ll)
    scan_prepare_each_kernel<<<(unsigned)((total + 255) / 256), 256, 0, (hipStream_t)stream>>>(dt, lddt, dt_bias, z, ldz, gate, C, (unsigned)total);
  else if (vec) scan_prepare_kernel<true><<<grid, 256, 0, (hipStream_t)stream>>>(dt, lddt, dt_bias, z, ldz, gate, C);
  else scan_prepare_kernel<false><<<grid, 256, 0, (hipStream_t)stream>>>(dt, lddt, dt_bias, z, ldz, gate, C);
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" long long vk_selective_scan_channel_floats(int states) { return 16LL * lanes_share(states); }

extern "C" int vk_selective_scan(const float* x, const float* dtraw, long long lddt, const float* dt_bias,
                                 const float* bmat, const float* cmat, long long ldbc, const float* a_log,
                                 const float* skip, const float* z, long long ldz, float* state,
                                 long long state_stride, const int* entry_start, const int* entry_first,
                                 const int* slots, int num_entries, int num_tokens, int C, int N, int prepared, void* out,
                                 int out_dtype, void* stream) {
  if (num_entries <= 0) return 0;
  if (C < 1 || N < 1) return VK_BAD_ARGUMENT;
  if (N > 256) return VK_UNSUPPORTED_SIZE;
  if (state_stride < (long long)C * vk_selective_scan_channel_floats(N)) return VK_BAD_ARGUMENT;
  dim3 grid(num_entries, (C + SCAN_CHANNELS - 1) / SCAN_CHANNELS);
  if (grid.y > 65535) return VK_UNSUPPORTED_SIZE;
  hipStream_t s = (hipStream_t)stream;
  const dim3 run_grid(num_entries, (C + 15) / 16);
  // the walk in blocks counts a block's numbers from its first token in 32 bits
  const bool long_blocks = num_tokens >= 32ll * num_entries;
  const bool runs = prepared && C < (1 << 26) && lddt < (1 << 26) && ldbc < (1 << 26) && ldz < (1 << 26);
#define VK_SS_RUN(RR, BLOCK, ALL, TO)                                                                                 \
  selective_run_kernel<RR, BLOCK, ALL, TO><<<run_grid, 256, 0, s>>>(x, dtraw, lddt, bmat, cmat, ldbc, a_log, skip, z, ldz, \
                                                                    state, state_stride, entry_start, entry_first, slots, \
                                                                    C, N, (TO*)out)
#define VK_SS(RR, TO)                                                                                               \
  if constexpr (RR <= 4) {                                                                                          \
    if (runs) {                                                                                                     \
      if (RR == 1 && long_blocks && N == 16) VK_SS_RUN(1, 32, true, TO);                                            \
      else if (RR == 1 && long_blocks) VK_SS_RUN(1, 32, false, TO);                                                 \
      else if (N == 16 * RR) VK_SS_RUN(RR, 16, true, TO);                                                           \
      else VK_SS_RUN(RR, 16, false, TO);                                                                            \
      break;                                                                                                        \
    }                                                                                                               \
  }                                                                                                                 \
  selective_scan_kernel<RR, TO><<<grid, SCAN_THREADS, 0, s>>>(x, dtraw, lddt, dt_bias, bmat, cmat, ldbc, a_log, skip, \
                                                              z, ldz, state, state_stride, entry_start, entry_first, \
                                                              slots, C, N, prepared, (TO*)out)
#define VK_SS_R(TO)                       \
  switch (lanes_share(N)) {               \
    case 1: VK_SS(1, TO); break;          \
    case 2: VK_SS(2, TO); break;          \
    case 4: VK_SS(4, TO); break;          \
    case 8: VK_SS(8, TO); break;          \
    default: VK_SS(16, TO); break;        \
  }
  if (out_dtype == DT_F32) { VK_SS_R(float) }
  else if (out_dtype == DT_BF16) { VK_SS_R(bf16_t) }
  else return VK_BAD_ARGUMENT;
#undef VK_SS_R
#undef VK_SS
#undef VK_SS_RUN
  VK_LAUNCH_CHECK();
  return 0;
}
