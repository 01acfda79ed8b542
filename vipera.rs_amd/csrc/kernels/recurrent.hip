// Recurrent mixers: linear-attention layers that carry a matrix of state per head from token to token.
//
// Everything that enters a recurrence is 32-bit: the state, decays, gates, unit norms.  A request's state is one
// row of a `[slots + 1, floats]` tensor; an entry that starts at position 0 treats its row as zeros, so a slot
// that is used again needs no clearing.  The tokens of a step lie flat, entry after entry; `entry_start[e]` is
// the first token of entry e, `entry_first_pos[e]` its position in the request, `slots[e]` the state row.
//
// The recurrence kernels keep a head's state matrix in registers, a column of it spread over four lanes, and walk an
// entry's tokens in order; a sum over the key channels has one fixed order, whatever else is in the launch.
#include "common.h"
#include "scan_parts.h"

__device__ __forceinline__ float silu_f(float z) { return z / (1.0f + expf(-z)); }
__device__ __forceinline__ float sigmoid_f(float z) { return 1.0f / (1.0f + expf(-z)); }
__device__ __forceinline__ float softplus_f(float z) { return z > 20.0f ? z : log1pf(expf(z)); }

// ---------------------------------------------------------------------------------------------
// Short causal convolution over time per channel, then silu; q and k heads made unit vectors; gates.
//   proj  [T, ldp] 32-bit: channels [q: kh*dim | k: kh*dim | v: heads*vdim] first, later columns are the caller's
//   conv  [C, taps] 32-bit, the last column is the current token's
//   state row: `(taps - 1) * C` floats from `conv_offset` on, the inputs of the last taps - 1 tokens, oldest first
//   ba    columns `b_col + h` and `a_col + h` of proj hold the projections for beta and the decay's step
// Outputs (32-bit): qkv [T, ldq >= C] (q unit * dim^-1/2, k unit, v), beta [T, heads], decay [T, heads] (a_col < 0:
// the decay is the caller's business, see channel_decay_kernel).
// Grid (tokens, segments): a segment is one q or k head (its unit norm needs the whole head) or up to 1,024 value
// channels.  No load sits behind a branch: where an input comes from (the step, the state, nowhere) picks an
// address, and the value is masked.
constexpr int PREP_SPAN = 1024;

__device__ __forceinline__ float conv_input(const float* __restrict__ proj, long long ldp, const float* __restrict__ old,
                                            int C, int taps, int t, int offset, bool fresh, int back, int c) {
  const bool in_step = back <= offset, in_state = !in_step && !fresh;
  const float* from = in_step ? proj + (long long)(t - back) * ldp + c
                              : in_state ? old + (long long)(taps - 1 - (back - offset)) * C + c : proj + (long long)t * ldp + c;
  const float x = *from;
  return (in_step || in_state) ? x : 0.f;
}

__global__ __launch_bounds__(256) void delta_prepare_kernel(
    const float* __restrict__ proj, long long ldp, const float* __restrict__ conv, int taps,
    const float* __restrict__ state, long long state_stride, long long conv_offset, const int* __restrict__ entry_of,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots,
    const float* __restrict__ a_log, const float* __restrict__ dt_bias, int kv_heads, int dim, int heads, int vdim,
    int b_col, int a_col, float unit_eps, float* __restrict__ qkv, long long ldq, float* __restrict__ beta,
    float* __restrict__ decay) {
  __shared__ float scratch[16];
  const int t = blockIdx.x, seg = blockIdx.y;
  const int e = entry_of[t];
  const int offset = t - entry_start[e];
  const bool fresh = entry_first[e] == 0;
  const int unit_heads = 2 * kv_heads;
  const int C = unit_heads * dim + heads * vdim;
  const float* old = state + (long long)slots[e] * state_stride + conv_offset;
  float* out = qkv + (long long)t * ldq;
  const bool unit = seg < unit_heads;
  const int first = unit ? seg * dim : unit_heads * dim + (seg - unit_heads) * PREP_SPAN;
  const int last = unit ? first + dim : min(C, first + PREP_SPAN);
  float kept[PREP_SPAN / 256];      // a segment is at most 1,024 channels: four to a thread
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < PREP_SPAN / 256; ++i) {
    const int c = first + threadIdx.x + i * 256;
    float y = 0.f;
    if (c < last) {
      float sum = 0.f;
      for (int j = 0; j < taps; ++j)
        sum = fmaf(conv[(long long)c * taps + j], conv_input(proj, ldp, old, C, taps, t, offset, fresh, taps - 1 - j, c), sum);
      y = silu_f(sum);
    }
    kept[i] = y;
    ss += y * y;
  }
  float scale = 1.f;
  if (unit) {       // the same for all threads of the workgroup
    ss = block_sum(ss, scratch);
    scale = 1.0f / sqrtf(ss + unit_eps);
    if (seg < kv_heads) scale *= 1.0f / sqrtf((float)dim);
  }
#pragma unroll
  for (int i = 0; i < PREP_SPAN / 256; ++i) {
    const int c = first + threadIdx.x + i * 256;
    if (c < last) out[c] = kept[i] * scale;
  }
  if (seg == 0)
    for (int h = threadIdx.x; h < heads; h += blockDim.x) {
      const float* p = proj + (long long)t * ldp;
      beta[(long long)t * heads + h] = sigmoid_f(p[b_col + h]);
      if (a_col >= 0) decay[(long long)t * heads + h] = expf(-expf(a_log[h]) * softplus_f(p[a_col + h] + dt_bias[h]));
    }
}

// The same for prompts' portions, every number formed as above: a thread per channel and PREP_RUN consecutive tokens of the
// step, whose rows it asks for at once; the heads' sums of squares meet in LDS, a token's wave by wave as block_sum adds
// them.  Above, a workgroup of one token and 128 channels of its head leaves half its threads idle and waits for entry, taps and
// inputs one behind another, a few microseconds for a kilobyte.  dim: 64, 128 or 256, so that a head lies in one workgroup.
// us with the state's rows after it, 4,096 channels of four taps, before and so: 2,048 tokens 74.0 / 26.3 (their rows' way from
// and to memory takes some 15), 512 25.4 / 10.8, 128 9.9 / 7.9.  Runs of 8: 25.4, 11.6 and 10.4; of 16: 24.5, 16.1 and 15.3.
// A run's own chain is longer than a token's: it is taken where the workgroups above are more than the chip holds at once, or where
// they walk 1,024 channels of values in four turns.  us, a token and a run a thread, one entry: 128 tokens of 2 key heads of 64 and 256
// channels of values (640 workgroups) 6.6 / 8.0, of 4 of 128 and 512 (1,152) 7.5 / 8.2, of 4 of 128 and 1,024 (1,152) 9.8 / 8.2; 800 of 1 of
// 128 and 66 (2,400) 6.9 / 7.4, 512 of 2 of 64 and 256 (2,560) 7.9 / 8.1, 300 of 4 of 128 and 512 (2,700) 9.5 / 8.4, 800 of 2 of 64 and 256
// (4,000) 9.5 / 8.0.
constexpr int PREP_RUN = 4, PREP_RUN_TOKENS = 128;
constexpr long long PREP_RUN_BLOCKS = 2600;
template <int TAPS>
__global__ __launch_bounds__(256) void delta_prepare_run_kernel(
    const float* __restrict__ proj, long long ldp, const float* __restrict__ conv, const float* __restrict__ state,
    long long state_stride, long long conv_offset, const int* __restrict__ entry_of, const int* __restrict__ entry_start,
    const int* __restrict__ entry_first, const int* __restrict__ slots, const float* __restrict__ a_log,
    const float* __restrict__ dt_bias, int kv_heads, int dim, int heads, int vdim, int b_col, int a_col, float unit_eps,
    float* __restrict__ qkv, long long ldq, float* __restrict__ beta, float* __restrict__ decay, int num_tokens) {
  __shared__ float squares[PREP_RUN][4];
  const int t0 = blockIdx.x * PREP_RUN, tokens = min(PREP_RUN, num_tokens - t0);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int unit_channels = 2 * kv_heads * dim, C = unit_channels + heads * vdim;
  const int first = blockIdx.y * 256, c = first + threadIdx.x, from = min(c, C - 1);
  const bool unit = first + wave * 64 < unit_channels;      // heads begin at multiples of 64
  float w[TAPS], in[PREP_RUN + TAPS - 1], y[PREP_RUN];
#pragma unroll
  for (int i = 0; i < PREP_RUN + TAPS - 1; ++i)
    in[i] = proj[(long long)min(max(t0 + i - (TAPS - 1), 0), num_tokens - 1) * ldp + from];
#pragma unroll
  for (int i = 0; i < TAPS; ++i) w[i] = conv[(long long)from * TAPS + i];
#pragma unroll
  for (int j = 0; j < PREP_RUN; ++j) {
    const int t = min(t0 + j, num_tokens - 1), e = entry_of[t], offset = t - entry_start[e];
    float sum = 0.f;
    if (offset >= TAPS - 1) {
#pragma unroll
      for (int i = 0; i < TAPS; ++i) sum = fmaf(w[i], in[j + i], sum);
    } else {       // the entry's first tokens: what came before them is the state, or nothing
      const bool fresh = entry_first[e] == 0;
      const float* old = state + (long long)slots[e] * state_stride + conv_offset + from;
#pragma unroll
      for (int i = 0; i < TAPS; ++i) {
        const int before = TAPS - 1 - i - offset;      // tokens before the entry's first
        sum = fmaf(w[i], before <= 0 ? in[j + i] : fresh ? 0.f : old[(long long)(TAPS - 1 - before) * C], sum);
      }
    }
    y[j] = silu_f(sum);
  }
  if (unit) {
#pragma unroll
    for (int j = 0; j < PREP_RUN; ++j) {
      const float sum = wave_sum(fmaf(y[j], y[j], 0.f));      // a square of its own, not a term of the first addition
      if ((threadIdx.x & 63) == 0) squares[j][wave] = sum;
    }
  }
  __syncthreads();
  const int head_waves = dim / 64, head_wave = unit ? wave / head_waves * head_waves : 0;
#pragma unroll
  for (int j = 0; j < PREP_RUN; ++j) {
    float scale = 1.f;
    if (unit) {
      float total = 0.f;
      for (int i = 0; i < head_waves; ++i) total += squares[j][head_wave + i];
      scale = 1.0f / sqrtf(total + unit_eps);
      if (first + wave * 64 < kv_heads * dim) scale *= 1.0f / sqrtf((float)dim);
    }
    if (j < tokens && c < C) qkv[(long long)(t0 + j) * ldq + c] = y[j] * scale;
  }
  if (blockIdx.y == 0)
    for (int i = threadIdx.x; i < tokens * heads; i += 256) {
      const int t = t0 + i / heads, h = i % heads;
      const float* p = proj + (long long)t * ldp;
      beta[(long long)t * heads + h] = sigmoid_f(p[b_col + h]);
      if (a_col >= 0) decay[(long long)t * heads + h] = expf(-expf(a_log[h]) * softplus_f(p[a_col + h] + dt_bias[h]));
    }
}

// The convolution's inputs of an entry's last taps - 1 tokens become the state.  Grid (entries, ceil(C / 256)), a
// thread per channel; runs after delta_prepare has read the old rows.
__global__ __launch_bounds__(256) void conv_state_kernel(const float* __restrict__ proj, long long ldp, int taps, int C,
                                                         float* __restrict__ state, long long state_stride,
                                                         long long conv_offset, const int* __restrict__ entry_start,
                                                         const int* __restrict__ entry_first,
                                                         const int* __restrict__ slots) {
  const int e = blockIdx.x;
  const int c = blockIdx.y * 256 + threadIdx.x;
  if (c >= C) return;
  const int start = entry_start[e], count = entry_start[e + 1] - start;
  const bool fresh = entry_first[e] == 0;
  float* rows = state + (long long)slots[e] * state_stride + conv_offset;
  const int keep = taps - 1;
  for (int j = 0; j < keep; ++j) {           // ascending: row j + count is read before it is written
    const int from = j + count;              // index into [old rows (keep) | the entry's tokens (count)]
    const bool in_step = from >= keep;
    const float* source = in_step ? proj + (long long)(start + from - keep) * ldp + c : rows + (long long)from * C + c;
    const float x = *source;
    rows[(long long)j * C + c] = (in_step || !fresh) ? x : 0.f;
  }
}

// ---------------------------------------------------------------------------------------------
// The two recurrences share their shape.  A workgroup of four waves owns 16 value channels of one (entry, head), a
// wave four of them; the sixteen lanes of a row of the wave share one value channel and each keeps R of its key
// channels in registers (16 R >= dim; rows past dim stay zero).  A sum over the key channels is R terms in a lane, in
// ascending order, then four exchanges inside the 16-lane row (DPP, no LDS).  The entry's tokens are walked in
// blocks of 16: a block's k, q (or r, k, decay), values and gates are fetched into registers while the block before
// is worked on, and passed on through LDS, so that a token's step waits for no memory.
//
// This form runs the steps of single tokens (BLOCK 1: few registers, many waves a SIMD); prompts' portions run on
// the scan kernels further down, a wave to a value channel.
//
// The state of a head lies in memory as [value channel, padded to 16][key channel, padded to 16 R]: a lane's R
// numbers are contiguous, a row's sixteen lanes hold one value channel's run, and a workgroup reads and writes one
// contiguous run.  Both forms read it; nobody else does.
constexpr int REC_BLOCK = 16;    // tokens per LDS block; 1 for steps of single tokens (few registers, many waves a SIMD)
constexpr int REC_COLS = 16;     // value channels per workgroup

template <int CTRL>
__device__ __forceinline__ float dpp_add(float v) {
  const int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xF, 0xF, false);
  return v + __int_as_float(moved);
}

// Lane l of a row of 16 gets the value of lane l - N of its row, or `edge` where the row has no such lane.
template <int N>
__device__ __forceinline__ float row_shifted(float v, float edge) {
  return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(edge), __float_as_int(v), 0x110 + N, 0xF, 0xF, false));
}

// The sum over the 16 lanes of a row, in every lane: neighbours, pairs of neighbours, the halves of eight, the eights.
__device__ __forceinline__ float row_sum16(float v) {
  v = dpp_add<0xB1>(v);     // quad_perm [1, 0, 3, 2]
  v = dpp_add<0x4E>(v);     // quad_perm [2, 3, 0, 1]
  v = dpp_add<0x141>(v);    // row_half_mirror: the other quad of the eight
  v = dpp_add<0x140>(v);    // row_mirror: the other eight
  return v;
}

// Gated delta rule.  Per head, with S [dim, vdim]:  S <- g S;  u = beta (v - S^T k);  S <- S + k u^T;  o = S^T q.
// Grid (entries, heads, ceil(vdim / 16)).  An LDS row of a token: [q: 16R | k: 16R | (CH: g: 16R) | v: 16 | beta, decay].
// CH: one decay per head and key channel, which scales that row of S; it lies in the token's qkv row from column
// g_col on, [heads, dim].  `ldq` is the row stride of qkv.
template <int R, int BLOCK, bool CH>
__global__ __launch_bounds__(256) void delta_rule_kernel(
    const float* __restrict__ qkv, long long ldq, int g_col, const float* __restrict__ beta,
    const float* __restrict__ decay, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots,
    int kv_heads, int dim, int heads, int vdim, float* __restrict__ out) {
  constexpr int DP = 16 * R, VOFF = (CH ? 3 : 2) * DP, ROW = VOFF + REC_COLS + 2, COUNT = BLOCK * ROW;
  constexpr int LOADS = (COUNT + 255) / 256;
  __shared__ float rows[COUNT];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = lane & 15, d0 = grp * R;
  const int v0 = blockIdx.z * REC_COLS, mine_col = wave * 4 + (lane >> 4), v = v0 + mine_col;
  const bool live = v < vdim;
  const int kh = h / (heads / kv_heads);
  const int start = entry_start[e], end = entry_start[e + 1];
  float* mine = state + (long long)slots[e] * state_stride + (((long long)h * gridDim.z * REC_COLS + v) * 16 + grp) * R;
  const bool fresh = entry_first[e] == 0;
  float S[R];
#pragma unroll
  for (int i = 0; i < R; ++i) S[i] = fresh ? 0.f : mine[i];
  // what this thread fetches of a block: element x of the block is token x / ROW, column x % ROW
  float held[LOADS];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int x = tid + i * 256, j = x / ROW, col = x % ROW, t = t0 + j;
      // one load per element and no branch around it (a load inside a branch would be waited for there, and a
      // block's loads would arrive one after the other): the address is chosen by selects, a clamped one where
      // the element does not exist, and the value is masked afterwards
      const bool is_q = col < DP, is_k = !is_q && col < 2 * DP, is_g = CH && !is_q && !is_k && col < VOFF;
      const bool is_v = col >= VOFF && col < VOFF + REC_COLS;
      const bool is_b = col == VOFF + REC_COLS;
      const int d = is_q ? col : is_k ? col - DP : col - 2 * DP, c = col - VOFF;
      const bool ok = x < COUNT && t < end && (is_q || is_k || is_g ? d < dim : is_v ? v0 + c < vdim : (is_b || !CH));
      const long long tt = ok ? t : start;
      const float* base = (is_q || is_k || is_g || is_v) ? qkv + tt * ldq : ((is_b || CH) ? beta : decay) + tt * heads + h;
      const int within = is_q ? kh * dim + d : is_k ? (kv_heads + kh) * dim + d : is_g ? g_col + h * dim + d
                         : is_v ? 2 * kv_heads * dim + h * vdim + v0 + c : 0;
      const float loaded = base[ok ? within : 0];
      const float value = ok ? loaded : 0.f;
      held[i] = value;
    }
  };
  fetch(start);
  for (int t0 = start; t0 < end; t0 += BLOCK) {
    __syncthreads();     // the block before has been read
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if (tid + i * 256 < COUNT) rows[tid + i * 256] = held[i];
    __syncthreads();
    if (t0 + BLOCK < end) fetch(t0 + BLOCK);
    const int count = min(BLOCK, end - t0);
    // a token's numbers are read from LDS while the token before it is worked on
    float kk[R], qq[R], gg[CH ? R : 1], b, g, val;
    auto read = [&](int j) {
      const float* row = rows + j * ROW;
      b = row[VOFF + REC_COLS], g = row[VOFF + REC_COLS + 1], val = row[VOFF + mine_col];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        kk[i] = row[DP + d0 + i];
        qq[i] = row[d0 + i];
        if (CH) gg[i] = row[2 * DP + d0 + i];
      }
    };
    read(0);
    for (int j = 0; j < count; ++j) {
      float k_now[R], q_now[R], g_rows[CH ? R : 1];
      const float b_now = b, g_now = g, val_now = val;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        k_now[i] = kk[i];
        q_now[i] = qq[i];
        if (CH) g_rows[i] = gg[i];
      }
      if (j + 1 < count) read(j + 1);
      float dot[2] = {0.f, 0.f};     // two chains, even and odd rows, added at the end: a fixed order
#pragma unroll
      for (int i = 0; i < R; ++i) {
        S[i] *= CH ? g_rows[i] : g_now;
        dot[i & 1] = fmaf(S[i], k_now[i], dot[i & 1]);
      }
      const float u = b_now * (val_now - row_sum16(dot[0] + dot[1]));
      float o[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < R; ++i) {
        S[i] = fmaf(k_now[i], u, S[i]);
        o[i & 1] = fmaf(S[i], q_now[i], o[i & 1]);
      }
      const float sum = row_sum16(o[0] + o[1]);
      if (live && grp == 0) out[((long long)(t0 + j) * heads + h) * vdim + v] = sum;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) mine[i] = S[i];
}

// RWKV-style time mixing.  Per head, with S [dim, dim]:  o = (S + diag(u) k v^T)^T r;  S <- diag(w) S + k v^T,
// w = exp(-exp(wraw + w0)) per key channel.  r, k, v, wraw are 32-bit [T, heads * dim] with row strides of their own.
// Grid (entries, heads, ceil(dim / 16)).  An LDS row of a token: [r: 16R | k: 16R | w: 16R | v: 16].
template <int R, int BLOCK>
__global__ __launch_bounds__(256) void wkv_rule_kernel(
    const float* __restrict__ r, long long ldr, const float* __restrict__ k, long long ldk, const float* __restrict__ v,
    long long ldv, const float* __restrict__ wraw, long long ldw, const float* __restrict__ w0,
    const float* __restrict__ bonus, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int dim,
    int heads, int decayed, float* __restrict__ out) {
  constexpr int DP = 16 * R, ROW = 3 * DP + REC_COLS, COUNT = BLOCK * ROW, LOADS = (COUNT + 255) / 256;
  __shared__ float rows[COUNT];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = lane & 15, d0 = grp * R;
  const int v0 = blockIdx.z * REC_COLS, mine_col = wave * 4 + (lane >> 4), col_v = v0 + mine_col;
  const bool live = col_v < dim;
  const int start = entry_start[e], end = entry_start[e + 1];
  float* mine = state + (long long)slots[e] * state_stride + (((long long)h * gridDim.z * REC_COLS + col_v) * 16 + grp) * R;
  const bool fresh = entry_first[e] == 0;
  float S[R], U[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    S[i] = fresh ? 0.f : mine[i];
    U[i] = d0 + i < dim ? bonus[h * dim + d0 + i] : 0.f;
  }
  float held[LOADS];
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int x = tid + i * 256, j = x / ROW, col = x % ROW, t = t0 + j;
      // branch-free, as in the delta rule's kernel: selected addresses, one load each, masked values
      const bool is_r = col < DP, is_k = !is_r && col < 2 * DP, is_w = !is_r && !is_k && col < 3 * DP;
      const int d = is_r ? col : is_k ? col - DP : col - 2 * DP, c = col - 3 * DP;
      const bool ok = x < COUNT && t < end && (is_r || is_k || is_w ? d < dim : v0 + c < dim);
      const long long tt = ok ? t : start;
      const float* base = is_r ? r + tt * ldr : is_k ? k + tt * ldk : is_w ? wraw + tt * ldw : v + tt * ldv;
      const int within = ok ? h * dim + ((is_r || is_k || is_w) ? d : v0 + c) : 0;
      const float loaded = base[within];
      const float shift = w0[(ok && is_w) ? h * dim + d : 0];
      const float value = !ok ? 0.f : (is_w && !decayed) ? expf(-expf(loaded + shift)) : loaded;
      held[i] = value;
    }
  };
  fetch(start);
  for (int t0 = start; t0 < end; t0 += BLOCK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if (tid + i * 256 < COUNT) rows[tid + i * 256] = held[i];
    __syncthreads();
    if (t0 + BLOCK < end) fetch(t0 + BLOCK);
    const int count = min(BLOCK, end - t0);
    float rr[R], kk[R], ww[R], val;
    auto read = [&](int j) {
      const float* row = rows + j * ROW;
      val = row[3 * DP + mine_col];
#pragma unroll
      for (int i = 0; i < R; ++i) {
        rr[i] = row[d0 + i];
        kk[i] = row[DP + d0 + i];
        ww[i] = row[2 * DP + d0 + i];
      }
    };
    read(0);
    for (int j = 0; j < count; ++j) {
      float r_now[R], k_now[R], w_now[R];
      const float val_now = val;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        r_now[i] = rr[i];
        k_now[i] = kk[i];
        w_now[i] = ww[i];
      }
      if (j + 1 < count) read(j + 1);
      float o[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float kv = k_now[i] * val_now;
        o[i & 1] = fmaf(fmaf(U[i], kv, S[i]), r_now[i], o[i & 1]);
        S[i] = fmaf(w_now[i], S[i], kv);
      }
      const float sum = row_sum16(o[0] + o[1]);
      if (live && grp == 0) out[((long long)(t0 + j) * heads + h) * dim + col_v] = sum;
    }
  }
#pragma unroll
  for (int i = 0; i < R; ++i) mine[i] = S[i];
}

// ---------------------------------------------------------------------------------------------
// The same recurrences for prompts' portions: a wave owns ONE value channel and its 64 lanes the key channels, Q of
// them each (64 Q >= the state's padded key width), so that one prompt of a few thousand tokens is heads x value
// channels waves, two or more to a SIMD, each with a short step per token: Q terms a lane, four DPP exchanges inside
// the rows, and the four rows' sums read by every lane.  A workgroup is eight waves (eight value channels) that share a
// block's k, q (r, k, decay) in LDS.  A whole block is unrolled without a branch, with a token's (four tokens') LDS reads
// before the arithmetic of the token (four) before it, so that only the recurrence itself is waited for: the delta rule's
// dot product, six exchanges and update, about 130 ns a token at two waves a SIMD; the time mixing has one FMA a token
// there and its vector instructions and LDS reads bound it.  With a loop of one branch a token, reads right before their
// use and a number's address worked out by its thread: delta rule, 16 heads of 128 x 128, 2,048 tokens 400 -> 262 us,
// portions of 1,000 and 834 314 -> 213 us, with a decay per key channel 422 -> 280 and 333 -> 226 us; time mixing, 32
// heads of 64, 292 -> 157 and 197 -> 114 us.
constexpr int SCAN_COLS = 8;
constexpr int SCAN_THREADS = SCAN_COLS * 64;

// (row 0 + row 1) + (row 2 + row 3), to every lane, of a number that is the same in a row's lanes: row 0's joins row 1's
// and row 2's row 3's, then the first two row 3, whose last lane everybody reads.
__device__ __forceinline__ float rows_total(float v) {
  v = dpp_add<0x143>(dpp_add<0x142>(v));
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ float wave_total(float v) { return rows_total(row_sum16(v)); }

// row 0 + row 1 to the lanes of both, row 2 + row 3 to theirs.
__device__ __forceinline__ float pair_total(float v) {
  const unsigned bits = (unsigned)__float_as_int(v);
  const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
  return __int_as_float((int)rows[0]) + __int_as_float((int)rows[1]);
}

// How a block gets into LDS: a wave takes whole pieces of sixty-four numbers of one token and one kind (k, q, ...), so
// that where a piece begins is worked out by the scalar unit and a lane only adds its own number; the sixteen tokens'
// eight values are 128 threads'.  A fetch only issues loads, the same number in every thread and none inside a
// branch, from addresses that exist whatever the block holds: the entry's last token stands in for tokens past its end,
// which are never worked on, and a channel past the last is the last one, stored as zero.  A loaded number is first used
// when it is stored into LDS, a block later, so that nothing waits for memory before the block in between has been
// worked on.  (Every thread working out its own numbers' addresses took a third of the walk's vector instructions.)
template <int Q, bool CH>
__global__ __launch_bounds__(SCAN_THREADS) void delta_scan_kernel(
    const float* __restrict__ qkv, long long ldq, int g_col, const float* __restrict__ beta,
    const float* __restrict__ decay, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots,
    int kv_heads, int dim, int heads, int vdim, int key_pad, int value_pad, float* __restrict__ out) {
  constexpr int DP = 64 * Q, KINDS = CH ? 3 : 2, VOFF = KINDS * DP, ROW = VOFF + SCAN_COLS;
  constexpr int TOKENS = REC_BLOCK / SCAN_COLS, PIECES = TOKENS * KINDS * Q;     // a wave's tokens of a block, and their pieces
  __shared__ float rows[REC_BLOCK * ROW];
  __shared__ float gates[REC_BLOCK][2];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d0 = lane * Q;
  const int v0 = blockIdx.z * SCAN_COLS, v = v0 + wave;
  const bool live = v < vdim;
  const int kh = h / (heads / kv_heads);
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* mine = state + (long long)slots[e] * state_stride + ((long long)h * value_pad + v) * key_pad + d0;
  const bool fresh = entry_first[e] == 0, kept = v < value_pad;
  float S[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) S[i] = (!fresh && kept && d0 + i < key_pad) ? mine[i] : 0.f;
  int from[Q];        // the lane's number of a piece in each part of a row of key channels
#pragma unroll
  for (int c = 0; c < Q; ++c) from[c] = min(c * 64 + lane, dim - 1);
  const int value_j = tid / SCAN_COLS & (REC_BLOCK - 1), value_col = min(v0 + tid % SCAN_COLS, vdim - 1);
  const float* values = qkv + 2 * kv_heads * dim + h * vdim + value_col;
  float held[PIECES], held_value, held_gate;
  const float* gate_src = ((tid & 1) && !CH ? decay : beta) + h;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int j = wave * TOKENS + i / (KINDS * Q), kind = i / Q % KINDS;
      const int col = kind == 0 ? kh * dim : kind == 1 ? (kv_heads + kh) * dim : g_col + h * dim;
      held[i] = (qkv + (long long)min(t0 + j, end - 1) * ldq + col)[from[i % Q]];
    }
    held_value = values[(long long)min(t0 + value_j, end - 1) * ldq];
    held_gate = gate_src[(long long)min(t0 + ((tid >> 1) & (REC_BLOCK - 1)), end - 1) * heads];
  };
  fetch(start);
  for (int t0 = start; t0 < end; t0 += REC_BLOCK) {
    __syncthreads();     // the block before has been read
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int j = wave * TOKENS + i / (KINDS * Q), kind = i / Q % KINDS;
      rows[j * ROW + kind * DP + i % Q * 64 + lane] = i % Q * 64 + lane < dim ? held[i] : 0.f;
    }
    if (tid < REC_BLOCK * SCAN_COLS) rows[value_j * ROW + VOFF + tid % SCAN_COLS] = v0 + tid % SCAN_COLS < vdim ? held_value : 0.f;
    if (tid < 2 * REC_BLOCK) gates[tid >> 1][tid & 1] = held_gate;
    __syncthreads();
    fetch(min(t0 + REC_BLOCK, end - 1));
    const int count = min(REC_BLOCK, end - t0);
    float outs = 0.f;      // lane j of every row: its row's part of token j's read-out, which nothing waits for
    auto read = [&](int j, float (&kk)[Q], float (&qq)[Q], float (&gg)[Q], float& b, float& val) {
      const float* row = rows + j * ROW;
      b = gates[j][0];
      val = row[VOFF + wave];
      const float g = gates[j][1];
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        kk[i] = row[DP + d0 + i];
        qq[i] = row[d0 + i];
        gg[i] = CH ? row[2 * DP + d0 + i] : g;
      }
    };
    // token j's update, with the read-out of the token before from the same state beside it: the update's chain (a dot
    // product, six exchanges, a lane's sum to all) is what a token costs, and the read-out's lies in its gaps
    auto token = [&](int j, const float (&kk)[Q], const float (&gg)[Q], float b, float val, const float (&before)[Q]) {
      float dot = 0.f, o = 0.f;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        o = fmaf(S[i], before[i], o);
        S[i] *= gg[i];
        dot = fmaf(S[i], kk[i], dot);
      }
      // the two sums' exchanges in turn: between two of one chain the chip would have to wait
#define VK_STEP(CTRL)                 \
  dot = dpp_add<CTRL>(dot);           \
  if (j) o = dpp_add<CTRL>(o);        \
  __builtin_amdgcn_sched_barrier(0);
      VK_STEP(0xB1)
      VK_STEP(0x4E)
      VK_STEP(0x141)
      VK_STEP(0x140)
#undef VK_STEP
      const float u = b * (val - rows_total(dot));
#pragma unroll
      for (int i = 0; i < Q; ++i) S[i] = fmaf(kk[i], u, S[i]);
      if (j) outs = (lane & (REC_BLOCK - 1)) == j - 1 ? o : outs;
    };
    auto read_out = [&](int j, const float (&qq)[Q]) {
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < Q; ++i) o = fmaf(S[i], qq[i], o);
      o = row_sum16(o);
      outs = (lane & (REC_BLOCK - 1)) == j ? o : outs;
    };
    float kk[2][Q], qq[3][Q], gg[2][Q], b[2], val[2];
    if (count == REC_BLOCK) {      // a token's LDS reads go before the arithmetic of the token before it
      read(0, kk[0], qq[0], gg[0], b[0], val[0]);
#pragma unroll
      for (int j = 0; j < REC_BLOCK; ++j) {
        const int now = j & 1, next = now ^ 1;
        if (j + 1 < REC_BLOCK) read(j + 1, kk[next], qq[(j + 1) % 3], gg[next], b[next], val[next]);
        __builtin_amdgcn_sched_barrier(0);
        token(j, kk[now], gg[now], b[now], val[now], qq[(j + 2) % 3]);
        __builtin_amdgcn_sched_barrier(0);
      }
      read_out(REC_BLOCK - 1, qq[(REC_BLOCK - 1) % 3]);
    } else {
      for (int j = 0; j < count; ++j) {
        read(j, kk[0], qq[0], gg[0], b[0], val[0]);
        token(0, kk[0], gg[0], b[0], val[0], qq[0]);
        read_out(j, qq[0]);
      }
    }
    outs += __shfl_xor(outs, 16, 64);     // (row 0 + row 1) + (row 2 + row 3), in every row
    outs += __shfl_xor(outs, 32, 64);
    if (live && lane < count) out[((long long)(t0 + lane) * heads + h) * vdim + v] = outs;
  }
  if (kept) {
#pragma unroll
    for (int i = 0; i < Q; ++i)
      if (d0 + i < key_pad) mine[i] = S[i];
  }
}

// The delta rule for key widths up to 128 in whole pieces of 16 bytes, with every number formed as above: a value channel
// has 32 lanes, each with the key channels of two of the 64 lanes above, and adds the two's parts itself where they would have
// met first.  What bounds the walk is a wave's instructions: one goes out every 1.95 ns on a wave alone on its SIMD and little
// faster on two, so that a token's step is worth what its instructions take (some 39 here for two value channels, 36 above for
// one), and what a block costs besides is worth its share of sixteen tokens: here a block goes straight from memory into LDS in
// pieces of 16 bytes, whose places are worked out once, and LDS reads and the read-out's products stand between the exchanges
// of the update's sum, which would wait there.  us, above and here, launches behind one another in a graph: 16 heads of 128 x 128, one entry of
// 2,048 tokens 259 / 200, of 512 67 / 53, of 1,000 and 834 194 / 135, eight of 250 169 / 114, of 31 8.1 / 7.4; 8 heads, 2,048 tokens 255 / 196; 6 heads of
// 64 x 64, 512, 456 and 399 59 / 46; with a decay per key channel, 16 heads 277 / 209.
template <int Q, bool CH>
__global__ __launch_bounds__(SCAN_COLS * 32) void delta_scan_direct_kernel(
    const float* __restrict__ qkv, long long ldq, int g_col, const float* __restrict__ beta,
    const float* __restrict__ decay, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots,
    int kv_heads, int dim, int heads, int vdim, int key_pad, int value_pad, float* __restrict__ out) {
  constexpr int DP = 64 * Q, KINDS = CH ? 3 : 2, N = 2 * Q, WAVES = SCAN_COLS / 2;
  constexpr int PIECES = KINDS * 4 * Q / WAVES, ROWS = 4 / Q;      // a wave's loads of a block (64 pieces of 16 bytes), rows each
  static_assert(WAVES == 4, "two waves fetch the values, one beta, one the decay");
  __shared__ __attribute__((aligned(16))) float rows[2][KINDS][REC_BLOCK][DP];
  __shared__ float values[2][REC_BLOCK][SCAN_COLS];
  __shared__ float gates[2][2][REC_BLOCK];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = tid >> 5, d0 = (lane & 31) * N;
  const int v0 = blockIdx.z * SCAN_COLS, v = v0 + col;
  const bool live = v < vdim;
  const int kh = h / (heads / kv_heads);
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* mine = state + (long long)slots[e] * state_stride + ((long long)h * value_pad + v) * key_pad + d0;
  const bool fresh = entry_first[e] == 0, kept = v < value_pad;
  float S[N];
#pragma unroll
  for (int i = 0; i < N; ++i) S[i] = (!fresh && kept && d0 + i < key_pad) ? mine[i] : 0.f;
  const int row_bytes = (int)ldq * 4;
  int piece_row[PIECES], piece_at[PIECES], piece_off[PIECES];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) {
    const int n = wave * PIECES + i, kind = n / (4 * Q), c = lane % (16 * Q) * 4;
    piece_row[i] = n % (4 * Q) * ROWS + lane / (16 * Q);
    piece_at[i] = c < dim ? ((kind == 0 ? kh * dim : kind == 1 ? (kv_heads + kh) * dim : g_col + h * dim) + c) * 4 : -1;
    piece_off[i] = c < dim ? piece_row[i] * row_bytes + piece_at[i] : -1;
  }
  // the wave's single numbers: values (waves 0 and 1, a row's eight side by side), beta (2) and the decay (3)
  const bool a_value = wave < 2, single = a_value || (lane < REC_BLOCK && !(CH && wave == 3));
  const float* single_from = a_value ? qkv : wave == 2 ? beta : decay;
  const int single_row = a_value ? tid >> 3 : lane, single_bytes = a_value ? row_bytes : heads * 4;
  const int single_at = !a_value ? h * 4 : v0 + (tid & 7) < vdim ? (2 * kv_heads * dim + h * vdim + v0 + (tid & 7)) * 4 : -1;
  const int single_off = single_at < 0 ? -1 : single_row * single_bytes + single_at;
  float* const single_to = a_value ? &values[0][0][0] + wave * 64 : &gates[0][0][0] + (wave - 2) * REC_BLOCK;
  const int single_next = a_value ? REC_BLOCK * SCAN_COLS : 2 * REC_BLOCK;
  // a row past the entry's end is its last one, which nobody works on; what does not exist (-1) reads zeros
  const float *next_row = qkv + start * ldq, *next_single = single_from + (long long)start * (single_bytes / 4);     // of the block fetched next
  auto fetch = [&](int t0, int buf) {
    const ScanView view = scan_view(next_row, 0x7fffffff), single_view = scan_view(next_single, 0x7fffffff);
    float* to = &rows[buf][0][0][0] + wave * PIECES * 256;
    if (t0 + REC_BLOCK <= end) {
#pragma unroll
      for (int i = 0; i < PIECES; ++i) scan_load_lds<true>(view, to + i * 256, piece_off[i]);
      if (single) scan_load_lds<false>(single_view, single_to + buf * single_next, single_off);
    } else {
      const int last = end - 1 - t0;
#pragma unroll
      for (int i = 0; i < PIECES; ++i)
        scan_load_lds<true>(view, to + i * 256, piece_at[i] < 0 ? -1 : min(piece_row[i], last) * row_bytes + piece_at[i]);
      if (single)
        scan_load_lds<false>(single_view, single_to + buf * single_next,
                             single_at < 0 ? -1 : min(single_row, last) * single_bytes + single_at);
    }
    next_row += REC_BLOCK * ldq;
    next_single += REC_BLOCK * (long long)(single_bytes / 4);
  };
  auto lane_sum = [&](const float (&x)[N], const float (&y)[N]) {
    float part[2] = {0.f, 0.f};
#pragma unroll
    for (int p = 0; p < 2; ++p)
#pragma unroll
      for (int i = 0; i < Q; ++i) part[p] = fmaf(x[p * Q + i], y[p * Q + i], part[p]);
    return part[0] + part[1];
  };
  float outs = 0.f;      // lane j of every row: its row's part of token j's read-out, which nothing waits for
  auto store = [&](int t0) {
    const float o = pair_total(outs);
    const int j = lane & 31;
    if (live && j < min(REC_BLOCK, end - t0)) out[((long long)(t0 + j) * heads + h) * vdim + v] = o;
  };
  fetch(start, 0);
  for (int t0 = start, buf = 0; t0 < end; t0 += REC_BLOCK, buf ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0F70);     // the wave's loads of this block, asked for a block ago
    __syncthreads();                        // everybody's; and nobody reads the block before any more
    if (t0 > start) store(t0 - REC_BLOCK);
    if (t0 + REC_BLOCK < end) fetch(t0 + REC_BLOCK, buf ^ 1);
    const int count = min(REC_BLOCK, end - t0);
    auto read_k = [&](int j, float (&kk)[N]) {
#pragma unroll
      for (int i = 0; i < N; ++i) kk[i] = rows[buf][1][j][d0 + i];
    };
    auto read_q = [&](int j, float (&qq)[N]) {
#pragma unroll
      for (int i = 0; i < N; ++i) qq[i] = rows[buf][0][j][d0 + i];
    };
    auto read_gates = [&](int j, float (&gg)[N], float& b) {
      b = gates[buf][0][j];
      const float g = CH ? 0.f : gates[buf][1][j];
#pragma unroll
      for (int i = 0; i < N; ++i) gg[i] = CH ? rows[buf][KINDS - 1][j][d0 + i] : g;
    };
    auto keep_out = [&](int j, float o) { outs = (lane & (REC_BLOCK - 1)) == j ? o : outs; };
    constexpr int AHEAD = 2, READS = CH ? 5 : 4;      // a token's LDS reads go two tokens before its arithmetic
    float kk[AHEAD + 1][N], qq[AHEAD + 2][N], gg[AHEAD + 1][N], b[AHEAD + 1], val[AHEAD + 1], part[2];
    if (count == REC_BLOCK) {
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        read_k(j, kk[j]);
        read_gates(j, gg[j], b[j]);
        val[j] = values[buf][j][col];
        read_q(j, qq[j]);
      }
      float o = 0.f, before = 0.f;     // lane sums of the read-outs of the token before and of the one before that
#define VK_FENCE __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int j = 0; j < REC_BLOCK; ++j) {
        const int now = j % (AHEAD + 1), next = (j + AHEAD) % (AHEAD + 1);
        const bool more = j + AHEAD < REC_BLOCK;
        const float(&q)[N] = qq[(j + AHEAD + 1) % (AHEAD + 2)];
        if (j + 1 < REC_BLOCK) __builtin_amdgcn_s_waitcnt(0xC07F | READS << 8);      // the token's LDS reads
        else __builtin_amdgcn_s_waitcnt(0xC07F);
        VK_FENCE
        float held[N];
#pragma unroll
        for (int i = 0; i < N; ++i) held[i] = S[i];
#pragma unroll
        for (int i = 0; i < N; ++i) S[i] *= gg[now][i];
        float dot = lane_sum(S, kk[now]);
        VK_FENCE
        before = o;
        if (j > 0) {
          part[0] = fmaf(held[0], q[0], 0.f);
          part[1] = fmaf(held[Q], q[Q], 0.f);
        }
        VK_FENCE
        dot = dpp_add<0xB1>(dot);
        if (j > 1) before = dpp_add<0xB1>(before);
        if (Q > 1 && j > 0) part[0] = fmaf(held[1], q[1], part[0]);
        VK_FENCE
        dot = dpp_add<0x4E>(dot);
        if (j > 1) before = dpp_add<0x4E>(before);
        if (Q > 1 && j > 0) part[1] = fmaf(held[Q + 1], q[Q + 1], part[1]);
        VK_FENCE
        dot = dpp_add<0x141>(dot);
        if (j > 1) before = dpp_add<0x141>(before);
        if (j > 0) o = part[0] + part[1];
        VK_FENCE
        dot = dpp_add<0x140>(dot);
        if (j > 1) before = dpp_add<0x140>(before);
        if (more) read_k(j + AHEAD, kk[next]);
        VK_FENCE
        if (more) {
          read_gates(j + AHEAD, gg[next], b[next]);
          val[next] = values[buf][j + AHEAD][col];
        }
        const float total = pair_total(dot);
        if (more) read_q(j + AHEAD, qq[(j + AHEAD) % (AHEAD + 2)]);
        if (j > 1) keep_out(j - 2, before);
        VK_FENCE
        const float u = b[now] * (val[now] - total);
#pragma unroll
        for (int i = 0; i < N; ++i) S[i] = fmaf(kk[now][i], u, S[i]);
        VK_FENCE
      }
#undef VK_FENCE
      const float last = lane_sum(S, qq[(REC_BLOCK - 1) % (AHEAD + 2)]);
      keep_out(REC_BLOCK - 2, row_sum16(o));
      keep_out(REC_BLOCK - 1, row_sum16(last));
    } else {
      for (int j = 0; j < count; ++j) {
        read_k(j, kk[0]);
        read_q(j, qq[0]);
        read_gates(j, gg[0], b[0]);
        val[0] = values[buf][j][col];
#pragma unroll
        for (int i = 0; i < N; ++i) S[i] *= gg[0][i];
        const float u = b[0] * (val[0] - pair_total(row_sum16(lane_sum(S, kk[0]))));
#pragma unroll
        for (int i = 0; i < N; ++i) S[i] = fmaf(kk[0][i], u, S[i]);
        keep_out(j, row_sum16(lane_sum(S, qq[0])));
      }
    }
  }
  store(start + (end - start - 1) / REC_BLOCK * REC_BLOCK);
  if (kept) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (d0 + i < key_pad) mine[i] = S[i];
  }
}

// An LDS row of a token: [r: 64Q | k: 64Q | w: 64Q | v: 8].
template <int Q>
__global__ __launch_bounds__(SCAN_THREADS) void wkv_scan_kernel(
    const float* __restrict__ r, long long ldr, const float* __restrict__ k, long long ldk, const float* __restrict__ v,
    long long ldv, const float* __restrict__ wraw, long long ldw, const float* __restrict__ w0,
    const float* __restrict__ bonus, float* __restrict__ state, long long state_stride,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int dim,
    int heads, int key_pad, int value_pad, int decayed, float* __restrict__ out) {
  constexpr int DP = 64 * Q, ROW = 3 * DP + SCAN_COLS, TOKENS = REC_BLOCK / SCAN_COLS, PIECES = TOKENS * 3 * Q;
  __shared__ float rows[REC_BLOCK * ROW];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int d0 = lane * Q;
  const int v0 = blockIdx.z * SCAN_COLS, col_v = v0 + wave;
  const bool live = col_v < dim;
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* mine = state + (long long)slots[e] * state_stride + ((long long)h * value_pad + col_v) * key_pad + d0;
  const bool fresh = entry_first[e] == 0, kept = col_v < value_pad;
  float S[Q], U[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    S[i] = (!fresh && kept && d0 + i < key_pad) ? mine[i] : 0.f;
    U[i] = d0 + i < dim ? bonus[h * dim + d0 + i] : 0.f;
  }
  int from[Q];
#pragma unroll
  for (int c = 0; c < Q; ++c) from[c] = min(c * 64 + lane, dim - 1);
  const int value_j = tid / SCAN_COLS & (REC_BLOCK - 1);
  const float* values = v + h * dim + min(v0 + tid % SCAN_COLS, dim - 1);
  float held[PIECES], held_value;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int j = wave * TOKENS + i / (3 * Q), kind = i / Q % 3;
      const long long t = min(t0 + j, end - 1);
      held[i] = ((kind == 0 ? r + t * ldr : kind == 1 ? k + t * ldk : wraw + t * ldw) + h * dim)[from[i % Q]];
    }
    held_value = values[min(t0 + value_j, end - 1) * ldv];
  };
  fetch(start);
  for (int t0 = start; t0 < end; t0 += REC_BLOCK) {
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const int j = wave * TOKENS + i / (3 * Q), kind = i / Q % 3;
      float value = held[i];
      if (kind == 2 && !decayed) value = expf(-expf(value + w0[h * dim + from[i % Q]]));     // wraw is not the decay yet
      rows[j * ROW + kind * DP + i % Q * 64 + lane] = i % Q * 64 + lane < dim ? value : 0.f;
    }
    if (tid < REC_BLOCK * SCAN_COLS) rows[value_j * ROW + 3 * DP + tid % SCAN_COLS] = v0 + tid % SCAN_COLS < dim ? held_value : 0.f;
    __syncthreads();
    fetch(min(t0 + REC_BLOCK, end - 1));
    const int count = min(REC_BLOCK, end - t0);
    float outs = 0.f;      // lane j of every row: its row's part of token j's read-out, which nothing waits for
    constexpr int AHEAD = Q == 1 ? 4 : 2;      // tokens read from LDS before the arithmetic of the AHEAD before them
    float rr[2][AHEAD][Q], kk[2][AHEAD][Q], ww[2][AHEAD][Q], val[2][AHEAD];
    auto read = [&](int j, int of, int n) {
      const float* row = rows + j * ROW;
      val[of][n] = row[3 * DP + wave];
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        rr[of][n][i] = row[d0 + i];
        kk[of][n][i] = row[DP + d0 + i];
        ww[of][n][i] = row[2 * DP + d0 + i];
      }
    };
    auto token = [&](int of, int n) {
      float o = 0.f;
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const float kv = kk[of][n][i] * val[of][n];
        o = fmaf(fmaf(U[i], kv, S[i]), rr[of][n][i], o);
        S[i] = fmaf(ww[of][n][i], S[i], kv);
      }
      return o;
    };
    if (count == REC_BLOCK) {
#pragma unroll
      for (int n = 0; n < AHEAD; ++n) read(n, 0, n);
#pragma unroll
      for (int j = 0; j < REC_BLOCK; j += AHEAD) {
        const int of = j / AHEAD & 1;
        if (j + AHEAD < REC_BLOCK) {
#pragma unroll
          for (int n = 0; n < AHEAD; ++n) read(j + AHEAD + n, of ^ 1, n);
        }
        __builtin_amdgcn_sched_barrier(0);
        float o[AHEAD];
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) o[n] = token(of, n);
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) o[n] = row_sum16(o[n]);
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) outs = (lane & (REC_BLOCK - 1)) == j + n ? o[n] : outs;
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int j = 0; j < count; ++j) {
        read(j, 0, 0);
        const float o = row_sum16(token(0, 0));
        outs = (lane & (REC_BLOCK - 1)) == j ? o : outs;
      }
    }
    outs += __shfl_xor(outs, 16, 64);     // (row 0 + row 1) + (row 2 + row 3), in every row
    outs += __shfl_xor(outs, 32, 64);
    if (live && lane < count) out[((long long)(t0 + lane) * heads + h) * dim + col_v] = outs;
  }
  if (kept) {
#pragma unroll
    for (int i = 0; i < Q; ++i)
      if (d0 + i < key_pad) mine[i] = S[i];
  }
}

// The time mixing for head widths up to 128 in whole pieces of 16 bytes and decays taken beforehand, shaped as
// delta_scan_direct_kernel is, with every number formed as above: 32 lanes a value channel, some 16 instructions a token for two of
// them (13 above for one).  Nothing waits for a token's sums over the lanes, so sixteen tokens' go through the tree together.  Blocks
// of 32 tokens cost half as much besides, but leave room for three workgroups a CU instead of six.  us, above and here, as
// chosen: 32 heads of 64, one entry of 2,048 tokens 154 / 96, of 512 41 / 27, of 1,000 and 834 (512 workgroups) 109 / 70, of 512, 456 and 399
// (768) 71 / 47, eight of 250 (2,048) 96 / 70; in blocks of 32 / 16, when a block's places were still worked out anew: 108 / 127, 31 / 36, 82 / 87, 55 / 59, 84 / 75.  Entries that have no block of 32
// are walked in blocks of 16: 31 tokens of 16 heads in either 6.5 / 5.6, 16 tokens 5.0 / 4.0.
constexpr int WKV_LONG_BLOCKS = 3 * 256;      // workgroups up to which blocks are of 32 tokens
template <int Q, int BLOCK>
__global__ __launch_bounds__(SCAN_COLS * 32) void wkv_scan_direct_kernel(
    const float* __restrict__ r, long long ldr, const float* __restrict__ k, long long ldk, const float* __restrict__ v,
    long long ldv, const float* __restrict__ w, long long ldw, const float* __restrict__ bonus, float* __restrict__ state,
    long long state_stride, const int* __restrict__ entry_start, const int* __restrict__ entry_first,
    const int* __restrict__ slots, int dim, int heads, int key_pad, int value_pad, float* __restrict__ out) {
  // rows of a load (64 pieces of 16 bytes) and a wave's loads of a kind
  constexpr int DP = 64 * Q, N = 2 * Q, ROWS = 4 / Q, LOADS = BLOCK / ROWS / 4;
  __shared__ __attribute__((aligned(16))) float rows[2][3][BLOCK][DP];
  __shared__ float values[2][BLOCK][SCAN_COLS];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = tid >> 5, d0 = (lane & 31) * N;
  const int v0 = blockIdx.z * SCAN_COLS, col_v = v0 + col;
  const bool live = col_v < dim;
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* mine = state + (long long)slots[e] * state_stride + ((long long)h * value_pad + col_v) * key_pad + d0;
  const bool fresh = entry_first[e] == 0, kept = col_v < value_pad;
  float S[N], U[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    S[i] = (!fresh && kept && d0 + i < key_pad) ? mine[i] : 0.f;
    U[i] = d0 + i < dim ? bonus[h * dim + d0 + i] : 0.f;
  }
  const int first_row = wave * LOADS * ROWS + lane / (16 * Q), piece = lane % (16 * Q) * 4, value = v0 + (tid & 7);
  const float* next[3] = {r + start * ldr + h * dim, k + start * ldk + h * dim, w + start * ldw + h * dim};     // of the block fetched next
  const float* next_value = v + start * ldv + h * dim;
  const long long ld[3] = {ldr, ldk, ldw};
  int off[3][LOADS];
#pragma unroll
  for (int n = 0; n < 3; ++n)
#pragma unroll
    for (int i = 0; i < LOADS; ++i) off[n][i] = piece < dim ? ((first_row + i * ROWS) * (int)ld[n] + piece) * 4 : -1;
  const int value_off = value < dim ? ((tid >> 3) * (int)ldv + value) * 4 : -1;
  // a row past the entry's end is its last one, which nobody works on; what does not exist (-1) reads zeros
  auto fetch = [&](int t0, int buf) {
    const int last = end - 1 - t0;
    if (last >= BLOCK - 1) {
#pragma unroll
      for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
          scan_load_lds<true>(scan_view(next[n], 0x7fffffff), &rows[buf][n][(wave * LOADS + i) * ROWS][0], off[n][i]);
      if (wave * 8 < BLOCK) scan_load_lds<false>(scan_view(next_value, 0x7fffffff), &values[buf][wave * 8][0], value_off);
    } else {
#pragma unroll
      for (int n = 0; n < 3; ++n)
#pragma unroll
        for (int i = 0; i < LOADS; ++i)
          scan_load_lds<true>(scan_view(next[n], 0x7fffffff), &rows[buf][n][(wave * LOADS + i) * ROWS][0],
                              piece < dim ? (min(first_row + i * ROWS, last) * (int)ld[n] + piece) * 4 : -1);
      if (wave * 8 < BLOCK)
        scan_load_lds<false>(scan_view(next_value, 0x7fffffff), &values[buf][wave * 8][0],
                             value < dim ? (min(tid >> 3, last) * (int)ldv + value) * 4 : -1);
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) next[n] += BLOCK * ld[n];
    next_value += BLOCK * ldv;
  };
  const RowMerge merge(lane);
  float outs[BLOCK / REC_BLOCK];      // lane j of every row: its row's part of token j's read-out, which nothing waits for
  auto store = [&](int t0) {
#pragma unroll
    for (int half = 0; half < BLOCK / REC_BLOCK; ++half) {
      const float o = pair_total(outs[half]);
      const int j = half * REC_BLOCK + (lane & 31);
      if (live && (lane & 31) < REC_BLOCK && j < end - t0) out[((long long)(t0 + j) * heads + h) * dim + col_v] = o;
    }
  };
  fetch(start, 0);
  for (int t0 = start, buf = 0; t0 < end; t0 += BLOCK, buf ^= 1) {
    __builtin_amdgcn_s_waitcnt(0x0F70);     // the wave's loads of this block, asked for a block ago
    __syncthreads();                        // everybody's; and nobody reads the block before any more
    if (t0 > start) store(t0 - BLOCK);
    if (t0 + BLOCK < end) fetch(t0 + BLOCK, buf ^ 1);
    const int count = min(BLOCK, end - t0);
    constexpr int AHEAD = Q == 1 ? 4 : 2;      // tokens read from LDS before the arithmetic of the AHEAD before them
    float rr[2][AHEAD][N], kk[2][AHEAD][N], ww[2][AHEAD][N], val[2][AHEAD];
    auto read = [&](int j, int of, int n) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        rr[of][n][i] = rows[buf][0][j][d0 + i];
        kk[of][n][i] = rows[buf][1][j][d0 + i];
        ww[of][n][i] = rows[buf][2][j][d0 + i];
      }
      val[of][n] = values[buf][j][col];
    };
    auto token = [&](int of, int n) {
      float part[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float kv = kk[of][n][i] * val[of][n];
        part[i / Q] = fmaf(fmaf(U[i], kv, S[i]), rr[of][n][i], part[i / Q]);
        S[i] = fmaf(ww[of][n][i], S[i], kv);
      }
      return part[0] + part[1];
    };
    if (count == BLOCK) {
#pragma unroll
      for (int n = 0; n < AHEAD; ++n) read(n, 0, n);
      float o[4], quads[4];
#pragma unroll
      for (int j = 0; j < BLOCK; j += AHEAD) {
        const int of = j / AHEAD & 1;
        if (j + AHEAD < BLOCK) {
#pragma unroll
          for (int n = 0; n < AHEAD; ++n) read(j + AHEAD + n, of ^ 1, n);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int n = 0; n < AHEAD; ++n) o[(j + n) % 4] = token(of, n);
        if ((j + AHEAD) % 4 == 0) quads[j / 4 % 4] = merge.quads(o[0], o[1], o[2], o[3]);
        if ((j + AHEAD) % REC_BLOCK == 0) outs[j / REC_BLOCK] = merge.rows(quads);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int j = 0; j < count; ++j) {
        read(j, 0, 0);
        const float o = row_sum16(token(0, 0));
#pragma unroll
        for (int half = 0; half < BLOCK / REC_BLOCK; ++half)
          outs[half] = (lane & (REC_BLOCK - 1)) + half * REC_BLOCK == j ? o : outs[half];
      }
    }
  }
  store(start + (end - start - 1) / BLOCK * BLOCK);
  if (kept) {
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (d0 + i < key_pad) mine[i] = S[i];
  }
}

// ---------------------------------------------------------------------------------------------
// Token shift: mix_s[t] = h[t] + (h[t-1] - h[t]) * mu_s for `mixes` vectors mu; h[t-1] of an entry's first token
// is the state's saved row (zeros at position 0).  out [mixes, T, width] in the run's dtype.
template <typename T>
__global__ __launch_bounds__(256) void token_shift_kernel(const T* __restrict__ h, int width, const float* __restrict__ mu,
                                                          int mixes, const float* __restrict__ state,
                                                          long long state_stride, long long prev_offset,
                                                          const int* __restrict__ entry_of,
                                                          const int* __restrict__ entry_start,
                                                          const int* __restrict__ entry_first,
                                                          const int* __restrict__ slots, int num_tokens,
                                                          T* __restrict__ out) {
  const int t = blockIdx.x;
  const int e = entry_of[t];
  const bool first = t == entry_start[e];
  const bool fresh = entry_first[e] == 0;
  const float* saved = state + (long long)slots[e] * state_stride + prev_offset;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < width; c += gridDim.y * blockDim.x) {
    const float cur = to_float<T>(h[(long long)t * width + c]);
    // one load from a selected address, masked: no load behind a branch
    const float before = first ? saved[c] : to_float<T>(h[(long long)(t - 1) * width + c]);
    const float prev = (first && fresh) ? 0.f : before;
    const float diff = prev - cur;
    for (int s = 0; s < mixes; ++s)
      out[((long long)s * num_tokens + t) * width + c] = from_float<T>(fmaf(diff, mu[(long long)s * width + c], cur));
  }
}

// The same for many tokens: four channels of SHIFT_RUN consecutive tokens a thread, so that a vector of factors is read once for
// them and everything moves in pieces of four numbers.  2,048 tokens of 2,048 channels, six vectors, 16-bit: 27.0 -> 15.5 us;
// 512 of them 14.0 -> 8.3.  A row of up to 256 channels is one turn of a workgroup above and a quarter of one here: there runs are for
// many tokens.  us, six vectors, 16-bit: 512 tokens of 64 channels 4.8 / 5.7, of 256 5.0 / 5.6, of 320 6.0 / 6.0; 1,300 of 256 5.9 / 6.1, 2,048
// of 192 6.1 / 6.1, of 256 6.5 / 6.3.
constexpr int SHIFT_RUN = 4, SHIFT_TURN = 256;
constexpr long long SHIFT_MANY = 1 << 19;
template <typename T>
__global__ __launch_bounds__(256) void token_shift_run_kernel(const T* __restrict__ h, int width, const float* __restrict__ mu,
                                                              int mixes, const float* __restrict__ state,
                                                              long long state_stride, long long prev_offset,
                                                              const int* __restrict__ entry_of,
                                                              const int* __restrict__ entry_start,
                                                              const int* __restrict__ entry_first,
                                                              const int* __restrict__ slots, int num_tokens,
                                                              T* __restrict__ out) {
  typedef T four __attribute__((ext_vector_type(4)));
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  const int t0 = blockIdx.x * SHIFT_RUN, tokens = min(SHIFT_RUN, num_tokens - t0);
  for (int c = (blockIdx.y * blockDim.x + threadIdx.x) * 4; c < width; c += gridDim.y * blockDim.x * 4) {
    four row[SHIFT_RUN + 1];       // the token before the first, then the run's
#pragma unroll
    for (int i = 0; i <= SHIFT_RUN; ++i)
      row[i] = *(const four*)(h + (long long)min(max(t0 + i - 1, 0), num_tokens - 1) * width + c);
    f32x4 cur[SHIFT_RUN], diff[SHIFT_RUN];
#pragma unroll
    for (int i = 0; i < SHIFT_RUN; ++i) {
      const int t = min(t0 + i, num_tokens - 1), e = entry_of[t];
      f32x4 prev;
      if (t == entry_start[e]) {
        prev = f32x4{0.f, 0.f, 0.f, 0.f};
        if (entry_first[e] != 0) prev = *(const f32x4*)(state + (long long)slots[e] * state_stride + prev_offset + c);
      } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) prev[k] = to_float<T>(row[i][k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        cur[i][k] = to_float<T>(row[i + 1][k]);
        diff[i][k] = prev[k] - cur[i][k];
      }
    }
    for (int s = 0; s < mixes; ++s) {
      const f32x4 m = *(const f32x4*)(mu + (long long)s * width + c);
#pragma unroll
      for (int i = 0; i < SHIFT_RUN; ++i) {
        if (i >= tokens) break;
        four mixed;
#pragma unroll
        for (int k = 0; k < 4; ++k) mixed[k] = from_float<T>(fmaf(diff[i][k], m[k], cur[i][k]));
        *(four*)(out + ((long long)s * num_tokens + t0 + i) * width + c) = mixed;
      }
    }
  }
}

// An entry's last h becomes the state's saved row; one workgroup per entry, after token_shift has read the old one.
template <typename T>
__global__ __launch_bounds__(256) void save_last_kernel(const T* __restrict__ h, int width, float* __restrict__ state,
                                                        long long state_stride, long long prev_offset,
                                                        const int* __restrict__ entry_start,
                                                        const int* __restrict__ slots) {
  const int e = blockIdx.x;
  const int last = entry_start[e + 1] - 1;
  float* saved = state + (long long)slots[e] * state_stride + prev_offset;
  for (int c = blockIdx.y * blockDim.x + threadIdx.x; c < width; c += gridDim.y * blockDim.x)
    saved[c] = to_float<T>(h[(long long)last * width + c]);
}

// ---------------------------------------------------------------------------------------------
// Read-out of a recurrent head: o / rms(o) (per head, over its `vdim` channels) * weight * gate.
// weight: [vdim] shared by the heads, or [heads * vdim]; gate: a column range of a [T, ldg] buffer of type TG,
// as it is (`gate_silu` 0), through silu (1) or through the sigmoid (2).  One wave per (token, head).  N: 64 N >= vdim, a lane
// asks for everything at once; 0: any width, read twice.  2,048 tokens of 16 heads of 128, 32-bit gates: 15.8 -> 12.3 us.
template <typename TG, typename TO, int N>
__global__ __launch_bounds__(256) void head_norm_gate_kernel(const float* __restrict__ o, const float* __restrict__ weight,
                                                             int weight_per_head, const TG* __restrict__ gate,
                                                             long long ldg, int gate_silu, float eps, int heads,
                                                             int vdim, int num_tokens, TO* __restrict__ out) {
  const int lane = threadIdx.x & (WAVE - 1);
  const long long unit = (long long)blockIdx.x * (blockDim.x / WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
  const long long units = (long long)num_tokens * heads;
  if (unit >= units) return;
  const int t = units <= 0xffffffffll ? (int)((unsigned)unit / (unsigned)heads) : (int)(unit / heads), h = (int)(unit - (long long)t * heads);
  const float* src = o + unit * vdim;
  const TG* gates = gate + (long long)t * ldg + h * vdim;
  const float* weights = weight + (weight_per_head ? h * vdim : 0);
  auto result = [&](float x, float inv, float w, float g) {
    if (gate_silu == 1) g = silu_f(g);
    else if (gate_silu == 2) g = sigmoid_f(g);
    return from_float<TO>(x * inv * w * g);
  };
  float ss = 0.f;
  if constexpr (N > 0) {
    float x[N], g[N], w[N];
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const int c = min(lane + i * WAVE, vdim - 1);
      x[i] = src[c];
      g[i] = to_float<TG>(gates[c]);
      w[i] = weights[c];
    }
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (lane + i * WAVE < vdim) ss = fmaf(x[i], x[i], ss);
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)vdim + eps);
#pragma unroll
    for (int i = 0; i < N; ++i)
      if (lane + i * WAVE < vdim) out[unit * vdim + lane + i * WAVE] = result(x[i], inv, w[i], g[i]);
  } else {
    for (int c = lane; c < vdim; c += WAVE) ss += src[c] * src[c];
    ss = wave_sum(ss);
    const float inv = 1.0f / sqrtf(ss / (float)vdim + eps);
    for (int c = lane; c < vdim; c += WAVE) out[unit * vdim + c] = result(src[c], inv, weights[c], to_float<TG>(gates[c]));
  }
}

// ---------------------------------------------------------------------------------------------
// Matrix memory with exponential gates (mLSTM).  Per head, with S [dim, vdim], n [dim] and a running maximum m of the
// gates' logarithms (all zero at position 0):
//   li = cap tanh(i_raw / cap),  lf = logsigmoid(cap tanh(f_raw / cap))
//   m' = max(lf + m, li);  a = exp(lf + m - m'),  b = exp(li - m')
//   S <- a S + b k v^T;  n <- a n + b k;  o = S^T q / (max(|n . q|, exp(-m')) + 1e-6)
// All operands are columns of one 32-bit buffer `proj [T, ldp]`: q (heads * dim) from q_col on, k from k_col, v
// (heads * vdim) from v_col, the raw gates at i_col + h and f_col + h; q is multiplied by `q_scale` as it is read.
// State row of a request: the heads' matrices in the recurrences' common layout, then n and m once per tile of eight
// value channels ([heads][tiles][key_pad] and [heads][tiles]): every workgroup carries n and m itself, so it reads and
// writes copies of its own and no workgroup waits for another.
struct MemoryColumns {
  int q, k, v, i, f;
};

__device__ __forceinline__ float log_sigmoid_f(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }
__device__ __forceinline__ float log_gate(float raw, float cap, bool forget) {
  const float z = cap * tanhf(raw / cap);
  return forget ? log_sigmoid_f(z) : z;
}

// Steps of single tokens: the delta rule's shape (a workgroup owns 16 value channels of one (entry, head), the sixteen
// lanes of a row keep R key channels each of S and of n).  Grid (entries, heads, ceil(vdim / 16)).
template <int R>
__global__ __launch_bounds__(256) void memory_rule_kernel(
    const float* __restrict__ proj, long long ldp, MemoryColumns col, float q_scale, float cap,
    float* __restrict__ state, long long state_stride, long long n_offset, long long m_offset,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int dim,
    int heads, int vdim, float* __restrict__ out) {
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int grp = lane & 15, d0 = grp * R, key_pad = 16 * R;
  const int v0 = blockIdx.z * REC_COLS, v = v0 + wave * 4 + (lane >> 4);
  const bool live = v < vdim;
  const int tiles = 2 * gridDim.z;       // tiles of eight value channels: this workgroup owns 2 z and 2 z + 1
  const int start = entry_start[e], end = entry_start[e + 1];
  float* row = state + (long long)slots[e] * state_stride;
  float* mine = row + (((long long)h * gridDim.z * REC_COLS + v) * 16 + grp) * R;
  float* my_n = row + n_offset + ((long long)h * tiles + 2 * blockIdx.z) * key_pad + d0;
  float* my_m = row + m_offset + (long long)h * tiles + 2 * blockIdx.z;
  const bool fresh = entry_first[e] == 0;
  float S[R], N[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const float s_old = mine[i], n_old = my_n[i];
    S[i] = fresh ? 0.f : s_old;
    N[i] = fresh ? 0.f : n_old;
  }
  const float m_old = my_m[0];
  float m = fresh ? 0.f : m_old;
  for (int t = start; t < end; ++t) {
    const float* p = proj + (long long)t * ldp;
    const float li = log_gate(p[col.i + h], cap, false), lf = log_gate(p[col.f + h], cap, true);
    const float val_loaded = p[col.v + h * vdim + (live ? v : 0)];
    const float val = live ? val_loaded : 0.f;
    float kk[R], qq[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const bool in = d0 + i < dim;
      const float k_loaded = p[col.k + h * dim + (in ? d0 + i : 0)], q_loaded = p[col.q + h * dim + (in ? d0 + i : 0)];
      kk[i] = in ? k_loaded : 0.f;
      qq[i] = in ? q_loaded * q_scale : 0.f;
    }
    const float m_new = fmaxf(lf + m, li);
    const float a = expf(lf + m - m_new), b = expf(li - m_new);
    m = m_new;
    float num[2] = {0.f, 0.f}, den[2] = {0.f, 0.f};     // two chains each, even and odd rows: a fixed order
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const float bk = b * kk[i];
      S[i] = fmaf(bk, val, a * S[i]);
      N[i] = fmaf(a, N[i], bk);
      num[i & 1] = fmaf(S[i], qq[i], num[i & 1]);
      den[i & 1] = fmaf(N[i], qq[i], den[i & 1]);
    }
    const float top = row_sum16(num[0] + num[1]), under = row_sum16(den[0] + den[1]);
    if (live && grp == 0) out[((long long)t * heads + h) * vdim + v] = top / (fmaxf(fabsf(under), expf(-m)) + 1e-6f);
  }
#pragma unroll
  for (int i = 0; i < R; ++i) mine[i] = S[i];
  if (wave == 0 && lane < 16) {
#pragma unroll
    for (int i = 0; i < R; ++i) {
      my_n[i] = N[i];
      my_n[key_pad + i] = N[i];
    }
    if (lane == 0) my_m[0] = my_m[1] = m;
  }
}

// The gates' logarithms of a step's tokens, in place: proj[t, i_col + h] <- li, proj[t, f_col + h] <- lf.  A prompt's
// recurrence reads them a block of tokens at a time and takes no tanh or logarithm itself.
__global__ __launch_bounds__(256) void memory_gates_kernel(float* __restrict__ proj, long long ldp, int i_col, int f_col,
                                                           int heads, float cap, long long count) {
  const long long x = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (x >= count) return;
  float* p = proj + x / heads * ldp + x % heads;
  p[i_col] = log_gate(p[i_col], cap, false);
  p[f_col] = log_gate(p[f_col], cap, true);
}

// Prompts' portions: the scan shape (a wave owns one value channel and its 64 lanes the key channels, eight waves to a
// workgroup, tokens through LDS in blocks of 16 fetched a block ahead).  Every wave carries n and m itself, but n . q
// is the same number in all eight waves: each works it out for two of the block's tokens and leaves it in LDS.  Nothing
// of a token's read-out goes back into the state, so S^T q is summed inside each row of sixteen lanes as the tokens
// pass (lane j of a row keeps token j's) and across the four rows once per block.
// An LDS row of a token: [q: 64Q | k: 64Q | v: 8]; the two gates' logarithms lie beside.  Grid (entries, heads, tiles).
// The gates' columns of `proj` hold the logarithms li and lf already (memory_gates_kernel).
template <int Q>
__global__ __launch_bounds__(SCAN_THREADS) void memory_scan_kernel(
    const float* __restrict__ proj, long long ldp, MemoryColumns col, float q_scale,
    float* __restrict__ state, long long state_stride, long long n_offset, long long m_offset,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int dim,
    int heads, int vdim, int key_pad, int value_pad, float* __restrict__ out) {
  constexpr int DP = 64 * Q, ROW = 2 * DP + SCAN_COLS, COUNT = REC_BLOCK * ROW, LOADS = (COUNT + SCAN_THREADS - 1) / SCAN_THREADS;
  constexpr int PER_WAVE = REC_BLOCK / SCAN_COLS;     // tokens of a block whose n . q a wave works out
  static_assert(PER_WAVE * SCAN_COLS == REC_BLOCK && REC_BLOCK == 16, "a block's tokens are a row of lanes, dealt to the waves");
  __shared__ float rows[COUNT];
  __shared__ float gates[REC_BLOCK][2];
  __shared__ float dens[REC_BLOCK];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int d0 = lane * Q;
  const int v0 = blockIdx.z * SCAN_COLS, v = v0 + wave;
  const bool live = v < vdim;
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* row0 = state + (long long)slots[e] * state_stride;
  float* mine = row0 + ((long long)h * value_pad + v) * key_pad + d0;
  float* my_n = row0 + n_offset + ((long long)h * gridDim.z + blockIdx.z) * key_pad + d0;
  float* my_m = row0 + m_offset + (long long)h * gridDim.z + blockIdx.z;
  const bool fresh = entry_first[e] == 0;
  float S[Q], N[Q];
#pragma unroll
  for (int i = 0; i < Q; ++i) {
    const bool in = d0 + i < key_pad;
    const float s_old = mine[in ? i : -d0], n_old = my_n[in ? i : -d0];     // a clamped address where the lane has no row
    S[i] = (!fresh && in) ? s_old : 0.f;
    N[i] = (!fresh && in) ? n_old : 0.f;
  }
  const float m_old = my_m[0];
  float m = fresh ? 0.f : m_old;
  // a block's fetch plan: token * 2^24 + the column inside the token's row of proj, or -1 for what is always zero
  int plan[LOADS];
  unsigned is_q = 0;     // bit i: element i of this thread is a query's number
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int x = tid + i * SCAN_THREADS, j = x / ROW, c = x % ROW;
    int within = -1;
    if (x < COUNT) {
      if (c < DP) { if (c < dim) within = col.q + h * dim + c; }
      else if (c < 2 * DP) { if (c - DP < dim) within = col.k + h * dim + c - DP; }
      else if (v0 + c - 2 * DP < vdim) within = col.v + h * vdim + v0 + c - 2 * DP;
    }
    plan[i] = within < 0 ? -1 : (j << 24) | within;
    is_q |= (unsigned)(c < DP) << i;
  }
  // A fetch only issues loads, every thread the same number of them and none inside a branch, from addresses that
  // exist whatever the block holds (the entry's last token stands in for tokens past its end, column 0 for numbers that
  // are always zero); what a loaded number becomes is decided when it is stored into LDS, a block later, so that
  // nothing waits for memory before the block in between has been worked on.
  float held[LOADS], held_gate;
  const int gate_col = ((tid & 1) ? col.f : col.i) + h;
  auto fetch = [&](int t0) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int t = min(t0 + (plan[i] >> 24 & 127), end - 1);
      held[i] = proj[(long long)t * ldp + (plan[i] < 0 ? 0 : plan[i] & 0xFFFFFF)];
    }
    held_gate = proj[(long long)min(t0 + ((tid >> 1) & (REC_BLOCK - 1)), end - 1) * ldp + gate_col];
  };
  fetch(start);
  for (int t0 = start; t0 < end; t0 += REC_BLOCK) {
    // the block before has been read: every wave has passed the barrier at its end
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      if (tid + i * SCAN_THREADS < COUNT)
        rows[tid + i * SCAN_THREADS] = plan[i] < 0 ? 0.f : (is_q >> i & 1) ? held[i] * q_scale : held[i];
    if (tid < 2 * REC_BLOCK) gates[tid >> 1][tid & 1] = held_gate;
    __syncthreads();
    fetch(min(t0 + REC_BLOCK, end - 1));
    const int count = min(REC_BLOCK, end - t0);
    // The block's running maxima in closed form, so that no exponential waits for the token before it: with F_j the sum
    // of the forget gates' logarithms up to token j of the block and m0 the maximum the block starts from,
    // m_j = F_j + max(m0, max over l <= j of (li_l - F_l)).  Lane l of every row of sixteen works out token l & 15: two
    // scans along the row (sum, then maximum), its maximum and its neighbour's before it, and from those its three
    // exponentials; the token loop fetches them by lane.  Which sequence of maxima is used does not change the result
    // beyond rounding, as long as S, n and the floor of the denominator use the same one; the sequence here is one fixed
    // function of the block's gates and m0.
    float keep_j, take_j, floor_j, m_j;
    {
      const int jj = lane & (REC_BLOCK - 1);
      const float li_j = gates[jj][0], lf_j = gates[jj][1];
      float F = lf_j;
      F += row_shifted<1>(F, 0.f);
      F += row_shifted<2>(F, 0.f);
      F += row_shifted<4>(F, 0.f);
      F += row_shifted<8>(F, 0.f);
      float p = li_j - F;
      p = fmaxf(p, row_shifted<1>(p, -INFINITY));
      p = fmaxf(p, row_shifted<2>(p, -INFINITY));
      p = fmaxf(p, row_shifted<4>(p, -INFINITY));
      p = fmaxf(p, row_shifted<8>(p, -INFINITY));
      m_j = F + fmaxf(m, p);
      const float m_before = row_shifted<1>(m_j, m);      // the first token's: what the block starts from
      keep_j = expf(lf_j + m_before - m_j), take_j = expf(li_j - m_j), floor_j = expf(-m_j);
    }
    m = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_j), count - 1));
    float tops = 0.f;      // lane j of every row: its row's part of token j's S^T q
    auto token = [&](int j) {
      const float* row = rows + j * ROW;
      const float val = row[2 * DP + wave];
      const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(keep_j), j));
      const float b = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(take_j), j));
      float num = 0.f, qq[Q];
#pragma unroll
      for (int i = 0; i < Q; ++i) {
        const float bk = b * row[DP + d0 + i];
        qq[i] = row[d0 + i];
        S[i] = fmaf(bk, val, a * S[i]);
        N[i] = fmaf(a, N[i], bk);
        num = fmaf(S[i], qq[i], num);
      }
      if (wave == j / PER_WAVE) {       // the whole wave or none of it
        float den = 0.f;
#pragma unroll
        for (int i = 0; i < Q; ++i) den = fmaf(N[i], qq[i], den);
        den = wave_total(den);
        if (lane == 0) dens[j] = den;
      }
      num = row_sum16(num);
      tops = (lane & (REC_BLOCK - 1)) == j ? num : tops;
    };
    if (count == REC_BLOCK) {      // a whole block: every lane index and LDS offset is a constant
#pragma unroll
      for (int j = 0; j < REC_BLOCK; ++j) token(j);
    } else {
      for (int j = 0; j < count; ++j) token(j);
    }
    // the four rows' parts: (row 0 + row 1) + (row 2 + row 3) in every row, whichever it is
    tops += __shfl_xor(tops, 16, 64);
    tops += __shfl_xor(tops, 32, 64);
    __syncthreads();     // every token's n . q is in LDS, and the block has been read
    if (live && lane < count)     // lane j < 16 also holds token j's floor; the division waits for the block's end
      out[((long long)(t0 + lane) * heads + h) * vdim + v] = tops / (fmaxf(fabsf(dens[lane]), floor_j) + 1e-6f);
  }
#pragma unroll
  for (int i = 0; i < Q; ++i)
    if (d0 + i < key_pad) {
      mine[i] = S[i];
      if (wave == 0) my_n[i] = N[i];
    }
  if (tid == 0) my_m[0] = m;
}

// The matrix memory for key widths up to 128 in whole pieces of 16 bytes, with 32 lanes a value channel as in
// delta_scan_direct_kernel and every number formed as above.  What bounds it is a wave's instructions, in the assembly some 780 for a
// block of sixteen tokens and two value channels: twenty a token are the recurrence, as many again its LDS reads, the sums through the lanes and n . q, and
// the rest the block's, 49 a token together or 95 ns at one every 1.95 ns; a token takes 110, and what the others pass with was not measured.  What a token needs once for all its value channels
// is done before the walk: the wave that has fetched a piece of q or k multiplies it by the scale or by the token's share on its way
// into LDS, and lane j of a row reads token j's gates itself, whose exponentials are taken among the products of the block before.
// Four tokens' LDS reads go before the arithmetic of the four before them, sixteen tokens' sums through the lanes together, and a
// wave works out n . q for four tokens of a block.  (Loads straight into LDS, scaled there: the compiler has every later LDS read of the
// rows wait for them, 253 us a prompt of 2,048.)  us, above and here, with the gates' kernel, launches behind one another in a graph: 16 heads of 128 x
// 128, one entry of 2,048 tokens 363 / 227, of 512 96 / 62, of 1,000 and 834 255 / 151, of 512, 456 and 399 200 / 94, eight of 250 251 / 124; 8 heads,
// 2,048 tokens 362 / 225; 6 heads of 64 x 64, 512, 456 and 399 81 / 50; 31 tokens 13 / 11.
template <int Q>
__global__ __launch_bounds__(SCAN_COLS * 32) void memory_scan_direct_kernel(
    const float* __restrict__ proj, long long ldp, MemoryColumns col, float q_scale,
    float* __restrict__ state, long long state_stride, long long n_offset, long long m_offset,
    const int* __restrict__ entry_start, const int* __restrict__ entry_first, const int* __restrict__ slots, int dim,
    int heads, int vdim, int key_pad, int value_pad, float* __restrict__ out) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr int DP = 64 * Q, N = 2 * Q, WAVES = SCAN_COLS / 2, GROUP = REC_BLOCK / WAVES;
  constexpr int PIECES = 2 * Q, ROWS = 4 / Q;      // a wave's loads of a block (64 pieces of 16 bytes), rows each
  static_assert(WAVES == 4 && GROUP == 4, "two waves fetch q, two k; a wave's n . q are of four tokens");
  __shared__ __attribute__((aligned(16))) float rows[2][2][REC_BLOCK][DP];
  __shared__ float values[2][REC_BLOCK][SCAN_COLS];
  __shared__ float dens[2][REC_BLOCK];
  const int e = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int who = tid >> 5, d0 = (lane & 31) * N, jj = lane & (REC_BLOCK - 1);
  const int v0 = blockIdx.z * SCAN_COLS, v = v0 + who;
  const bool live = v < vdim;
  const int start = entry_start[e], end = entry_start[e + 1];
  if (start >= end) return;      // the whole workgroup
  float* row0 = state + (long long)slots[e] * state_stride;
  float* mine = row0 + ((long long)h * value_pad + v) * key_pad + d0;
  float* my_n = row0 + n_offset + ((long long)h * gridDim.z + blockIdx.z) * key_pad + d0;
  float* my_m = row0 + m_offset + (long long)h * gridDim.z + blockIdx.z;
  const bool fresh = entry_first[e] == 0;
  float S[N], norm[N];
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const bool in = !fresh && d0 + i < key_pad;
    S[i] = in ? mine[i] : 0.f;
    norm[i] = in ? my_n[i] : 0.f;
  }
  float m = fresh ? 0.f : my_m[0];
  const int row_bytes = (int)ldp * 4, piece = lane % (16 * Q) * 4;
  const bool a_query = wave < 2;
  const int piece_at = piece < dim ? ((a_query ? col.q : col.k) + h * dim + piece) * 4 : -1;
  const int first_row = (wave & 1) * PIECES * ROWS + lane / (16 * Q);
  const int value_at = v0 + (tid & 7) < vdim ? (col.v + h * vdim + v0 + (tid & 7)) * 4 : -1;
  int piece_off[PIECES];
#pragma unroll
  for (int i = 0; i < PIECES; ++i) piece_off[i] = piece_at < 0 ? -1 : (first_row + i * ROWS) * row_bytes + piece_at;
  const int value_off = value_at < 0 ? -1 : (tid >> 3) * row_bytes + value_at;
  // a row past the entry's end is its last one, which nobody works on; what does not exist (-1) reads zeros
  f32x4 held[PIECES];
  float held_value = 0.f;
  auto fetch = [&](int t0) {
    const int last = min(REC_BLOCK, end - t0) - 1;
    const ScanView view = scan_view(proj + t0 * ldp, (last + 1) * row_bytes);
    const bool whole = last == REC_BLOCK - 1;
#pragma unroll
    for (int i = 0; i < PIECES; ++i)
      held[i] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(
          view.rsrc, whole || piece_at < 0 ? piece_off[i] : min(first_row + i * ROWS, last) * row_bytes + piece_at, 0, 0));
    if (a_query)
      held_value = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
          view.rsrc, whole || value_at < 0 ? value_off : min(tid >> 3, last) * row_bytes + value_at, 0, 0));
  };
  float li, lf;      // token jj's gates, of the block behind the one whose exponentials are next
  auto fetch_gates = [&](int t0) {
    const float* gates = proj + min(t0 + jj, end - 1) * ldp + h;
    li = gates[col.i];
    lf = gates[col.f];
  };
  // A block's running maxima in closed form, as above, of `count` tokens from the maximum m on.
  struct Gates { float keep, take, floor, m; };
  auto gates_of = [&](float li_j, float lf_j, float m, int count) {
    float F = lf_j;
    F += row_shifted<1>(F, 0.f);
    F += row_shifted<2>(F, 0.f);
    F += row_shifted<4>(F, 0.f);
    F += row_shifted<8>(F, 0.f);
    float p = li_j - F;
    p = fmaxf(p, row_shifted<1>(p, -INFINITY));
    p = fmaxf(p, row_shifted<2>(p, -INFINITY));
    p = fmaxf(p, row_shifted<4>(p, -INFINITY));
    p = fmaxf(p, row_shifted<8>(p, -INFINITY));
    const float m_j = F + fmaxf(m, p), m_before = row_shifted<1>(m_j, m);
    return Gates{expf(lf_j + m_before - m_j), expf(li_j - m_j), expf(-m_j),
                 __int_as_float(__builtin_amdgcn_readlane(__float_as_int(m_j), count - 1))};
  };
  // the wave's pieces of a block, times the scale (q) or the tokens' shares (k), into LDS
  auto share = [&](int buf, float take) {
#pragma unroll
    for (int i = 0; i < PIECES; ++i) {
      const float taken = __shfl(take, first_row + i * ROWS, 64);
      *(f32x4*)(&rows[buf][0][0][0] + (wave * PIECES + i) * 256 + lane * 4) = held[i] * (a_query ? q_scale : taken);
    }
    if (a_query) values[buf][tid >> 3][tid & 7] = held_value;
  };
  const RowMerge merge(lane);
  float tops = 0.f, floor_before = 0.f;      // lane j of every row: its row's part of token j's S^T q, and the token's floor
  auto store = [&](int t0, int buf) {
    const float top = pair_total(tops);
    if (live && (lane & 31) < min(REC_BLOCK, end - t0))
      out[((long long)(t0 + jj) * heads + h) * vdim + v] = top / (fmaxf(fabsf(dens[buf][jj]), floor_before) + 1e-6f);
  };
  fetch_gates(start);
  fetch(start);
  Gates now = gates_of(li, lf, m, min(REC_BLOCK, end - start));
  share(0, now.take);
  fetch_gates(start + REC_BLOCK);
  for (int t0 = start, buf = 0; t0 < end; t0 += REC_BLOCK, buf ^= 1) {
    const int count = min(REC_BLOCK, end - t0);
    const bool more = t0 + REC_BLOCK < end;
    // what was asked for a block ago, the gates among it: asked for here, or the compiler waits for them behind the loads below
    __builtin_amdgcn_s_waitcnt(0x0F70);
    __syncthreads();                        // everybody's part of the block; and nobody reads the block before any more
    float kk[2][GROUP][N], qq[2][GROUP][N], val[2][GROUP], quads[GROUP];
    auto read = [&](int j, int of, int n) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        kk[of][n][i] = rows[buf][1][j][d0 + i];
        qq[of][n][i] = rows[buf][0][j][d0 + i];
      }
      val[of][n] = values[buf][j][who];
    };
#pragma unroll
    for (int n = 0; n < GROUP; ++n) read(n, 0, n);
    if (t0 > start) store(t0 - REC_BLOCK, buf ^ 1);
    floor_before = now.floor;
    const float next_li = li, next_lf = lf;
    if (more) fetch(t0 + REC_BLOCK);
    fetch_gates(t0 + 2 * REC_BLOCK);
    auto lane_sum = [&](const float (&x)[N], const float (&y)[N]) {
      float part[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < N; ++i) part[i / Q] = fmaf(x[i], y[i], part[i / Q]);
      return part[0] + part[1];
    };
    auto token = [&](int j, int of, int n) {
      const float a = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(now.keep), j));
#pragma unroll
      for (int i = 0; i < N; ++i) S[i] = fmaf(kk[of][n][i], val[of][n], a * S[i]);
#pragma unroll
      for (int i = 0; i < N; ++i) norm[i] = fmaf(a, norm[i], kk[of][n][i]);
      return lane_sum(S, qq[of][n]);
    };
    Gates next = now;
    if (count == REC_BLOCK) {
      auto group = [&](int g, auto with_dens) {
        if (g == 1) next = gates_of(next_li, next_lf, now.m, min(REC_BLOCK, end - t0 - REC_BLOCK));
        float num[GROUP], den[GROUP];
#pragma unroll
        for (int n = 0; n < GROUP; ++n) {
          num[n] = token(g * GROUP + n, g & 1, n);
          if constexpr (decltype(with_dens)::value) den[n] = lane_sum(norm, qq[g & 1][n]);
        }
        quads[g] = merge.quads(num[0], num[1], num[2], num[3]);
        if constexpr (decltype(with_dens)::value) {      // lane n of every four: token n's
          float d = merge.quads(den[0], den[1], den[2], den[3]);
          int moved = __builtin_amdgcn_update_dpp(0, __float_as_int(d), 0x104, 0xF, 0x5, false);
          moved = __builtin_amdgcn_update_dpp(moved, __float_as_int(d), 0x114, 0xF, 0xA, false);
          d += __int_as_float(moved);
          d = pair_total(dpp_add<0x128>(d));
          if (lane < GROUP) dens[buf][g * GROUP + lane] = d;
        }
      };
#pragma unroll
      for (int g = 0; g < WAVES; ++g) {
        if (g + 1 < WAVES) {
#pragma unroll
          for (int n = 0; n < GROUP; ++n) read((g + 1) * GROUP + n, (g + 1) & 1, n);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (wave == g) group(g, std::integral_constant<bool, true>{});      // the whole wave or none of it
        else group(g, std::integral_constant<bool, false>{});
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) share(buf ^ 1, next.take);      // asked for a block ago
      tops = merge.rows(quads);
    } else {
      for (int j = 0; j < count; ++j) {
        read(j, 0, 0);
        const float num = row_sum16(token(j, 0, 0));
        tops = jj == j ? num : tops;
        if (wave == j / GROUP) {
          const float den = pair_total(row_sum16(lane_sum(norm, qq[0][0])));
          if (lane == 0) dens[buf][j] = den;
        }
      }
    }
    m = now.m;
    now = next;
  }
  __syncthreads();     // the last block's n . q are in LDS
  const int blocks = (end - start - 1) / REC_BLOCK;
  store(start + blocks * REC_BLOCK, blocks & 1);
#pragma unroll
  for (int i = 0; i < N; ++i)
    if (d0 + i < key_pad) {
      mine[i] = S[i];
      if (tid < 32) my_n[i] = norm[i];
    }
  if (tid == 0) my_m[0] = m;
}

// x[t, c] = exp(-exp(x[t, c] + w0[c])) in place: time mixing's decay, for a step whose recurrence reads it many times.
__global__ void decay_kernel(float* __restrict__ x, const float* __restrict__ w0, int width, long long count) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) x[i] = expf(-expf(x[i] + w0[i % width]));
}

// out = tanh(x), elementwise, 32-bit in, TO out.
template <typename TO>
__global__ void tanh_kernel(const float* __restrict__ x, TO* __restrict__ out, long long count) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < count) out[i] = from_float<TO>(tanhf(x[i]));
}

// ---------------------------------------------------------------------------------------------

extern "C" int vk_delta_prepare_strided(const float* proj, long long ldp, const float* conv, int taps, float* state,
                                        long long state_stride, long long conv_offset, const int* entry_of,
                                        const int* entry_start, const int* entry_first, const int* slots,
                                        const float* a_log, const float* dt_bias, int kv_heads, int dim, int heads,
                                        int vdim, int b_col, int a_col, float unit_eps, float* qkv, long long ldq,
                                        float* beta, float* decay, int num_tokens, int num_entries, void* stream) {
  if (num_tokens <= 0) return 0;
  if (taps < 1 || kv_heads < 1 || heads < 1 || dim < 1 || vdim < 1 || heads % kv_heads) return VK_BAD_ARGUMENT;
  const long long C = 2LL * kv_heads * dim + (long long)heads * vdim;
  if (dim > PREP_SPAN || C > 0x7fffffff) return VK_UNSUPPORTED_SIZE;
  if (ldq < C || (a_col >= 0 && (!decay || !a_log || !dt_bias))) return VK_BAD_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const long long segments = 2LL * kv_heads + ((long long)heads * vdim + PREP_SPAN - 1) / PREP_SPAN;
  if (segments > 65535) return VK_UNSUPPORTED_SIZE;
  const dim3 run_grid((num_tokens + PREP_RUN - 1) / PREP_RUN, (unsigned)((C + 255) / 256));
#define VK_PREPARE_RUN(TAPS)                                                                                            \
  delta_prepare_run_kernel<TAPS><<<run_grid, 256, 0, s>>>(proj, ldp, conv, state, state_stride, conv_offset, entry_of,   \
                                                          entry_start, entry_first, slots, a_log, dt_bias, kv_heads, dim, \
                                                          heads, vdim, b_col, a_col, unit_eps, qkv, ldq, beta, decay, num_tokens)
  const bool runs = (dim == 64 || dim == 128 || dim == 256) && num_tokens >= PREP_RUN_TOKENS && run_grid.y <= 65535 &&
                    (num_tokens * segments >= PREP_RUN_BLOCKS || (long long)heads * vdim >= PREP_SPAN);
  if (runs && taps == 4) VK_PREPARE_RUN(4);
  else if (runs && taps == 3) VK_PREPARE_RUN(3);
  else if (runs && taps == 2) VK_PREPARE_RUN(2);
  else
    delta_prepare_kernel<<<dim3(num_tokens, (unsigned)segments), 256, 0, s>>>(
        proj, ldp, conv, taps, state, state_stride, conv_offset, entry_of, entry_start, entry_first, slots, a_log, dt_bias,
        kv_heads, dim, heads, vdim, b_col, a_col, unit_eps, qkv, ldq, beta, decay);
#undef VK_PREPARE_RUN
  VK_LAUNCH_CHECK();
  if (taps > 1) {
    conv_state_kernel<<<dim3(num_entries, (unsigned)((C + 255) / 256)), 256, 0, s>>>(
        proj, ldp, taps, (int)C, state, state_stride, conv_offset, entry_start, entry_first, slots);
    VK_LAUNCH_CHECK();
  }
  return 0;
}

extern "C" int vk_delta_prepare(const float* proj, long long ldp, const float* conv, int taps, float* state,
                                long long state_stride, long long conv_offset, const int* entry_of,
                                const int* entry_start, const int* entry_first, const int* slots, const float* a_log,
                                const float* dt_bias, int kv_heads, int dim, int heads, int vdim, int b_col, int a_col,
                                float unit_eps, float* qkv, float* beta, float* decay, int num_tokens, int num_entries,
                                void* stream) {
  if (a_col < 0) return VK_BAD_ARGUMENT;
  return vk_delta_prepare_strided(proj, ldp, conv, taps, state, state_stride, conv_offset, entry_of, entry_start,
                                  entry_first, slots, a_log, dt_bias, kv_heads, dim, heads, vdim, b_col, a_col, unit_eps,
                                  qkv, 2LL * kv_heads * dim + (long long)heads * vdim, beta, decay, num_tokens,
                                  num_entries, stream);
}

// out[t, h * dim + d] = exp(-exp(a_log[h]) * softplus(raw[t, h * dim + d] + dt_bias[h * dim + d])): the delta rule's
// decay per head and key channel.  `raw` and `out` are 32-bit with row strides of their own.
__global__ void channel_decay_kernel(const float* __restrict__ raw, long long ldr, const float* __restrict__ a_log,
                                     const float* __restrict__ dt_bias, int dim, int width, long long total,
                                     float* __restrict__ out, long long ldo) {
  const long long idx = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= total) return;
  const long long t = idx / width;
  const int c = (int)(idx % width);
  out[t * ldo + c] = expf(-expf(a_log[c / dim]) * softplus_f(raw[t * ldr + c] + dt_bias[c]));
}

extern "C" int vk_channel_decay(const float* raw, long long ldr, const float* a_log, const float* dt_bias, int heads,
                                int dim, int num_tokens, float* out, long long ldo, void* stream) {
  if (num_tokens <= 0) return 0;
  if (heads < 1 || dim < 1) return VK_BAD_ARGUMENT;
  const int width = heads * dim;
  const long long total = (long long)num_tokens * width;
  channel_decay_kernel<<<(unsigned)((total + 255) / 256), 256, 0, (hipStream_t)stream>>>(raw, ldr, a_log, dt_bias, dim,
                                                                                        width, total, out, ldo);
  VK_LAUNCH_CHECK();
  return 0;
}

// Key channels a lane of the single-token form keeps: the state's key width is padded to 16 times this.
static inline int rows_of(int dim) { return dim <= 16 ? 1 : dim <= 32 ? 2 : dim <= 64 ? 4 : dim <= 128 ? 8 : 16; }

// Floats of one head's state as the recurrence kernels lay it out: [value channels padded to 16][key channels padded].
extern "C" long long vk_recurrent_head_floats(int dim, int vdim) {
  return (long long)((vdim + REC_COLS - 1) / REC_COLS) * REC_COLS * 16 * rows_of(dim);
}

// `g_col` >= 0: one decay per head and key channel, in columns g_col.. of the qkv rows ([heads, dim]; `decay` is not
// read); below 0: one decay per head, `decay` [T, heads].  `ldq` is the row stride of qkv.
extern "C" int vk_delta_rule_strided(const float* qkv, long long ldq, int g_col, const float* beta, const float* decay,
                                     float* state, long long state_stride, const int* entry_start,
                                     const int* entry_first, const int* slots, int kv_heads, int dim, int heads, int vdim,
                                     float* out, int num_entries, int short_entries, void* stream) {
  if (num_entries <= 0) return 0;
  if (kv_heads < 1 || heads < 1 || dim < 1 || vdim < 1 || heads % kv_heads) return VK_BAD_ARGUMENT;
  if (dim > 256 || heads > 65535) return VK_UNSUPPORTED_SIZE;
  const long long C = 2LL * kv_heads * dim + (long long)heads * vdim;
  if (ldq < C || (g_col < 0 && !decay) || (g_col >= 0 && g_col + (long long)heads * dim > ldq)) return VK_BAD_ARGUMENT;
  if (ldq >= (1 << 24)) return VK_UNSUPPORTED_SIZE;      // refused in both forms alike
  dim3 grid(num_entries, heads, (vdim + REC_COLS - 1) / REC_COLS);
  hipStream_t s = (hipStream_t)stream;
  const int key_pad = 16 * rows_of(dim), value_pad = (vdim + REC_COLS - 1) / REC_COLS * REC_COLS;
  const bool ch = g_col >= 0;
  if (!short_entries) {
    dim3 scan_grid(num_entries, heads, value_pad / SCAN_COLS);
#define VK_DELTA_SCAN(Q, CH)                                                                                         \
  delta_scan_kernel<Q, CH><<<scan_grid, SCAN_THREADS, 0, s>>>(qkv, ldq, g_col, beta, decay, state, state_stride,       \
                                                              entry_start, entry_first, slots, kv_heads, dim, heads,  \
                                                              vdim, key_pad, value_pad, out)
#define VK_DELTA_DIRECT(Q, CH)                                                                                       \
  delta_scan_direct_kernel<Q, CH><<<scan_grid, SCAN_COLS * 32, 0, s>>>(qkv, ldq, g_col, beta, decay, state,            \
                                                                       state_stride, entry_start, entry_first, slots, \
                                                                       kv_heads, dim, heads, vdim, key_pad, value_pad, out)
    if (key_pad <= 128 && dim % 4 == 0 && ldq % 4 == 0 && ((uintptr_t)qkv & 15) == 0 && (!ch || g_col % 4 == 0)) {
      if (key_pad <= 64) { if (ch) VK_DELTA_DIRECT(1, true); else VK_DELTA_DIRECT(1, false); }
      else { if (ch) VK_DELTA_DIRECT(2, true); else VK_DELTA_DIRECT(2, false); }
    }
    else if (key_pad <= 64) { if (ch) VK_DELTA_SCAN(1, true); else VK_DELTA_SCAN(1, false); }
    else if (key_pad <= 128) { if (ch) VK_DELTA_SCAN(2, true); else VK_DELTA_SCAN(2, false); }
    else { if (ch) VK_DELTA_SCAN(4, true); else VK_DELTA_SCAN(4, false); }
#undef VK_DELTA_SCAN
#undef VK_DELTA_DIRECT
    VK_LAUNCH_CHECK();
    return 0;
  }
#define VK_DELTA(R)                                                                                                     \
  do {                                                                                                                  \
    if (ch)                                                                                                             \
      delta_rule_kernel<R, 1, true><<<grid, 256, 0, s>>>(qkv, ldq, g_col, beta, decay, state, state_stride, entry_start, \
                                                         entry_first, slots, kv_heads, dim, heads, vdim, out);          \
    else                                                                                                                \
      delta_rule_kernel<R, 1, false><<<grid, 256, 0, s>>>(qkv, ldq, g_col, beta, decay, state, state_stride,            \
                                                          entry_start, entry_first, slots, kv_heads, dim, heads, vdim,  \
                                                          out);                                                         \
  } while (0)
  if (dim <= 16) { VK_DELTA(1); }
  else if (dim <= 32) { VK_DELTA(2); }
  else if (dim <= 64) { VK_DELTA(4); }
  else if (dim <= 128) { VK_DELTA(8); }
  else { VK_DELTA(16); }
#undef VK_DELTA
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_delta_rule(const float* qkv, const float* beta, const float* decay, float* state,
                             long long state_stride, const int* entry_start, const int* entry_first, const int* slots,
                             int kv_heads, int dim, int heads, int vdim, float* out, int num_entries, int short_entries,
                             void* stream) {
  return vk_delta_rule_strided(qkv, 2LL * kv_heads * dim + (long long)heads * vdim, -1, beta, decay, state, state_stride,
                               entry_start, entry_first, slots, kv_heads, dim, heads, vdim, out, num_entries,
                               short_entries, stream);
}

// Floats of one request's matrix-memory state: the heads' matrices, then n and m per tile of eight value channels.
extern "C" long long vk_memory_state_floats(int heads, int dim, int vdim) {
  const long long tiles = (vdim + REC_COLS - 1) / REC_COLS * (REC_COLS / SCAN_COLS);
  return (long long)heads * (vk_recurrent_head_floats(dim, vdim) + tiles * 16 * rows_of(dim) + tiles);
}

// `proj` holds `num_tokens` rows.  Unless `short_entries` says that every entry is a single token, the gates' columns
// of `proj` are overwritten with their logarithms.
extern "C" int vk_memory_rule(float* proj, long long ldp, int num_tokens, int q_col, int k_col, int v_col, int i_col,
                              int f_col, float q_scale, float cap, float* state, long long state_stride,
                              const int* entry_start, const int* entry_first, const int* slots, int dim, int heads,
                              int vdim, float* out, int num_entries, int short_entries, void* stream) {
  if (num_entries <= 0 || num_tokens <= 0) return 0;
  if (heads < 1 || dim < 1 || vdim < 1 || !(cap > 0.f)) return VK_BAD_ARGUMENT;
  if (dim > 256 || heads > 65535 || ldp >= (1 << 24)) return VK_UNSUPPORTED_SIZE;
  if (min(min(q_col, k_col), min(v_col, min(i_col, f_col))) < 0) return VK_BAD_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  const int key_pad = 16 * rows_of(dim), value_pad = (vdim + REC_COLS - 1) / REC_COLS * REC_COLS;
  const long long tiles = value_pad / SCAN_COLS;
  const long long n_offset = (long long)heads * vk_recurrent_head_floats(dim, vdim);
  const long long m_offset = n_offset + (long long)heads * tiles * key_pad;
  const MemoryColumns col{q_col, k_col, v_col, i_col, f_col};
  if (!short_entries) {
    const long long gates = (long long)num_tokens * heads;
    memory_gates_kernel<<<(unsigned)((gates + 255) / 256), 256, 0, s>>>(proj, ldp, i_col, f_col, heads, cap, gates);
    dim3 scan_grid(num_entries, heads, (unsigned)tiles);
#define VK_MEMORY_SCAN(Q)                                                                                            \
  memory_scan_kernel<Q><<<scan_grid, SCAN_THREADS, 0, s>>>(proj, ldp, col, q_scale, state, state_stride, n_offset,     \
                                                           m_offset, entry_start, entry_first, slots, dim, heads, vdim, \
                                                           key_pad, value_pad, out)
#define VK_MEMORY_DIRECT(Q)                                                                                          \
  memory_scan_direct_kernel<Q><<<scan_grid, SCAN_COLS * 32, 0, s>>>(proj, ldp, col, q_scale, state, state_stride,      \
                                                                    n_offset, m_offset, entry_start, entry_first,     \
                                                                    slots, dim, heads, vdim, key_pad, value_pad, out)
    const bool pieces = (dim | q_col | k_col) % 4 == 0 && ldp % 4 == 0 && ((uintptr_t)proj & 15) == 0;
    if (pieces && key_pad <= 64) VK_MEMORY_DIRECT(1);
    else if (pieces && key_pad <= 128) VK_MEMORY_DIRECT(2);
    else if (key_pad <= 64) VK_MEMORY_SCAN(1);
    else if (key_pad <= 128) VK_MEMORY_SCAN(2);
    else VK_MEMORY_SCAN(4);
#undef VK_MEMORY_SCAN
#undef VK_MEMORY_DIRECT
    VK_LAUNCH_CHECK();
    return 0;
  }
  dim3 grid(num_entries, heads, value_pad / REC_COLS);
#define VK_MEMORY(R)                                                                                                  \
  memory_rule_kernel<R><<<grid, 256, 0, s>>>(proj, ldp, col, q_scale, cap, state, state_stride, n_offset, m_offset,   \
                                             entry_start, entry_first, slots, dim, heads, vdim, out)
  if (dim <= 16) { VK_MEMORY(1); }
  else if (dim <= 32) { VK_MEMORY(2); }
  else if (dim <= 64) { VK_MEMORY(4); }
  else if (dim <= 128) { VK_MEMORY(8); }
  else { VK_MEMORY(16); }
#undef VK_MEMORY
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_wkv_rule(const float* r, long long ldr, const float* k, long long ldk, const float* v, long long ldv,
                           const float* wraw, long long ldw, const float* w0, const float* bonus, float* state,
                           long long state_stride, const int* entry_start, const int* entry_first, const int* slots,
                           int dim, int heads, float* out, int num_entries, int num_tokens, int short_entries,
                           int decayed, void* stream) {
  if (num_entries <= 0) return 0;
  if (heads < 1 || dim < 1) return VK_BAD_ARGUMENT;
  if (dim > 256 || heads > 65535) return VK_UNSUPPORTED_SIZE;
  dim3 grid(num_entries, heads, (dim + REC_COLS - 1) / REC_COLS);
  hipStream_t s = (hipStream_t)stream;
  const int key_pad = 16 * rows_of(dim), value_pad = (dim + REC_COLS - 1) / REC_COLS * REC_COLS;
  if (!short_entries) {
    dim3 scan_grid(num_entries, heads, value_pad / SCAN_COLS);
#define VK_WKV_SCAN(Q)                                                                                               \
  wkv_scan_kernel<Q><<<scan_grid, SCAN_THREADS, 0, s>>>(r, ldr, k, ldk, v, ldv, wraw, ldw, w0, bonus, state,          \
                                                        state_stride, entry_start, entry_first, slots, dim, heads,    \
                                                        key_pad, value_pad, decayed, out)
#define VK_WKV_DIRECT(Q, BLOCK)                                                                                      \
  wkv_scan_direct_kernel<Q, BLOCK><<<scan_grid, SCAN_COLS * 32, 0, s>>>(r, ldr, k, ldk, v, ldv, wraw, ldw, bonus,      \
                                                                        state, state_stride, entry_start, entry_first, \
                                                                        slots, dim, heads, key_pad, value_pad, out)
    const bool pieces = dim % 4 == 0 && (ldr | ldk | ldw) % 4 == 0 && (((uintptr_t)r | (uintptr_t)k | (uintptr_t)wraw) & 15) == 0 &&
                        std::max(std::max(ldr, ldk), std::max(ldv, ldw)) < (1 << 24);
    const long long groups = (long long)num_entries * heads * (value_pad / SCAN_COLS);
    const bool long_blocks = groups <= WKV_LONG_BLOCKS && num_tokens >= 32ll * num_entries;
    if (decayed && pieces && key_pad <= 64 && long_blocks) VK_WKV_DIRECT(1, 2 * REC_BLOCK);
    else if (decayed && pieces && key_pad <= 64) VK_WKV_DIRECT(1, REC_BLOCK);
    else if (decayed && pieces && key_pad <= 128) VK_WKV_DIRECT(2, REC_BLOCK);
    else if (key_pad <= 64) VK_WKV_SCAN(1);
    else if (key_pad <= 128) VK_WKV_SCAN(2);
    else VK_WKV_SCAN(4);
#undef VK_WKV_SCAN
#undef VK_WKV_DIRECT
    VK_LAUNCH_CHECK();
    return 0;
  }
#define VK_WKV(R)                                                                                                     \
  wkv_rule_kernel<R, 1><<<grid, 256, 0, s>>>(r, ldr, k, ldk, v, ldv, wraw, ldw, w0, bonus, state, state_stride,       \
                                             entry_start, entry_first, slots, dim, heads, decayed, out)
  if (dim <= 16) { VK_WKV(1); }
  else if (dim <= 32) { VK_WKV(2); }
  else if (dim <= 64) { VK_WKV(4); }
  else if (dim <= 128) { VK_WKV(8); }
  else { VK_WKV(16); }
#undef VK_WKV
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_token_shift(const void* h, int dtype, int width, const float* mu, int mixes, float* state,
                              long long state_stride, long long prev_offset, const int* entry_of,
                              const int* entry_start, const int* entry_first, const int* slots, int num_tokens,
                              int num_entries, void* out, void* stream) {
  if (num_tokens <= 0) return 0;
  if (width < 1 || mixes < 1) return VK_BAD_ARGUMENT;
  hipStream_t s = (hipStream_t)stream;
  // a step of few tokens spreads a row over several workgroups; a prompt's many tokens fill the GPU by themselves
  const unsigned spans = num_tokens >= 512 ? 1u : (unsigned)min(64, (width + 255) / 256);
  const dim3 tokens_grid(num_tokens, spans), entries_grid(num_entries, spans);
  const int bytes = dtype == DT_F32 ? 4 : 2;
  const bool runs = num_tokens >= 512 && (width > SHIFT_TURN || (long long)num_tokens * width >= SHIFT_MANY) && width % 4 == 0 && state_stride % 4 == 0 && prev_offset % 4 == 0 &&
                    (((uintptr_t)mu | (uintptr_t)state) & 15) == 0 && (((uintptr_t)h | (uintptr_t)out) % (4 * bytes)) == 0;
  const dim3 runs_grid((num_tokens + SHIFT_RUN - 1) / SHIFT_RUN, (unsigned)min(64, (width + 1023) / 1024));
  if (dtype == DT_F32) {
    if (runs)
      token_shift_run_kernel<float><<<runs_grid, 256, 0, s>>>((const float*)h, width, mu, mixes, state, state_stride, prev_offset,
                                                              entry_of, entry_start, entry_first, slots, num_tokens, (float*)out);
    else
      token_shift_kernel<float><<<tokens_grid, 256, 0, s>>>((const float*)h, width, mu, mixes, state, state_stride,
                                                           prev_offset, entry_of, entry_start, entry_first, slots,
                                                           num_tokens, (float*)out);
    VK_LAUNCH_CHECK();
    save_last_kernel<float><<<entries_grid, 256, 0, s>>>((const float*)h, width, state, state_stride, prev_offset,
                                                        entry_start, slots);
  } else if (dtype == DT_BF16) {
    if (runs)
      token_shift_run_kernel<bf16_t><<<runs_grid, 256, 0, s>>>((const bf16_t*)h, width, mu, mixes, state, state_stride, prev_offset,
                                                               entry_of, entry_start, entry_first, slots, num_tokens, (bf16_t*)out);
    else
      token_shift_kernel<bf16_t><<<tokens_grid, 256, 0, s>>>((const bf16_t*)h, width, mu, mixes, state, state_stride,
                                                            prev_offset, entry_of, entry_start, entry_first, slots,
                                                            num_tokens, (bf16_t*)out);
    VK_LAUNCH_CHECK();
    save_last_kernel<bf16_t><<<entries_grid, 256, 0, s>>>((const bf16_t*)h, width, state, state_stride, prev_offset,
                                                         entry_start, slots);
  } else {
    return VK_BAD_ARGUMENT;
  }
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_head_norm_gate(const float* o, const float* weight, int weight_per_head, const void* gate,
                                 int gate_dtype, long long ldg, int gate_silu, float eps, int heads, int vdim,
                                 int num_tokens, void* out, int out_dtype, void* stream) {
  if (num_tokens <= 0) return 0;
  if (heads < 1 || vdim < 1) return VK_BAD_ARGUMENT;
  const long long units = (long long)num_tokens * heads;
  const unsigned blocks = (unsigned)((units + 3) / 4);
  hipStream_t s = (hipStream_t)stream;
#define VK_HNG_N(TG, TO, N)                                                                                    \
  head_norm_gate_kernel<TG, TO, N><<<blocks, 256, 0, s>>>(o, weight, weight_per_head, (const TG*)gate, ldg,   \
                                                          gate_silu, eps, heads, vdim, num_tokens, (TO*)out)
#define VK_HNG(TG, TO)                     \
  do {                                     \
    if (vdim <= 64) VK_HNG_N(TG, TO, 1);   \
    else if (vdim <= 128) VK_HNG_N(TG, TO, 2); \
    else VK_HNG_N(TG, TO, 0);              \
  } while (0)
  if (gate_dtype == DT_F32 && out_dtype == DT_F32) VK_HNG(float, float);
  else if (gate_dtype == DT_F32 && out_dtype == DT_BF16) VK_HNG(float, bf16_t);
  else if (gate_dtype == DT_BF16 && out_dtype == DT_BF16) VK_HNG(bf16_t, bf16_t);
  else if (gate_dtype == DT_BF16 && out_dtype == DT_F32) VK_HNG(bf16_t, float);
  else return VK_BAD_ARGUMENT;
#undef VK_HNG
#undef VK_HNG_N
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_decay(float* x, const float* w0, int width, long long count, void* stream) {
  if (count <= 0) return 0;
  if (width < 1) return VK_BAD_ARGUMENT;
  decay_kernel<<<(unsigned)((count + 255) / 256), 256, 0, (hipStream_t)stream>>>(x, w0, width, count);
  VK_LAUNCH_CHECK();
  return 0;
}

extern "C" int vk_tanh(const float* x, void* out, int out_dtype, long long count, void* stream) {
  if (count <= 0) return 0;
  const unsigned blocks = (unsigned)((count + 255) / 256);
  hipStream_t s = (hipStream_t)stream;
  if (out_dtype == DT_F32) tanh_kernel<float><<<blocks, 256, 0, s>>>(x, (float*)out, count);
  else if (out_dtype == DT_BF16) tanh_kernel<bf16_t><<<blocks, 256, 0, s>>>(x, (bf16_t*)out, count);
  else return VK_BAD_ARGUMENT;
  VK_LAUNCH_CHECK();
  return 0;
}
