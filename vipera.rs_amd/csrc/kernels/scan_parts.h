// What the walks over prompts' tokens share (recurrent.hip, scan.hip).
#pragma once
#include "common.h"

// Sums over the sixteen lanes of a row, of sixteen numbers a lane at once: of two numbers that are summed alike each lane passes
// one on and keeps the other, so that a level of the tree (row_sum16's: neighbours, pairs, quads, eights) halves the numbers
// that are left instead of taking all of them through it.  In the end lane j has number j's sum.
template <int CTRL, int CTRL_ODD = 0>
__device__ __forceinline__ float row_merge(bool odd, float even_number, float odd_number) {
  const float kept = odd ? odd_number : even_number;
  const int sent = __float_as_int(odd ? even_number : odd_number);
  int moved;
  if constexpr (CTRL_ODD == 0) {
    moved = __builtin_amdgcn_update_dpp(0, sent, CTRL, 0xF, 0xF, false);
  } else {       // lanes of the even quads through one move, of the odd ones through the other
    moved = __builtin_amdgcn_update_dpp(0, sent, CTRL, 0xF, 0x5, false);
    moved = __builtin_amdgcn_update_dpp(moved, sent, CTRL_ODD, 0xF, 0xA, false);
  }
  return kept + __int_as_float(moved);
}
struct RowMerge {
  bool bit0, bit1, bit2, bit3;
  __device__ __forceinline__ explicit RowMerge(int lane) : bit0(lane & 1), bit1(lane & 2), bit2(lane & 4), bit3(lane & 8) {}
  __device__ __forceinline__ float quads(float a, float b, float c, float d) const {     // numbers 4 n .. 4 n + 3
    return row_merge<0x4E>(bit1, row_merge<0xB1>(bit0, a, b), row_merge<0xB1>(bit0, c, d));
  }
  __device__ __forceinline__ float rows(const float (&q)[4]) const {                     // quads() of n = 0 .. 3
    return row_merge<0x128>(bit3, row_merge<0x104, 0x114>(bit2, q[0], q[1]), row_merge<0x104, 0x114>(bit2, q[2], q[3]));
  }
};

// 16 or 4 bytes a lane from memory into LDS, one lane's behind the other's from `to` on; past the view's end zeros.
struct ScanView {
  __amdgpu_buffer_rsrc_t rsrc;
};
__device__ __forceinline__ ScanView scan_view(const float* base, int bytes) {
  return ScanView{__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), 0, bytes, 0x00020000)};
}
template <bool QUAD>
__device__ __forceinline__ void scan_load_lds(const ScanView view, float* to, int offset) {
  typedef __attribute__((address_space(3))) void* lds_ptr;
  if constexpr (QUAD)
    __builtin_amdgcn_raw_ptr_buffer_load_lds(view.rsrc, (lds_ptr)to, 16, offset, 0, 0, 0);
  else
    __builtin_amdgcn_raw_ptr_buffer_load_lds(view.rsrc, (lds_ptr)to, 4, offset, 0, 0, 0);
}
