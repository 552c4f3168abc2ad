// Shared by the sparse MLA decode kernels: the call's arguments and the fp8 /
// LDS helpers.
#pragma once

#include "ekv_common.h"

namespace ekv {

constexpr int kDv = 512;
constexpr int kMaxHeads = 64;
constexpr int kXcds = 8;                     // workgroup b runs on XCD b % 8
constexpr float kRescaleSlack = 8.0f;        // log2 units over a head's reference max that move it
constexpr float kLog2e = 0x1.715476p+0f;
constexpr float kLn2 = 0x1.62e430p-1f;

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) i16x4 lds_i16x4;

struct DecodeArgs {
  const uint16_t* q;        // [T, H, D] bf16
  int64_t q_tok_stride, q_head_stride;
  const uint8_t* cache;     // fp8 pages [num_pages, page_stride] or bf16 rows
  int64_t page_stride;      // bytes (fp8 layout)
  int64_t num_rows;         // addressable rows (num_pages * 64), < 2**31
  const int32_t* indices;   // [T, idx_stride]
  int64_t idx_stride;
  int32_t width;            // entries per index row
  const int32_t* lengths;   // [T] or null
  const int32_t* block_table;  // logical indices when non-null
  int64_t bt_stride;
  const int32_t* req_ids;   // [T] with block_table
  float scale;              // softmax scale
  int32_t heads;
  int32_t rows;             // T
  int32_t groups;           // G workgroups (a multiple of 8), >= T + T * tiles(width) / 32
  float* ws_o;              // [G, H, 512] fp32, O / l of workgroup g's split
  float* ws_ml;             // [G, H, 2] (m in log2 units, l)
  int2* ws_rows;            // [T] (first workgroup, splits) of each row
  const float* sinks;       // [H] or null
  uint16_t* out;            // [T, H, 512] bf16
  int64_t out_tok_stride, out_head_stride;
  float* lse;               // [T, H] or null
  int64_t lse_stride;
};

// Entries of row t.
__device__ __forceinline__ int row_len(const DecodeArgs& a, int t) {
  return a.lengths ? min(max(a.lengths[t], 0), a.width) : a.width;
}

// Four e4m3fn bytes -> four bf16 (exact: every e4m3fn value is a bf16 value).
__device__ __forceinline__ uint2 fp8x4_bf16(uint32_t w) {
  const bf16x2 lo = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, false);
  const bf16x2 hi = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.0f, true);
  return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}
__device__ __forceinline__ bf16x8 fp8x8_bf16(uint2 w) {
  const uint2 lo = fp8x4_bf16(w.x), hi = fp8x4_bf16(w.y);
  return __builtin_bit_cast(bf16x8, make_uint4(lo.x, lo.y, hi.x, hi.y));
}

__device__ __forceinline__ uint32_t bf16x2_bits(float a, float b) {
  const bf16x2 v = {static_cast<__bf16>(a), static_cast<__bf16>(b)};  // round to nearest even
  return __builtin_bit_cast(uint32_t, v);
}

// ds_read_b64_tr_b8: in each row of 16 lanes, lane j receives byte j % 8 of
// the 8 bytes addressed by lanes j / 8 + 2m (m = 0..7), as byte m.
typedef int i32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint2 lds_read_tr8(const uint8_t* p) {
  const i32x2 v = __builtin_amdgcn_ds_read_tr8_b64_v2i32(
      (__attribute__((address_space(3))) i32x2*)((__attribute__((address_space(3))) uint8_t*)(p)));
  return make_uint2(static_cast<uint32_t>(v.x), static_cast<uint32_t>(v.y));
}
// ds_read_b64_tr_b16: lane j receives 16-bit element j % 4 of the 8 bytes
// addressed by lanes j / 4 + 4m (m = 0..3), as element m.
__device__ __forceinline__ i16x4 lds_read_tr16(const uint8_t* p) {
  return __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (lds_i16x4*)((__attribute__((address_space(3))) uint8_t*)(p)));
}

// The whole-row kernel (ekv_decode_rows.hip): whether a call of num_tokens rows
// of `width` entries takes it (the few-row kernel would launch split_groups
// workgroups), and its launch.
bool decode_rows_takes(int32_t num_tokens, int32_t heads, int32_t width, bool cache_bf16, int64_t split_groups);
int launch_decode_rows(const DecodeArgs& a, int32_t dim, bool cache_bf16, hipStream_t s);

}  // namespace ekv
