// Shared by the codec's archive and reconstruction kernels: the item
// decomposition (fc_codec.hip's header comment), the raw-tail rows of a view
// and the launch descriptions of the register-resident jpeg kernels
// (fc_jpeg_encode.hip, fc_jpeg_decode.hip).
#pragma once

#include <type_traits>

#include "fc_attn_internal.h"
#include "fc_common.h"

namespace fc {

constexpr int kThreads = 256;

struct ItemMap {
  int64_t item;
  int lane;  // lane index inside the item group
};

// lpi_log2: log2 of the lanes per item.
__device__ __forceinline__ ItemMap item_of_thread(int lpi_log2) {
  ItemMap m;
  m.item = (int64_t)blockIdx.x * (kThreads >> lpi_log2) + (threadIdx.x >> lpi_log2);
  m.lane = threadIdx.x & ((1 << lpi_log2) - 1);
  return m;
}

// Raw-tail rows a reconstruction appends to its output (fc_jpeg_view): the
// item after the archived blocks of every sequence copies the n contiguous
// tail tokens behind them.
struct TailRows {
  const void* p = nullptr;
  int64_t sb = 0, sh = 0;  // elements
  int n = 0;
};

// Quantizer of an archive: none (coefficients in the stream dtype), one
// scale per row, one scale per 32 features.
enum JpegMode { kJpegFp = 0, kJpegRow = 1, kJpegGroup = 2 };

// VEC consecutive values rounded to T (to nearest even; a bf16 NaN becomes
// 0x7FC0, as from_f32).  bf16 pairs on the conversion instruction: from_f32's
// integer rounding costs twice the instructions.
template <typename T, int VEC>
__device__ __forceinline__ vec_t<T, VEC> round_row(const float (&v)[VEC]) {
  vec_t<T, VEC> o;
  if constexpr (std::is_same<T, bf16_t>::value) {
#pragma unroll
    for (int i = 0; i < VEC; ++i) {
      const float f = v[i] == v[i] ? v[i] : __uint_as_float(0x7fc00000u);
      o.v[i] = __builtin_bit_cast(bf16_t, (__bf16)f);
    }
  } else {
#pragma unroll
    for (int i = 0; i < VEC; ++i) o.v[i] = from_f32<T>(v[i]);
  }
  return o;
}

// Kernel arguments besides the arrays: kept small, since a call of a few
// microseconds waits for them (see fc_jpeg_decode.hip).
struct JpegEncodeArgs {
  int64_t sb, sh, ss, H, m, D, s_valid, cap, n0, items;
  int k, lpi_log2;
};

struct JpegEncodeLaunch {
  JpegEncodeArgs p;
  const void* x;
  int dtype, r;
  const float* basis;
  void* out;
  float* scales;
  int vec;
  JpegMode mode;
  const int64_t* gate;  // device (n_blocks, n_tail) of a gated decode-step archive, or NULL
  hipStream_t stream;
};

struct JpegDecodeArgs {
  int64_t H, cap, a, nper, D;  // nper: items per sequence (blocks, and the tail's)
  int64_t osb, osh, oss, out_len, items;
  int r, k, lpi_log2;
};

struct JpegDecodeLaunch {
  JpegDecodeArgs p;
  const void* store;
  int in_dtype, out_dtype;
  const float* scales;
  const float* basis;
  void* out;
  int vec;
  JpegMode mode;
  TailRows tail;
  hipStream_t stream;
};

// Whether the register-resident kernels run this shape, and their launches
// (FC_OK, or FC_ERR_UNSUPPORTED for a shape outside them).
int jpeg_vec_fast(int dtype, int vec, int64_t D);
// whole: every block complete (s_valid >= m * r)
bool jpeg_encode_fast_supported(int r, int dtype, int vec, JpegMode mode, bool whole,
                                bool gated);
int jpeg_encode_fast(const JpegEncodeLaunch& a);
bool jpeg_decode_fast_supported(int r, int k, int out_dtype, int vec, JpegMode mode);
int jpeg_decode_fast(const JpegDecodeLaunch& a);

}  // namespace fc
