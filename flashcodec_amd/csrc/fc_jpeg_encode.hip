// Register-resident jpeg archive kernels (blocks of 4, 8 or 16 tokens).
//
// The arithmetic of jpeg_encode_kernel (fc_codec.hip) bit for bit: the same
// fma chain over the taps, the rounding to the stream dtype, scale and codes.
// Bound by HBM: 16 bytes per lane and token row (8 features of 16 bits, 4 of
// fp32), all token loads of a block issued before the first is used, the
// row maximum on DPP instead of LDS-permute shuffles, the divisions replaced
// by exact shortcuts, nontemporal stores (the archive is written once).
// 67 MB of bf16 tokens (4 x 8 x 8192 x 128), general kernel -> this one:
// coefficients k = 2 of 8 20.9 -> 13.8 us (6.1 TB/s), k = 4 of 16 32.2 -> 16.8
// us; int8 per 32 features k = 4 of 8 31 -> 18.7 us; int8 per row k = 4 of 16
// 35.9 -> 18.1 us, k = 2 of 4 28.2 -> 16.6 us, k = 4 of 8 18.3 us (the 8-token
// kernel of before: 18.1 us).
#include "fc_codec_items.h"

namespace fc {

namespace {

// Max over aligned groups of `width` lanes of non-negative, non-NaN floats
// (compared as integers, which orders them the same way): DPP row permutes
// inside 16 lanes (quad swaps, half-row and row mirrors), shuffles beyond.
template <int CTRL>
__device__ __forceinline__ uint32_t dpp_umax(uint32_t v) {
  return max(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xF, 0xF, false));
}
__device__ __forceinline__ float group_amax(float v, int width) {
  uint32_t u = __float_as_uint(v);
  if (width > 1) u = dpp_umax<0xB1>(u);   // quad_perm [1,0,3,2]
  if (width > 2) u = dpp_umax<0x4E>(u);   // quad_perm [2,3,0,1]
  if (width > 4) u = dpp_umax<0x141>(u);  // row_half_mirror
  if (width > 8) u = dpp_umax<0x140>(u);  // row_mirror
  if (width > 16) u = max(u, (uint32_t)__shfl_xor((int)u, 16, 64));
  if (width > 32) u = max(u, (uint32_t)__shfl_xor((int)u, 32, 64));
  return __uint_as_float(u);
}

// fl(a / 127) for every finite a >= 0: y0 = fl(a R) with R = fl(1/127) is
// within an ulp of the quotient, the residual a - 127 y0 is exact in one
// fma, and one correction step rounds correctly (checked exhaustively over
// all 2^31 non-negative finite floats by tests/test_quant_shortcut.py).
__device__ __forceinline__ float div127(float a) {
  constexpr float R = 1.0f / 127.0f;
  const float y0 = a * R;
  const float e = __builtin_fmaf(-y0, 127.0f, a);
  return __builtin_fmaf(e, R, y0);
}

// stream-dtype rounding of a value that is only used again as fp32 (NaN
// stays NaN; the payload is irrelevant here)
template <typename T>
__device__ __forceinline__ float round_trip(float f) {
  if constexpr (std::is_same<T, bf16_t>::value) {
    return (float)(__bf16)f;
  } else {
    return to_f32(from_f32<T>(f));
  }
}

// Smallest normal scale of the stream dtype: with a normal scale the
// row's quotients stay below 127.5 in magnitude (the scale is absmax / 127
// rounded with relative error <= 2^-8), so their rounded values need no
// clamp.
template <typename T>
__device__ __forceinline__ constexpr float min_normal_scale() {
  return std::is_same<T, f16_t>::value ? 0x1p-14f : 0x1p-126f;
}

// Codes of VEC (4 or 8) coefficients of one quantizer row with scale s,
// packed four to a dword; the same codes as quant_code.  rs is the hardware reciprocal
// (relative error <= 2^-23): for |c / s| < 128, x = fl(c rs) lies within
// 1.5 * 2^-16 of c / s and fl(c / s) within 2^-18, so both round to the
// same integer unless x is within 2^-14 of a half-integer.  x + 1.5 * 2^23
// rounds x to an integer held in the low mantissa bits (two's complement
// in the low byte), so one add gives rint(x) and the code byte.  Rows with a
// tie candidate or a scale outside the normal range take the IEEE quotient
// for all its elements (a few rows in a thousand).
template <int VEC>
struct code_words {
  typedef uint32_t type __attribute__((ext_vector_type(VEC / 4)));
};

template <typename T, int VEC>
__device__ __forceinline__ typename code_words<VEC>::type quantize_vec(const float (&c)[VEC],
                                                                       float s) {
  constexpr float kMagic = 0x1.8p23f;
  const bool normal = s >= min_normal_scale<T>() && s <= 0x1p126f;
  const float rs = __builtin_amdgcn_rcpf(s);
  float y[VEC];
  float dm = 0.f;
#pragma unroll
  for (int v = 0; v < VEC; ++v) {
    const float x = c[v] * rs;
    y[v] = x + kMagic;
    dm = fmaxf(dm, fabsf(x - (y[v] - kMagic)));
  }
  // NaN elements (dropped by the max) have NaN y and code 0, as below
  if (!normal || !(dm < 0.5f - 0x1p-14f)) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const float q = __builtin_rintf(c[v] / s);
      y[v] = (q == q ? fminf(fmaxf(q, -127.f), 127.f) : 0.f) + kMagic;
    }
  }
  typename code_words<VEC>::type w;
#pragma unroll
  for (int i = 0; i < VEC / 4; ++i)
    w[i] = __builtin_amdgcn_perm(
        __builtin_amdgcn_perm(__float_as_uint(y[4 * i + 3]), __float_as_uint(y[4 * i + 2]),
                              0x0c0c0400u),
        __builtin_amdgcn_perm(__float_as_uint(y[4 * i + 1]), __float_as_uint(y[4 * i]),
                              0x0c0c0400u),
        0x05040100u);
  return w;
}

// VEC consecutive outputs rounded to T, as nontemporal 16-byte (8-byte) stores.
template <typename T, int VEC>
__device__ __forceinline__ void nt_store_row(T* p, const float (&v)[VEC]) {
  typedef uint32_t w4 __attribute__((ext_vector_type(4)));
  typedef uint32_t w2 __attribute__((ext_vector_type(2)));
  const vec_t<T, VEC> o = round_row<T, VEC>(v);
  if constexpr (sizeof(o) == 32) {
    struct Two { w4 a, b; };
    const Two t = __builtin_bit_cast(Two, o);
    __builtin_nontemporal_store(t.a, reinterpret_cast<w4*>(p));
    __builtin_nontemporal_store(t.b, reinterpret_cast<w4*>(p) + 1);
  } else if constexpr (sizeof(o) == 16) {
    __builtin_nontemporal_store(__builtin_bit_cast(w4, o), reinterpret_cast<w4*>(p));
  } else {
    __builtin_nontemporal_store(__builtin_bit_cast(w2, o), reinterpret_cast<w2*>(p));
  }
}

// KT: kept frequencies, 0 = runtime k.  The arrays come as restrict arguments
// besides the launch description, so that the basis stays in scalar registers
// across the stores.  Tokens at or past s_valid (the padded
// end of the last block, coefficients only: streams archive whole blocks)
// are zero.
template <typename T, int VEC, int R, int KT, JpegMode MODE, bool GATED>
__global__ __launch_bounds__(kThreads) void jpeg_encode_fast_kernel(
    const T* __restrict__ x, const float* __restrict__ basis, void* __restrict__ out,
    float* __restrict__ scales, JpegEncodeArgs p, const int64_t* __restrict__ gate) {
  int64_t n0 = p.n0;
  if constexpr (GATED) {
    // gate = device (n_blocks, n_tail): archive only a completed tail
    if (gate[1] != R - 1) return;
    n0 = gate[0];
    if (n0 < 0 || n0 + p.m > p.cap) return;
  }
  const int k = KT > 0 ? KT : p.k;
  const ItemMap im = item_of_thread(p.lpi_log2);
  // lanes without work still take part in the row maximum: they hold zeros
  // and store nothing
  const bool live = im.item < p.items;
  const int64_t item = live ? im.item : 0;
  const int64_t bh = item / p.m, blk = item - bh * p.m;
  const int64_t b = bh / p.H, h = bh - b * p.H;
  const int64_t d0 = (int64_t)im.lane * VEC;
  const bool active = live && d0 < p.D;
  const int64_t tok0 = blk * R;
  const T* src = x + b * p.sb + h * p.sh + tok0 * p.ss + (active ? d0 : 0);

  // All R token loads are issued before any of them is consumed (the
  // scheduling barrier keeps the backend from waiting on the first load to
  // widen it while the others are still unissued).
  vec_t<T, VEC> raw[R];
  if (active && (MODE != kJpegFp || tok0 + R <= p.s_valid)) {
#pragma unroll
    for (int t = 0; t < R; ++t) raw[t] = *reinterpret_cast<const vec_t<T, VEC>*>(src + t * p.ss);
  } else {
#pragma unroll
    for (int t = 0; t < R; ++t) {
      if (MODE == kJpegFp && active && tok0 + t < p.s_valid) {
        raw[t] = *reinterpret_cast<const vec_t<T, VEC>*>(src + t * p.ss);
      } else {
#pragma unroll
        for (int v = 0; v < VEC; ++v) raw[t].v[v] = from_f32<T>(0.f);
      }
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  float xr[R][VEC];
#pragma unroll
  for (int t = 0; t < R; ++t)
#pragma unroll
    for (int v = 0; v < VEC; ++v) xr[t][v] = to_f32(raw[t].v[v]);

  const int64_t row0 = (bh * p.cap + n0 + blk) * k;
  const int width = MODE == kJpegGroup ? 32 / VEC : 1 << p.lpi_log2;  // lanes of a scale
#pragma unroll
  for (int j = 0; j < k; ++j) {
    const float* mj = basis + j * R;
    float c[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) c[v] = 0.f;
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const float w = mj[t];
#pragma unroll
      for (int v = 0; v < VEC; ++v) c[v] = __builtin_fmaf(xr[t][v], w, c[v]);
    }
    if constexpr (MODE == kJpegFp) {
      if (active) nt_store_row<T, VEC>(static_cast<T*>(out) + (row0 + j) * p.D + d0, c);
      continue;
    }
    float amax = 0.f;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      c[v] = round_trip<T>(c[v]);
      amax = fmaxf(amax, fabsf(c[v]));
    }
    amax = group_amax(amax, width);
    float s = round_trip<T>(amax <= 0x1.fffffep127f ? div127(amax) : amax / 127.0f);
    if (!(s > 0.f)) s = 1.0f;
    const auto qv = quantize_vec<T, VEC>(c, s);
    if (active) {
      typedef typename code_words<VEC>::type W;
      __builtin_nontemporal_store(
          qv, reinterpret_cast<W*>(static_cast<int8_t*>(out) + (row0 + j) * p.D + d0));
      if ((im.lane & (width - 1)) == 0)
        __builtin_nontemporal_store(
            s, MODE == kJpegGroup ? scales + (row0 + j) * (p.D / 32) + d0 / 32
                                  : scales + row0 + j);
    }
  }
}

template <typename T, int VEC, int R, JpegMode MODE, bool GATED>
void launch(const JpegEncodeLaunch& a) {
  const int64_t per = kThreads >> a.p.lpi_log2;
  const dim3 grid((unsigned)((a.p.items + per - 1) / per));
  if (a.p.k == 2)
    jpeg_encode_fast_kernel<T, VEC, R, 2, MODE, GATED><<<grid, kThreads, 0, a.stream>>>(
        static_cast<const T*>(a.x), a.basis, a.out, a.scales, a.p, a.gate);
  else if (a.p.k == 4)
    jpeg_encode_fast_kernel<T, VEC, R, 4, MODE, GATED><<<grid, kThreads, 0, a.stream>>>(
        static_cast<const T*>(a.x), a.basis, a.out, a.scales, a.p, a.gate);
  else if (R == 8 && MODE == kJpegRow && a.p.k == 8)
    jpeg_encode_fast_kernel<T, VEC, 8, 8, kJpegRow, GATED><<<grid, kThreads, 0, a.stream>>>(
        static_cast<const T*>(a.x), a.basis, a.out, a.scales, a.p, a.gate);
  else
    jpeg_encode_fast_kernel<T, VEC, R, 0, MODE, GATED><<<grid, kThreads, 0, a.stream>>>(
        static_cast<const T*>(a.x), a.basis, a.out, a.scales, a.p, a.gate);
}

template <typename T, int VEC>
int launch_type(const JpegEncodeLaunch& a) {
  if constexpr (sizeof(T) * VEC == 32) {  // fp32 rows of more than 64 lanes x 4
    if (a.gate)
      launch<T, VEC, 8, kJpegRow, true>(a);
    else
      launch<T, VEC, 8, kJpegRow, false>(a);
    return FC_OK;
  }
  if (a.gate) {  // gated: the int8 row quantizer on 8-token blocks
    launch<T, VEC, 8, kJpegRow, true>(a);
    return FC_OK;
  }
  auto with_mode = [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    switch (a.mode) {
      case kJpegFp: launch<T, VEC, R, kJpegFp, false>(a); break;
      case kJpegRow: launch<T, VEC, R, kJpegRow, false>(a); break;
      default: launch<T, VEC, R, kJpegGroup, false>(a); break;
    }
    return FC_OK;
  };
  switch (a.r) {
    case 4: return with_mode(std::integral_constant<int, 4>{});
    case 8: return with_mode(std::integral_constant<int, 8>{});
    case 16: return with_mode(std::integral_constant<int, 16>{});
    default: return FC_ERR_UNSUPPORTED;
  }
}

}  // namespace

// Elements per lane of the register-resident kernels for rows the general
// kernels would take `vec` elements of: 16 bytes.
int jpeg_vec_fast(int dtype, int vec, int64_t D) {
  return vec == 8 && dtype == FC_F32 && D <= 256 ? 4 : vec;
}

bool jpeg_encode_fast_supported(int r, int dtype, int vec, JpegMode mode, bool whole,
                                bool gated) {
  if (!whole && mode != kJpegFp) return false;
  if (gated || (dtype == FC_F32 && vec == 8))
    return r == 8 && mode == kJpegRow && (vec == 8 || dtype == FC_F32) && vec >= 4;
  return (r == 4 || r == 8 || r == 16) && vec == (dtype == FC_F32 ? 4 : 8);
}

int jpeg_encode_fast(const JpegEncodeLaunch& a) {
  switch (a.dtype) {
    case FC_F32: return a.vec == 8 ? launch_type<float, 8>(a) : launch_type<float, 4>(a);
    case FC_F16: return launch_type<f16_t, 8>(a);
    case FC_BF16: return launch_type<bf16_t, 8>(a);
    default: return FC_ERR_ARG;
  }
}

}  // namespace fc
