// Register-resident jpeg reconstruction kernels (up to 8 kept frequencies).
//
// The products and fma order of jpeg_decode_kernel (fc_codec.hip) bit for
// bit.  Bound by HBM, mostly by the reconstructed rows' writes: the k code or
// coefficient rows and scales of a block are all requested before the first
// is used, the tokens formed 8 at a time (64 or 32 accumulators, so blocks of
// any size fit the registers), rows written with nontemporal stores.
// Small calls wait for the kernel's arguments and its first loads: the
// arguments are few, and the tail rows of a view are a variant of their own
// (with both at run time calls of 3-5 us took 3% longer).  Stored rows are
// unrolled, except above 4 in blocks of 16 or of other sizes: guards on a
// runtime count held k = 8 of 8 bf16 coefficients at 18.5 us for 34 MB of
// tokens, 13.4 now, the general kernel 17.3 (in the caches 14.2, 9.4, 14.6).
// 34 MB of bf16 tokens (32 x 4096 x 128), general kernel -> this one, archive
// not in the caches: coefficients k = 2 of 8 11.4 -> 8.2 us, k = 4 13.7 -> 9.5,
// k = 4 of 16 14.2 -> 10.0; int8 per row k = 4 of 16 16.9 -> 11.7, per 32
// features k = 4 of 8 16.3 -> 12.1.
#include "fc_codec_items.h"

namespace fc {

namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

struct NoTail {};

template <int BYTES>
struct nt_word {
  typedef uint32_t type __attribute__((ext_vector_type(BYTES / 4)));
};

// VEC consecutive outputs of one token row, rounded to TO and written with
// nontemporal stores
template <typename TO, int VEC>
__device__ __forceinline__ void nt_store_row(TO* p, const float (&v)[VEC]) {
  const vec_t<TO, VEC> o = round_row<TO, VEC>(v);
  if constexpr (sizeof(o) == 32) {
    struct Two { u32x4 a, b; };
    const Two t = __builtin_bit_cast(Two, o);
    __builtin_nontemporal_store(t.a, reinterpret_cast<u32x4*>(p));
    __builtin_nontemporal_store(t.b, reinterpret_cast<u32x4*>(p) + 1);
  } else {
    typedef typename nt_word<sizeof(o)>::type W;
    __builtin_nontemporal_store(__builtin_bit_cast(W, o), reinterpret_cast<W*>(p));
  }
}

// R: tokens per block, 0 = runtime r (tokens formed 8 at a time); KT: kept
// frequencies, 0 = runtime k <= 8.  The arrays come as restrict arguments
// besides the launch description (loads ahead of the stores).
template <typename TI, typename TO, int VEC, int R, int KT, bool GROUP, bool TAIL>
__global__ __launch_bounds__(kThreads) void jpeg_decode_fast_kernel(
    const TI* __restrict__ store, const float* __restrict__ scales,
    const float* __restrict__ basis, TO* __restrict__ out, JpegDecodeArgs p,
    std::conditional_t<TAIL, TailRows, NoTail> tail) {
  constexpr bool QUANT = std::is_same<TI, int8_t>::value;
  constexpr int KMAX = KT > 0 ? KT : 8;
  constexpr int TB = R > 0 && R < 8 ? R : 8;  // tokens formed at a time
  const int k = KT > 0 ? KT : p.k;
  const int r = R > 0 ? R : p.r;
  const ItemMap im = item_of_thread(p.lpi_log2);
  if (im.item >= p.items) return;
  const int64_t bh = im.item / p.nper, rel = im.item - bh * p.nper, blk = p.a + rel;
  const int64_t b = bh / p.H, h = bh - b * p.H;
  const int64_t d0 = (int64_t)im.lane * VEC;
  if (d0 >= p.D) return;
  TO* const seq = out + b * p.osb + h * p.osh + d0;
  const int64_t tok0 = blk * r;
  if constexpr (TAIL) {
    if (rel + 1 == p.nper) {
      const TO* src = static_cast<const TO*>(tail.p) + b * tail.sb + h * tail.sh + d0;
      for (int t = 0; t < tail.n; ++t)
        *reinterpret_cast<vec_t<TO, VEC>*>(seq + (tok0 + t) * p.oss) =
            *reinterpret_cast<const vec_t<TO, VEC>*>(src + t * p.D);
      return;
    }
  }
  const int64_t row0 = (bh * p.cap + blk) * k;
  const TI* src = store + row0 * p.D + d0;

  // rows are read past the caches: 2-9% faster than with ordinary loads, more
  // for many codes (67 MB of bf16 tokens, int8 k = 8 of 8, 23.8 us for 28.6)
  typedef typename nt_word<sizeof(vec_t<TI, VEC>)>::type W;
  W q[KMAX];
  float s[KMAX];
#pragma unroll
  for (int j = 0; j < KMAX; ++j) {
    if (j < k) {
      q[j] = __builtin_nontemporal_load(reinterpret_cast<const W*>(src + (int64_t)j * p.D));
      if constexpr (QUANT)
        s[j] = GROUP ? scales[(row0 + j) * (p.D / 32) + d0 / 32] : scales[row0 + j];
    }
  }
  __builtin_amdgcn_sched_barrier(0);

#pragma unroll
  for (int t0 = 0; t0 < r; t0 += TB) {
    float acc[TB][VEC];
#pragma unroll
    for (int t = 0; t < TB; ++t)
#pragma unroll
      for (int v = 0; v < VEC; ++v) acc[t][v] = 0.f;
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
      if (j < k) {
        // (more than 4 rows: the conversion stays with its tokens, hoisted past
        // them it takes 64 registers)
        if constexpr (KMAX > 4 && R != 8) {
#pragma unroll
          for (int i = 0; i < (int)(sizeof(W) / 4); ++i) {
            uint32_t x = q[j][i];
            asm("" : "+v"(x));
            q[j][i] = x;
          }
        }
        const vec_t<TI, VEC> row = __builtin_bit_cast(vec_t<TI, VEC>, q[j]);
        float c[VEC];
#pragma unroll
        for (int v = 0; v < VEC; ++v) c[v] = QUANT ? to_f32(row.v[v]) * s[j] : to_f32(row.v[v]);
        const float* mj = basis + j * r + t0;
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          if (R > 0 || t0 + t < r) {
            const float w = mj[t];
#pragma unroll
            for (int v = 0; v < VEC; ++v) acc[t][v] = __builtin_fmaf(c[v], w, acc[t][v]);
          }
        }
      }
    }
#pragma unroll
    for (int t = 0; t < TB; ++t)
      if ((R > 0 || t0 + t < r) && tok0 + t0 + t < p.out_len)
        nt_store_row<TO, VEC>(seq + (tok0 + t0 + t) * p.oss, acc[t]);
  }
}

template <typename TI, typename TO, int VEC, bool GROUP>
void launch(const JpegDecodeLaunch& a) {
  const int64_t per = kThreads >> a.p.lpi_log2;
  const dim3 grid((unsigned)((a.p.items + per - 1) / per));
  auto go = [&](auto rc, auto kc) {
    constexpr int R = decltype(rc)::value, KT = decltype(kc)::value;
    const TI* store = static_cast<const TI*>(a.store);
    TO* out = static_cast<TO*>(a.out);
    // (a view is in the stream dtype: int8 codes, or rows of the same type)
    if constexpr (std::is_same<TI, int8_t>::value || std::is_same<TI, TO>::value) {
      if (a.tail.n) {
        jpeg_decode_fast_kernel<TI, TO, VEC, R, KT, GROUP, true>
            <<<grid, kThreads, 0, a.stream>>>(store, a.scales, a.basis, out, a.p, a.tail);
        return;
      }
    }
    jpeg_decode_fast_kernel<TI, TO, VEC, R, KT, GROUP, false>
        <<<grid, kThreads, 0, a.stream>>>(store, a.scales, a.basis, out, a.p, NoTail{});
  };
  using std::integral_constant;
  auto with_k = [&](auto rc) {
    constexpr int R = decltype(rc)::value;
    switch (a.p.k) {
      case 1: return go(rc, integral_constant<int, 1>{});
      case 2: return go(rc, integral_constant<int, 2>{});
      case 3: return go(rc, integral_constant<int, 3>{});
      case 4: return go(rc, integral_constant<int, 4>{});
      default: break;
    }
    if constexpr (R == 8) {
      switch (a.p.k) {
        case 5: return go(rc, integral_constant<int, 5>{});
        case 6: return go(rc, integral_constant<int, 6>{});
        case 7: return go(rc, integral_constant<int, 7>{});
        default: return go(rc, integral_constant<int, 8>{});
      }
    } else if constexpr (R != 4) {
      go(rc, integral_constant<int, 0>{});
    }
  };
  switch (a.p.r) {
    case 4: with_k(integral_constant<int, 4>{}); break;
    case 8: with_k(integral_constant<int, 8>{}); break;
    case 16: with_k(integral_constant<int, 16>{}); break;
    default: with_k(integral_constant<int, 0>{}); break;
  }
}

template <typename TO, int VEC>
int launch_out(const JpegDecodeLaunch& a) {
  if constexpr (sizeof(TO) * VEC == 32) {  // fp32 rows of more than 64 lanes x 4
    launch<int8_t, TO, VEC, false>(a);
  } else if (a.mode == kJpegRow) {
    launch<int8_t, TO, VEC, false>(a);
  } else if (a.mode == kJpegGroup) {
    launch<int8_t, TO, VEC, true>(a);
  } else if (a.in_dtype == a.out_dtype) {
    launch<TO, TO, VEC, false>(a);
  } else if constexpr (std::is_same<TO, float>::value) {  // 16-bit coefficients to fp32 tokens
    if (a.in_dtype == FC_F16)
      launch<f16_t, float, VEC, false>(a);
    else
      launch<bf16_t, float, VEC, false>(a);
  } else {
    return FC_ERR_UNSUPPORTED;
  }
  return FC_OK;
}

}  // namespace

// fp32 tokens of 16-token blocks with 1 stored row keep the general kernel
// and its plain stores: 67 MB of tokens at D = 256 take 23.5 us there, 26.5
// here, 2 MB 4.1 both (k = 2: 24.2 and 25, 2 MB 5.0 and 3.7).
bool jpeg_decode_fast_supported(int r, int k, int out_dtype, int vec, JpegMode mode) {
  if (k > 8) return false;
  if (out_dtype != FC_F32) return vec == 8;
  if (vec == 8) return mode == kJpegRow;  // rows of more than 64 lanes x 4
  return vec == 4 && !(r == 16 && k == 1);
}

int jpeg_decode_fast(const JpegDecodeLaunch& a) {
  switch (a.out_dtype) {
    case FC_F32: return a.vec == 8 ? launch_out<float, 8>(a) : launch_out<float, 4>(a);
    case FC_F16: return launch_out<f16_t, 8>(a);
    case FC_BF16: return launch_out<bf16_t, 8>(a);
    default: return FC_ERR_ARG;
  }
}

}  // namespace fc
