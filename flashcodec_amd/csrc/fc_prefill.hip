// Causal prefill attention over an int8 jpeg archive without the
// reconstructed view: the entry point, and the kernel variants with the
// vector-ALU softmax (the kernel and its description: fc_prefill_kernel.h).
#include "fc_prefill_kernel.h"
#include "fc_prefill_wg.h"

namespace fc {

template int launch_prefill<1, 0>(const PrefillArgs&, int, int, int, bool, unsigned, hipStream_t);
template int launch_prefill<2, 0>(const PrefillArgs&, int, int, int, bool, unsigned, hipStream_t);
template int launch_prefill<4, 0>(const PrefillArgs&, int, int, int, bool, unsigned, hipStream_t);

// Query heads of a wavefront's 16 queries.
static int prefill_heads_per_wave(int64_t G) {
  int gq = 1;
  while (gq < 16 && G % (2 * gq) == 0) gq *= 2;
  return gq;
}

// Compute units of the current device, 0 if it does not say.
static int device_cus() {
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess)
    return n;
  (void)hipGetLastError();
  return 0;
}

}  // namespace fc

using namespace fc;

extern "C" {

// The workgroup-shared pass takes D = 64 / 128 and blocks of 4 or 8 tokens (at
// 16 its 3-wavefront register budget spills and the register-resident pass
// is faster: 1326 vs 1542 us at 16 x 16 heads x 4096 tokens, D = 128).  With
// a scale per 32 features at D = 128 it needs two workgroups on some compute
// units: with one on each it waits at its barriers and LDS round trips (256
// workgroups, 9192 tokens, 197 us, the register-resident pass 176; 288: 240 and
// 268; 512: 245 and 270; 1008: 433 and 499).  The grid counts in longest tiles,
// since its end runs with fewer: a whole prompt of 4096 tokens in 512
// workgroups (260 of the longest) takes 101 us, in registers 96; 1000 on 300
// (315) 49.1 and 45.0; 1000 on 1000 (381) 64 and 69.
// Under 6 passes its longer start counts (485 of 300 tokens 27.6 us, in registers
// 25.3; 960 of 130 19.3 and 21.0), and wavefronts without tokens load for
// the others there, which in registers leave (1024 workgroups, 5 of 8 wavefronts
// with tokens, 1024 tokens: 73.5 and 62.4; 17 of 20, 1280: 62 and 73).
// D = 64 is as fast or faster shared at every grid (0-58%) but for such short,
// part-filled ones (512 workgroups, 2 of 4 wavefronts, 130 tokens 15.5 and 14.1).
int fc_prefill_shared_pass(int store_kind, int r, int s, int64_t D, int64_t B, int64_t Hkv,
                           int64_t G, int64_t Sq, int64_t P0, int n_cu) {
  if (B <= 0 || Hkv <= 0 || G <= 0 || Sq <= 0 || P0 < 0) return 0;
  if (s != 4 || (D != 64 && D != 128) || (r != 4 && r != 8)) return 0;
  if (store_kind != FC_STORE_JPEG_I8G) return store_kind == FC_STORE_JPEG_I8;
  if (n_cu <= 0) n_cu = 256;
  const int64_t gq = prefill_heads_per_wave(G), tq = 16 / gq, tile = 4 * tq;
  const int64_t nt = (Sq + tile - 1) / tile, cols = G / gq * Hkv * B;
  const int64_t waves = (Sq + tq - 1) / tq;  // with tokens, of 4 nt
  const int64_t passes = (P0 + Sq) / (16 * r);
  if (D == 64) return waves > 2 * nt || passes >= 2 || nt * cols <= n_cu;
  const bool filled = passes >= 6 ? 5 * waves >= 16 * nt : 3 * waves >= 10 * nt;  // 4/5, 5/6
  const double work = (double)nt * P0 + 0.5 * tile * nt * (nt - 1) + Sq;  // tokens of all tiles
  // longest tiles per unit: more where the tiles differ more
  const double f = (double)Sq / (double)(P0 + Sq);
  const double need = passes >= 6 ? 1.03125 + 0.375 * f * f : 3.625;
  return filled && work * cols >= need * n_cu * (double)(P0 + Sq);
}

int fc_prefill_attention(const void* q, int q_dtype, int64_t q_sb, int64_t q_sh, int64_t q_st,
                         int64_t B, int64_t Hq, int64_t Hkv, int64_t Sq, int64_t D, int64_t P0,
                         int stream_dtype, int store_kind, int r, int s, int64_t nb,
                         const fc_stream_view* key, const fc_stream_view* value, int64_t n_raw,
                         const float* A, float scale, void* out, int64_t o_sb, int64_t o_sh,
                         int64_t o_st, void* stream) {
  if (!q || !out || !key || !value || B <= 0 || Hq <= 0 || Hkv <= 0 || Sq <= 0 || Hq % Hkv)
    return FC_ERR_ARG;
  if (nb < 0 || n_raw < 0 || P0 < 0 || r < 1 || r > FC_MAX_BLOCK || s < 1 || s > r)
    return FC_ERR_ARG;
  if (P0 + Sq > nb * r + n_raw) return FC_ERR_ARG;  // every query is a cached token
  if (q_dtype != FC_F16 && q_dtype != FC_BF16) return FC_ERR_UNSUPPORTED;
  if (!(D == 64 || D == 128 || D == 256) || !(s == 1 || s == 2 || s == 4))
    return FC_ERR_UNSUPPORTED;
  if (stream_dtype != FC_F16 && stream_dtype != FC_BF16 && stream_dtype != FC_F32)
    return FC_ERR_ARG;
  if (store_kind != FC_STORE_JPEG_I8 && store_kind != FC_STORE_JPEG_I8G) return FC_ERR_ARG;
  const bool grouped = store_kind == FC_STORE_JPEG_I8G;
  if (nb > 0 && (!A || !key->rows || !value->rows || !key->scales || !value->scales ||
                 nb > key->cap || nb > value->cap))
    return FC_ERR_ARG;
  if (n_raw > 0 && (!key->raw || !value->raw)) return FC_ERR_ARG;
  const auto al16 = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; };
  if (!al16(q) || q_sb % 8 || q_sh % 8 || q_st % 8 || !al16(key->rows) || !al16(value->rows))
    return FC_ERR_UNSUPPORTED;
  // per-32 scales are read in 8 / 16-byte pieces per row
  if (grouped && nb > 0 && (!al16(key->scales) || !al16(value->scales))) return FC_ERR_UNSUPPORTED;
  const int64_t G = Hq / Hkv;
  PrefillArgs a{};
  a.q = q;
  a.q_dtype = q_dtype;
  a.q_sb = q_sb;
  a.q_sh = q_sh;
  a.q_st = q_st;
  a.Sq = Sq;
  a.P0 = P0;
  a.kcodes = static_cast<const int8_t*>(key->rows);
  a.kscales = key->scales;
  a.vcodes = static_cast<const int8_t*>(value->rows);
  a.vscales = value->scales;
  a.kcap = key->cap;
  a.vcap = value->cap;
  a.A = A;
  a.Hkv = Hkv;
  a.G = G;
  a.nb = nb;
  a.r = r;
  a.scale_log2 = scale * 1.4426950408889634f;
  a.kraw = key->raw;
  a.vraw = value->raw;
  a.kr_sb = key->raw_sb;
  a.kr_sh = key->raw_sh;
  a.kr_st = key->raw_st;
  a.vr_sb = value->raw_sb;
  a.vr_sh = value->raw_sh;
  a.vr_st = value->raw_st;
  a.n_raw = n_raw;
  a.out = out;
  a.o_sb = o_sb;
  a.o_sh = o_sh;
  a.o_st = o_st;
  // a wavefront's 16 queries: the largest power-of-two head count <= 16
  // that divides G, times 16 / that many consecutive tokens
  const int gq = prefill_heads_per_wave(G);
  a.gq = gq;
  a.tq = 16 / gq;
  a.hgroups = G / gq;
  a.ntiles = (Sq + 4 * a.tq - 1) / (4 * a.tq);
  const int64_t blocks = a.ntiles * a.hgroups * Hkv * B;
  if (blocks > 0x7fffffff) return FC_ERR_UNSUPPORTED;
  hipStream_t st = (hipStream_t)stream;
  const int dk = (int)(D / 32);
  const unsigned nblocks = (unsigned)blocks;
  int rc;
  // 4 stored rows per block of 4, 8 or 16 tokens: the softmax on the matrix
  // cores (one 4x4 product per block), each pass shared by the workgroup or in
  // registers
  const bool wg = n_raw < r && fc_prefill_shared_pass(store_kind, r, s, D, B, Hkv, G, Sq, P0,
                                                      grouped ? device_cus() : 0) == 1;
  if (wg && r == 8)
    rc = launch_prefill_wg<8>(a, dk, q_dtype, stream_dtype, grouped, nblocks, st);
  else if (wg && r == 4)
    rc = launch_prefill_wg<4>(a, dk, q_dtype, stream_dtype, grouped, nblocks, st);
  else if (s == 4 && r == 8)
    rc = launch_prefill<4, 8>(a, dk, q_dtype, stream_dtype, grouped, nblocks, st);
  else if (s == 4 && r == 4)
    rc = launch_prefill<4, 4>(a, dk, q_dtype, stream_dtype, grouped, nblocks, st);
  else if (s == 4 && r == 16)
    rc = launch_prefill<4, 16>(a, dk, q_dtype, stream_dtype, grouped, nblocks, st);
  else
    rc = prefill_with_int<1, 2, 4>(s, [&](auto sc) {
      return launch_prefill<decltype(sc)::value, 0>(a, dk, q_dtype, stream_dtype, grouped,
                                                     nblocks, st);
    });
  if (rc != FC_OK) return rc;
  return check_launch();
}

}  // extern "C"
