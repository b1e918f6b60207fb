// One low-bit Linear call per entry point: the launches of a forward, of its
// straight-through backward and of the quantized-gradient backward, issued
// from one host call over the codes of X and of W and one scratch buffer
// (te_backend.py:229-260 and its autograd; the recipe of benchmark config 3).
// The device work is that of the separate entry points; what this file adds
// on the device is the zeroing of the NaN row flags (int grid only, one
// launch for all of them) and the padded copy of a dY whose rows are not whole
// 64-column steps.
//
// NaN row flags: an int-grid code of -128 is an ordinary number to the matrix
// cores, so the GEMM needs flags.  e4m3 codes carry NaN themselves (0x7F): the
// MFMA's result is NaN wherever an operand row or column holds one, which is
// what the flags would write, so e4m3 products run without them.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ntlb_device.h"
#include "ntlb_gemm_bf16.h"
#include "ntlb_host.h"

namespace ntlb {

// p [n] and p2 [n2] cleared
__global__ void __launch_bounds__(256) zero_words_kernel(uint32_t* p, int64_t n, uint32_t* p2, int64_t n2) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n)
    p[i] = 0u;
  else if (i < n + n2)
    p2[i - n] = 0u;
}

// dst [M, ldd] (ldd % 8 == 0, 16-byte aligned) = src [M, N] of 16-bit values,
// zero past column N.  Eight columns per thread; bound by its 2-byte loads'
// issue when the rows are not aligned (they are not when this runs).
__global__ void __launch_bounds__(256) pad_rows16_kernel(const uint16_t* src, int64_t lds, int64_t M, int64_t N,
                                                         uint16_t* dst, int64_t ldd) {
  const int64_t per = ldd >> 3;
  const int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= M * per) return;
  const int64_t m = q / per, c = (q - m * per) * 8;
  const uint16_t* s = src + m * lds + c;
  uint32_t w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t lo = c + 2 * i < N ? s[2 * i] : 0u, hi = c + 2 * i + 1 < N ? s[2 * i + 1] : 0u;
    w[i] = lo | (hi << 16);
  }
  *reinterpret_cast<uint4*>(dst + m * ldd + c) = make_uint4(w[0], w[1], w[2], w[3]);
}

// The bf16 operands of small straight-through gradients, bf16(q * s) from the
// forward's codes: weight rows (one scale per 128x128 block) into wd, then
// activation rows (one per row and block) into xd, both with row pitch ld = K
// rounded up to 8; either can be absent (0 rows).  A workgroup of the gradient
// GEMMs' 256x256 tiles decodes inside the GEMM; on 16x16 to 128x128 tiles each
// code would be decoded again by every tile that reads it, and this one pass
// over a few MB costs less (N 1541, K 1000, 1003 rows: about 3 us).
struct DecodeArgs {
  const uint8_t* wc;
  const float* ws;
  const uint8_t* xc;
  const float* xs;
  int64_t wrows, xrows, kp, T, m4, ld;
  uint16_t *wd, *xd;
};

template <int GRID>
__global__ void __launch_bounds__(256) decode_operands_kernel(DecodeArgs a) {
#pragma clang fp contract(off)
  typedef float v2f __attribute__((ext_vector_type(2)));
  const int64_t per = a.ld >> 3, q = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (q >= (a.wrows + a.xrows) * per) return;
  int64_t r = q / per;
  const int64_t c = (q - r * per) * 8;
  const bool is_w = r < a.wrows;
  if (!is_w) r -= a.wrows;
  const uint2 w = *reinterpret_cast<const uint2*>((is_w ? a.wc : a.xc) + r * a.kp + c);
  const float s = is_w ? a.ws[(r >> 7) * a.T + (c >> 7)] : a.xs[(c >> 7) * a.m4 + r];
  const uint32_t words[2] = {w.x, w.y};
  uint32_t out[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    float v[4];
    if constexpr (GRID == GRID_E4M3) {
      const v2f lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)words[h], false);
      const v2f hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)words[h], true);
      v[0] = lo[0] * s; v[1] = lo[1] * s; v[2] = hi[0] * s; v[3] = hi[1] * s;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int code = (int)(int8_t)(uint8_t)(words[h] >> (8 * i));
        v[i] = code == -128 ? __uint_as_float(0x7FC00000u) : (float)code * s;
      }
    }
    out[2 * h] = (uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16);
    out[2 * h + 1] = (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16);
  }
  *reinterpret_cast<uint4*>((is_w ? a.wd : a.xd) + r * a.ld + c) = make_uint4(out[0], out[1], out[2], out[3]);
}

static int64_t up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// consecutive 256-byte aligned pieces of a buffer
struct Carve {
  int64_t at = 0;
  int64_t take(int64_t bytes) {
    const int64_t o = at;
    at += up(bytes, 256);
    return o;
  }
};

// the code buffers of X and of W, apart so that each can be kept as long as
// its gradient needs it: codes, scales, and the NaN flags of the rows (int
// grid; -1: none)
struct CodeLayout {
  int64_t c, s, flags, bytes;
};
static CodeLayout x_layout(const ntlb_linear_plan& p) {
  const int64_t kp = up(p.K, 128);
  Carve c;
  CodeLayout l;
  l.c = c.take(p.M * kp);
  l.s = c.take(kp / 128 * up(p.M, 4) * 4);
  l.flags = p.grid == NTLB_GRID_INT ? c.take(p.M * 4) : -1;
  l.bytes = c.at;
  return l;
}
static CodeLayout w_layout(const ntlb_linear_plan& p) {
  const int64_t kp = up(p.K, 128);
  Carve c;
  CodeLayout l;
  l.c = c.take(p.N * kp);
  l.s = c.take(cdiv(p.N, 128) * (kp / 128) * 4);
  l.flags = p.grid == NTLB_GRID_INT ? c.take(p.N * 4) : -1;
  l.bytes = c.at;
  return l;
}

// the straight-through backward's scratch: the column sum's partials, the
// decoded operands of the gradients that run on tiles below 256x256 (-1: the
// GEMM decodes), and the padded dY (only touched where dY needs it)
struct SteLayout {
  int64_t colsum, wd, xd, dy, bytes;
  Bf16Plan dx, dw;     // their tiles
  int64_t near_pitch;  // the widest row pitch of dY that those tiles take: beyond it 32-bit offsets could overflow
};
static SteLayout ste_layout(const ntlb_linear_plan& p) {
  Carve c;
  SteLayout l;
  l.near_pitch = up(p.N, 64) + 8;
  const int64_t k8 = up(p.K, 8), lim = (int64_t)0x7FFFFFFF;
  l.dx = bf16_small_plan(p.M, p.K, up(p.N, 64), true);
  l.dw = bf16_small_plan(p.N, p.K, up(p.M, 64), false);
  const bool small_dx = l.dx.fits() && (p.M + 256) * l.near_pitch * 2 < lim &&
                        (p.N + 64) * k8 * 2 < lim;
  const bool small_dw = l.dw.fits() && (p.M + 64) * l.near_pitch * 2 < lim &&
                        (p.M + 64) * k8 * 2 < lim;
  l.colsum = c.take(std::max<int64_t>(ntlb_colsum_workspace_bytes(p.M, p.N), 4));
  l.wd = small_dx ? c.take(p.N * k8 * 2) : -1;
  l.xd = small_dw ? c.take(p.M * k8 * 2) : -1;
  l.dy = c.take(p.M * up(p.N, 64) * 2);
  l.bytes = c.at;
  return l;
}

// the recipe backward's scratch
struct RecipeLayout {
  int64_t colsum, yc, ys, ytc, yts, wc, wtc, ws, xtc, xts, flags, bytes;
};
static RecipeLayout recipe_layout(const ntlb_linear_plan& p) {
  const int64_t kp = up(p.K, 128), np = up(p.N, 128), mp = up(p.M, 128);
  Carve c;
  RecipeLayout l;
  l.colsum = c.take(std::max<int64_t>(ntlb_colsum_workspace_bytes(p.M, p.N), 4));
  l.yc = c.take(p.M * np);
  l.ys = c.take(np / 128 * up(p.M, 4) * 4);
  l.ytc = c.take(p.N * mp);
  l.yts = c.take(mp / 128 * up(p.N, 4) * 4);
  l.wc = c.take(p.N * kp);
  l.wtc = c.take(p.K * np);
  l.ws = c.take(np / 128 * (kp / 128) * 4);
  l.xtc = c.take(p.K * mp);
  l.xts = c.take(mp / 128 * up(p.K, 4) * 4);
  l.flags = p.grid == NTLB_GRID_INT ? c.take((p.M + p.N + p.K) * 4) : -1;
  l.bytes = c.at;
  return l;
}

static int check_plan(const char* fn, const ntlb_linear_plan* p) {
  if (!p) return fail(NTLB_EINVAL, "%s: NULL plan", fn);
  if (p->M < 1 || p->N < 1 || p->K < 1 || p->ldx < p->K || p->ldw < p->K)
    return fail(NTLB_EINVAL, "%s: bad shape or row pitch", fn);
  if (!valid_dtype(p->x_dtype) || !valid_dtype(p->w_dtype)) return fail(NTLB_EINVAL, "%s: bad dtype", fn);
  if (p->grid != NTLB_GRID_INT && p->grid != NTLB_GRID_E4M3) return fail(NTLB_EINVAL, "%s: bad grid %d", fn, p->grid);
  return NTLB_OK;
}

static void zero_words(int32_t* p, int64_t n, int32_t* p2, int64_t n2, hipStream_t st) {
  zero_words_kernel<<<(unsigned)cdiv(n + n2, 256), 256, 0, st>>>(reinterpret_cast<uint32_t*>(p), n,
                                                                 reinterpret_cast<uint32_t*>(p2), n2);
}

}  // namespace ntlb

using namespace ntlb;

extern "C" int ntlb_linear_plan_init(ntlb_linear_plan* p) {
  const char* fn = "ntlb_linear_plan_init";
  if (int rc = check_plan(fn, p)) return rc;
  const int64_t kp = up(p->K, 128), np = up(p->N, 128), mp = up(p->M, 128);
  p->x_code_bytes = x_layout(*p).bytes;
  p->w_code_bytes = w_layout(*p).bytes;
  const SteLayout sl = ste_layout(*p);
  p->ste_bytes = sl.dy;
  p->ste_pad_bytes = sl.bytes;
  p->ste_free_pitch = sl.wd >= 0 ? sl.near_pitch : 0;
  p->recipe_bytes = recipe_layout(*p).bytes;
  p->forward_ws = ntlb_gemm_workspace_bytes(p->M, p->N, kp);
  p->ste_ws = ntlb_gemm_dq_workspace_bytes(NTLB_BF16, p->M, p->K, p->N);
  p->recipe_ws = std::max(ntlb_gemm_workspace_bytes(p->M, p->K, np), ntlb_gemm_workspace_bytes(p->N, p->K, mp));
  return NTLB_OK;
}

extern "C" int ntlb_linear_forward(const ntlb_linear_plan* p, const void* x, const void* w, const void* bias,
                                   void* x_codes, void* w_codes, void* y, void* workspace, int64_t ws_bytes,
                                   uint64_t offset, void* stream) {
  const char* fn = "ntlb_linear_forward";
  if (int rc = check_plan(fn, p)) return rc;
  if (!x || !w || !x_codes || !w_codes || !y) return fail(NTLB_EINVAL, "%s: NULL pointer", fn);
  if (!aligned(x_codes, 256) || !aligned(w_codes, 256))
    return fail(NTLB_EINVAL, "%s: the code buffers must be 256-byte aligned", fn);
  const CodeLayout lx = x_layout(*p), lw = w_layout(*p);
  uint8_t* xb = reinterpret_cast<uint8_t*>(x_codes);
  uint8_t* wb = reinterpret_cast<uint8_t*>(w_codes);
  float* xs = reinterpret_cast<float*>(xb + lx.s);
  float* ws = reinterpret_cast<float*>(wb + lw.s);
  const int64_t kp = up(p->K, 128), T = kp / 128, m4 = up(p->M, 4);
  int32_t* nan_x = lx.flags >= 0 ? reinterpret_cast<int32_t*>(xb + lx.flags) : nullptr;
  int32_t* nan_w = lw.flags >= 0 ? reinterpret_cast<int32_t*>(wb + lw.flags) : nullptr;
  if (nan_x) zero_words(nan_x, p->M, nan_w, p->N, as_stream(stream));
  int rc = ntlb_quant_tile_1x128(x, p->x_dtype, p->M, p->K, p->ldx, p->grid, p->qmax, p->rounding,
                                 NTLB_SCALE_AFTER_DIVIDE, p->seed, offset, xb + lx.c, kp, xs, 1, m4, nullptr, 0, 0,
                                 nan_x, stream);
  if (rc) return rc;
  rc = ntlb_quant_block_128x128(w, p->w_dtype, p->N, p->K, p->ldw, p->grid, p->qmax, p->rounding,
                                NTLB_SCALE_AFTER_DIVIDE, p->seed, offset + 1, wb + lw.c, kp, nullptr, 0, ws, T, 1,
                                nullptr, 0, 0, nan_w, stream);
  if (rc) return rc;
  return ntlb_gemm_blockscaled_ws(p->grid, xb + lx.c, kp, xs, 1, m4, 0, wb + lw.c, kp, ws, T, 1, 7, p->M, p->N, kp,
                                  bias, p->bias_dtype, y, p->x_dtype, p->N, nan_x, nan_w, workspace, ws_bytes,
                                  stream);
}

extern "C" int ntlb_linear_ste_backward(const ntlb_linear_plan* p, const void* dy, int64_t lddy, const void* x_codes,
                                        const void* w_codes, void* dx, void* dw, void* db, int db_dtype,
                                        void* scratch, int64_t scratch_bytes, void* workspace, int64_t ws_bytes,
                                        void* stream) {
  const char* fn = "ntlb_linear_ste_backward";
  if (int rc = check_plan(fn, p)) return rc;
  if (!dy || !scratch || (dx && !w_codes) || (dw && !x_codes)) return fail(NTLB_EINVAL, "%s: NULL pointer", fn);
  if (p->x_dtype != NTLB_BF16 || p->w_dtype != NTLB_BF16) return fail(NTLB_EUNSUPPORTED, "%s: bf16 only", fn);
  if (lddy < p->N) return fail(NTLB_EINVAL, "%s: lddy < N", fn);
  const CodeLayout lx = x_layout(*p), lw = w_layout(*p);
  const SteLayout sl = ste_layout(*p);
  const uint8_t* xb = reinterpret_cast<const uint8_t*>(x_codes);
  const uint8_t* wb = reinterpret_cast<const uint8_t*>(w_codes);
  uint8_t* s = reinterpret_cast<uint8_t*>(scratch);
  const int64_t kp = up(p->K, 128), T = kp / 128, m4 = up(p->M, 4), n64 = up(p->N, 64);
  const bool pad_dy = p->N % 64 || lddy % 8 || !aligned(dy, 16);
  if (!aligned(scratch, 256) || scratch_bytes < (pad_dy ? sl.bytes : sl.dy))
    return fail(NTLB_EINVAL, "%s: the scratch is misaligned or too small", fn);
  if (pad_dy) {
    // both GEMMs and the column sum read whole 16-byte chunks of dY's rows,
    // the dgrad whole 64-column steps: one padded copy serves all three
    const int64_t q = p->M * (n64 >> 3);
    if (cdiv(q, 256) > 0x7FFFFFFF) return fail(NTLB_EINVAL, "%s: too large", fn);
    uint16_t* pad = reinterpret_cast<uint16_t*>(s + sl.dy);
    pad_rows16_kernel<<<(unsigned)cdiv(q, 256), 256, 0, as_stream(stream)>>>(
        reinterpret_cast<const uint16_t*>(dy), lddy, p->M, p->N, pad, n64);
    dy = pad;
    lddy = n64;
  }
  const bool near_rows = lddy <= sl.near_pitch;
  const bool small_dx = dx && sl.wd >= 0 && near_rows, small_dw = dw && sl.xd >= 0 && near_rows;
  if (small_dx || small_dw) {
    DecodeArgs d{};
    if (small_dx) {
      d.wc = wb + lw.c;
      d.ws = reinterpret_cast<const float*>(wb + lw.s);
      d.wrows = p->N;
    }
    if (small_dw) {
      d.xc = xb + lx.c;
      d.xs = reinterpret_cast<const float*>(xb + lx.s);
      d.xrows = p->M;
    }
    d.kp = kp; d.T = T; d.m4 = m4; d.ld = up(p->K, 8);
    d.wd = reinterpret_cast<uint16_t*>(s + std::max<int64_t>(sl.wd, 0));
    d.xd = reinterpret_cast<uint16_t*>(s + std::max<int64_t>(sl.xd, 0));
    const int64_t q = (d.wrows + d.xrows) * (d.ld >> 3);
    if (cdiv(q, 256) > 0x7FFFFFFF) return fail(NTLB_EINVAL, "%s: too large", fn);
    const unsigned wgs = (unsigned)cdiv(q, 256);
    if (p->grid == NTLB_GRID_E4M3)
      decode_operands_kernel<GRID_E4M3><<<wgs, 256, 0, as_stream(stream)>>>(d);
    else
      decode_operands_kernel<GRID_INT><<<wgs, 256, 0, as_stream(stream)>>>(d);
    Bf16Args g{};
    g.y_dtype = NTLB_BF16;
    g.ldy = g.N = p->K;
    if (small_dx) {
      g.a = Bf16Operand{dy, lddy, p->M, 0, false};
      g.b = Bf16Operand{d.wd, d.ld, p->K, p->N, true};
      g.M = p->M;
      g.Kc = n64;
      g.y = dx;
      g.vec_out = aligned(dx, 16) && p->K % 8 == 0;
      if (int rc = bf16_small_launch(fn, sl.dx, g, as_stream(stream))) return rc;
    }
    if (small_dw) {
      g.a = Bf16Operand{dy, lddy, p->N, p->M, true};
      g.b = Bf16Operand{d.xd, d.ld, p->K, p->M, true};
      g.M = p->N;
      g.Kc = up(p->M, 64);
      g.y = dw;
      g.vec_out = aligned(dw, 16) && p->K % 8 == 0;
      if (int rc = bf16_small_launch(fn, sl.dw, g, as_stream(stream))) return rc;
    }
  }
  if (dx && !small_dx) {
    const int rc = ntlb_gemm_ste_dgrad_ws(NTLB_BF16, dy, lddy, p->M, p->N, p->grid, wb + lw.c, kp,
                                          reinterpret_cast<const float*>(wb + lw.s), T, 1, 7, p->K, dx, NTLB_BF16,
                                          p->K, workspace, ws_bytes, stream);
    if (rc) return rc;
  }
  if (dw && !small_dw) {
    const int rc = ntlb_gemm_ste_wgrad(NTLB_BF16, dy, lddy, p->M, p->N, p->grid, xb + lx.c, kp,
                                       reinterpret_cast<const float*>(xb + lx.s), 1, m4, 0, p->K, dw, NTLB_BF16,
                                       p->K, stream);
    if (rc) return rc;
  }
  if (db)
    return ntlb_colsum(dy, NTLB_BF16, p->M, p->N, lddy, reinterpret_cast<float*>(s + sl.colsum), sl.dy - sl.colsum,
                       db, db_dtype, stream);
  return check_launch(fn);
}

extern "C" int ntlb_linear_recipe_backward(const ntlb_linear_plan* p, const void* dy, int64_t lddy, const void* x,
                                           const void* w, void* dx, void* dw, void* db, int db_dtype, void* scratch,
                                           int64_t scratch_bytes, void* workspace, int64_t ws_bytes,
                                           uint64_t offset, void* stream) {
  const char* fn = "ntlb_linear_recipe_backward";
  if (int rc = check_plan(fn, p)) return rc;
  if (!dy || !scratch || !x || !w) return fail(NTLB_EINVAL, "%s: NULL pointer", fn);
  if (lddy < p->N) return fail(NTLB_EINVAL, "%s: lddy < N", fn);
  const RecipeLayout l = recipe_layout(*p);
  if (!aligned(scratch, 256) || scratch_bytes < l.bytes)
    return fail(NTLB_EINVAL, "%s: the scratch is misaligned or too small", fn);
  uint8_t* b = reinterpret_cast<uint8_t*>(scratch);
  const int64_t kp = up(p->K, 128), np = up(p->N, 128), mp = up(p->M, 128), T = kp / 128;
  const int64_t m4 = up(p->M, 4), n4 = up(p->N, 4), k4 = up(p->K, 4);
  const int rule = NTLB_SCALE_AFTER_DIVIDE, dt = p->x_dtype;
  int32_t* nan_m = l.flags >= 0 ? reinterpret_cast<int32_t*>(b + l.flags) : nullptr;
  int32_t* nan_n = nan_m ? nan_m + p->M : nullptr;
  int32_t* nan_k = nan_m ? nan_n + p->N : nullptr;
  float* ys = reinterpret_cast<float*>(b + l.ys);
  float* yts = reinterpret_cast<float*>(b + l.yts);
  float* wsc = reinterpret_cast<float*>(b + l.ws);
  float* xts = reinterpret_cast<float*>(b + l.xts);
  int rc = NTLB_OK;
  if (nan_m && (dx || dw)) zero_words(nan_m, p->M + p->N + p->K, nullptr, 0, as_stream(stream));
  // dY's 1x128 and 128x1 quantizations share one Philox offset: one pass over
  // dY writes both where its rows allow
  const bool dual = dx && dw && p->N % 8 == 0 && lddy % 8 == 0 && aligned(dy, 16) && dt != NTLB_F16;
  if (dual)
    rc = ntlb_quant_dual_1x128_128x1(dy, dt, p->M, p->N, lddy, p->grid, p->qmax, p->rounding, rule, p->seed,
                                     offset + 2, offset + 2, b + l.yc, np, ys, 1, m4, nan_m, b + l.ytc, mp, yts, 1,
                                     n4, nan_n, stream);
  if (dx && !rc) {
    if (!dual)
      rc = ntlb_quant_tile_1x128(dy, dt, p->M, p->N, lddy, p->grid, p->qmax, p->rounding, rule, p->seed, offset + 2,
                                 b + l.yc, np, ys, 1, m4, nullptr, 0, 0, nan_m, stream);
    if (!rc)
      rc = ntlb_quant_block_128x128(w, p->w_dtype, p->N, p->K, p->ldw, p->grid, p->qmax, p->rounding, rule, p->seed,
                                    offset + 1, b + l.wc, kp, b + l.wtc, np, wsc, T, 1, nullptr, 0, 0, nullptr,
                                    stream);
    if (!rc)
      rc = ntlb_gemm_blockscaled_ws(p->grid, b + l.yc, np, ys, 1, m4, 0, b + l.wtc, np, wsc, 1, T, 7, p->M, p->K, np,
                                    nullptr, 0, dx, dt, p->K, nan_m, nullptr, workspace, ws_bytes, stream);
  }
  if (dw && !rc) {
    if (!dual)
      rc = ntlb_quant_tile_128x1_t(dy, dt, p->M, p->N, lddy, p->grid, p->qmax, p->rounding, rule, p->seed,
                                   offset + 2, b + l.ytc, mp, yts, 1, n4, nullptr, 0, 0, nan_n, stream);
    if (!rc)
      rc = ntlb_quant_tile_128x1_t(x, p->x_dtype, p->M, p->K, p->ldx, p->grid, p->qmax, p->rounding, rule, p->seed,
                                   offset + 4, b + l.xtc, mp, xts, 1, k4, nullptr, 0, 0, nan_k, stream);
    if (!rc)
      rc = ntlb_gemm_blockscaled_ws(p->grid, b + l.ytc, mp, yts, 1, n4, 0, b + l.xtc, mp, xts, 1, k4, 0, p->N, p->K,
                                    mp, nullptr, 0, dw, dt, p->K, nan_n, nan_k, workspace, ws_bytes, stream);
  }
  if (db && !rc)
    rc = ntlb_colsum(dy, dt, p->M, p->N, lddy, reinterpret_cast<float*>(b + l.colsum), l.yc - l.colsum, db, db_dtype,
                     stream);
  return rc;
}
