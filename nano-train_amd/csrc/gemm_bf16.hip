// bf16 GEMM on tiles below 256x256, fp32 accumulation: the products of
// gemm_dq.hip over plain bf16 matrices whose 256x256 tiles would leave most of
// the chip idle (dX and dW of small straight-through layers, dW of persistent
// ones).
//
// 16*MB x 16*NB tiles, a workgroup's WK waves dividing the contraction, each
// wave with its own multi-stage LDS copies and no barrier in the K loop, as
// gemm_small.hip (whose comment gives the reasons); and 128x128 tiles, staged
// once per workgroup of four waves, as its gemm_mid_kernel.  A K step is 64
// values (128 bytes).  Operands stored transposed are copied as stored and read
// with ds_read_b64_tr_b16 (lane layout: gemm_dq.hip).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "ntlb_device.h"
#include "ntlb_gemm_bf16.h"
#include "ntlb_host.h"
#include "ntlb_small_tile.h"
#include "ntlb_splitk.h"

namespace ntlb {
namespace bfs {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(3))) v4s* lds_v4s_ptr;

constexpr int ROWB = 128;   // bytes of a row's K step
constexpr int KSTEP = 64;

// Row-major stage [16*B rows][128 bytes]: 16-byte chunk c of row r at slot
// c ^ perm(r), conflict-free for the 16-row fragment reads
__device__ __forceinline__ int row_perm(int r) { return (r & 7) ^ ((r >> 3) & 1); }

// Transposed stage [64 contraction rows][16*B operand rows]: 2*B chunks per
// contraction row.  A 16-lane group of ds_read_b64_tr_b16 reads 32 bytes of
// each of four consecutive contraction rows, the next group those 16 further:
// the XOR spreads these eight 32-byte pieces over the 256 bytes of banks (for
// rows of 32 bytes the two groups share them).
template <int B>
__device__ __forceinline__ int tr_perm(int k) {
  if constexpr (B >= 8) return (2 * (k & 3)) ^ (8 * ((k >> 4) & 1));  // 256-byte rows
  if constexpr (B == 4) return 2 * (((k >> 1) & 1) | (((k >> 4) & 1) << 1));
  if constexpr (B == 2) return 2 * ((k >> 4) & 1);
  return 0;
}

// MFMA fragments of one K step: row = lane%16 of 16 operand rows, contraction
// 16g .. 16g+15 with g = lane/16
template <bool TR, int B>
__device__ __forceinline__ v8i frag(const uint8_t* tile, int row0, int lane) {
  const int g = lane >> 4;
  v8i f;
  if constexpr (!TR) {
    const int r = row0 + (lane & 15);
    const uint4 lo = *reinterpret_cast<const uint4*>(tile + r * ROWB + (((2 * g) ^ row_perm(r)) << 4));
    const uint4 hi = *reinterpret_cast<const uint4*>(tile + r * ROWB + (((2 * g + 1) ^ row_perm(r)) << 4));
    f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
    f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
  } else {
    const int j = (lane >> 2) & 3, q = lane & 3;
    const int c = (row0 >> 3) + (q >> 1);
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const int k = 16 * g + 4 * h + j;
      const v4s v = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (lds_v4s_ptr)(tile + k * (32 * B) + ((c ^ tr_perm<B>(k)) << 4) + (q & 1) * 8));
      f[2 * h] = (int)(((uint32_t)(uint16_t)v[1] << 16) | (uint16_t)v[0]);
      f[2 * h + 1] = (int)(((uint32_t)(uint16_t)v[3] << 16) | (uint16_t)v[2]);
    }
  }
  return f;
}

__device__ __forceinline__ v4f mma(const v8i& p, const v8i& q, v4f acc) {
  const v4i pl = {p[0], p[1], p[2], p[3]}, ph = {p[4], p[5], p[6], p[7]};
  const v4i ql = {q[0], q[1], q[2], q[3]}, qh = {q[4], q[5], q[6], q[7]};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, pl), __builtin_bit_cast(v8bf, ql), acc, 0, 0,
                                                0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(v8bf, ph), __builtin_bit_cast(v8bf, qh), acc, 0,
                                                 0, 0);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t operand_rsrc(const Bf16Operand& o) {
  const int64_t bytes = o.tr ? stored_rows_extent(o.kvalid, o.ld, o.rows, 2) : o.rows * o.ld * 2;
  return __builtin_amdgcn_make_buffer_rsrc((void*)o.p, (short)0, (int)bytes, 0x00020000);
}

// The copies of one operand's K step (16*B operand rows, 2*B KiB-copies of 64
// lanes) by NW waves, wave w taking copies w, w + NW, ...  The LDS side is
// linear in (copy, lane); the lane's global offset carries the swizzle.  Copies
// of one parity differ by a constant, so two lane offsets serve all.
template <bool TR, int B, int NW>
struct Copies {
  static constexpr int COUNT = 2 * B / NW;
  static_assert(2 * B % NW == 0, "whole copies per wave");
  __amdgpu_buffer_rsrc_t rs;
  uint32_t off[COUNT];
  uint32_t kstep;  // bytes per K step
  int wave;
  __device__ __forceinline__ void init(const Bf16Operand& o, int64_t r0, int w, int lane) {
    rs = operand_rsrc(o);
    wave = w;
    kstep = TR ? (uint32_t)(KSTEP * o.ld * 2) : (uint32_t)ROWB;
#pragma unroll
    for (int i = 0; i < COUNT; ++i) {
      const int slot = (w + NW * i) * 64 + lane;
      if constexpr (TR) {
        const int k = slot / (2 * B), c = (slot % (2 * B)) ^ tr_perm<B>(k);
        off[i] = (uint32_t)(k * o.ld * 2 + (r0 + 8 * c) * 2);
      } else {
        const int r = slot >> 3, c = (slot & 7) ^ row_perm(r);
        off[i] = (uint32_t)((r0 + r) * o.ld * 2 + c * 16);
      }
    }
  }
  __device__ __forceinline__ void issue(uint8_t* stage, int ks) const {
#pragma unroll
    for (int i = 0; i < COUNT; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (lds_ptr_t)(stage + (wave + NW * i) * 1024), 16, off[i],
                                               (uint32_t)ks * kstep, 0, 0);
  }
};

__device__ __forceinline__ void store4(const Bf16Args& g, int64_t m, int64_t n, v4f v) {
  if (g.vec_out && n + 4 <= g.N && g.y_dtype == DT_BF16) {
    const v2bf p0 = {(__bf16)v[0], (__bf16)v[1]}, p1 = {(__bf16)v[2], (__bf16)v[3]};
    *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(g.y) + m * g.ldy + n) =
        make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
    return;
  }
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (n + q < g.N) store_elem(g.y, g.y_dtype, m * g.ldy + n + q, v[q]);
}

template <bool TA, int MB, int NB, int WK, int NS>
__global__ void __launch_bounds__(64 * WK) gemm_bf16_small_kernel(Bf16Args g) {
  constexpr int WB = (MB + NB) * 16 * ROWB;
  static_assert(MB * NB * 1024 <= WB, "the partial tiles fit the first stage");
  __shared__ __attribute__((aligned(16))) uint8_t st0[WK * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st1[WK * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st2[NS > 2 ? WK * WB : 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NB), m0 = (int64_t)blockIdx.y * (16 * MB);
  const int nk = (int)(g.Kc / KSTEP);
  const int k0 = (int)((int64_t)wave * nk / WK), k1 = (int)((int64_t)(wave + 1) * nk / WK);
  v4f acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = (v4f){0.f, 0.f, 0.f, 0.f};
  if (k0 < k1) {
    Copies<TA, MB, 1> ca;
    Copies<true, NB, 1> cb;
    ca.init(g.a, m0, 0, lane);
    cb.init(g.b, n0, 0, lane);
    uint8_t* const s0 = st0 + wave * WB;
    uint8_t* const s1 = st1 + wave * WB;
    uint8_t* const s2 = st2 + (NS > 2 ? wave * WB : 0);
    auto stage = [&](int i) { return i == 0 ? s0 : i == 1 ? s1 : s2; };
    auto issue = [&](int i, int ks) {
      ca.issue(stage(i), ks);
      cb.issue(stage(i) + MB * 16 * ROWB, ks);
    };
    auto each = [](auto f) {
      f(std::integral_constant<int, 0>());
      f(std::integral_constant<int, 1>());
      if constexpr (NS > 2) f(std::integral_constant<int, 2>());
    };
    auto step = [&](auto ic, int ks) {
      constexpr int I = decltype(ic)::value;
      __builtin_amdgcn_s_waitcnt(0xC07F);  // the reads of the stage refilled now are done
      asm volatile("" ::: "memory");
      issue((I + NS - 1) % NS, min(ks + NS - 1, k1 - 1));
      // in-order returns: with only the younger stages' copies outstanding,
      // this stage has landed
      __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * 2 * (MB + NB)));
      asm volatile("" ::: "memory");
      const uint8_t* ta = stage(I);
      const uint8_t* tb = ta + MB * 16 * ROWB;
      v8i bf[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) bf[nb] = frag<true, NB>(tb, nb * 16, lane);
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) {
        const v8i af = frag<TA, MB>(ta, mb * 16, lane);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = mma(bf[nb], af, acc[mb][nb]);
      }
    };
    each([&](auto ic) {
      if constexpr (decltype(ic)::value < NS - 1) issue(decltype(ic)::value, min(k0 + decltype(ic)::value, k1 - 1));
    });
    int ks = k0;
    for (; ks + NS <= k1; ks += NS) each([&](auto ic) { step(ic, ks + decltype(ic)::value); });
    each([&](auto ic) {
      if (ks + decltype(ic)::value < k1) step(ic, ks + decltype(ic)::value);
    });
    __builtin_amdgcn_s_waitcnt(0);  // nothing of this wave is in flight into LDS past here
    asm volatile("" ::: "memory");
  }
  sum_partials<MB, NB, WK>(reinterpret_cast<v4f*>(st0), acc, wave, lane, m0, n0, g.M, g.N,
                           [&](int64_t m, int64_t n, v4f v) { store4(g, m, n, v); });
}

template <bool TA, int ODT>
__global__ void __launch_bounds__(256, 2) gemm_bf16_mid_kernel(Bf16Args g) {
  constexpr int ST = MID * ROWB;  // 16 KiB per operand stage
  __shared__ __attribute__((aligned(16))) uint8_t la0[ST];
  __shared__ __attribute__((aligned(16))) uint8_t lb0[ST];
  __shared__ __attribute__((aligned(16))) uint8_t la1[ST];
  __shared__ __attribute__((aligned(16))) uint8_t lb1[ST];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  int64_t m0, n0;
  mid_tile(g.M, g.N, m0, n0);
  Copies<TA, 8, 4> ca;
  Copies<true, 8, 4> cb;
  ca.init(g.a, m0, wave, lane);
  cb.init(g.b, n0, wave, lane);
  const int nk = (int)(g.Kc / KSTEP);
  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
  ca.issue(la0, 0);
  cb.issue(lb0, 0);
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  auto step = [&](auto bufc, int ks) {
    constexpr int BUF = decltype(bufc)::value;
    const uint8_t* ta = BUF ? la1 : la0;
    const uint8_t* tb = BUF ? lb1 : lb0;
    const int kn = min(ks + 1, nk - 1);  // the last step copies itself into the idle stage
    ca.issue(BUF ? la0 : la1, kn);
    cb.issue(BUF ? lb0 : lb1, kn);
    v8i bf[4];
#pragma unroll
    for (int tn = 0; tn < 4; ++tn) bf[tn] = frag<true, 8>(tb, wn * 64 + tn * 16, lane);
#pragma unroll
    for (int tm = 0; tm < 4; ++tm) {
      const v8i af = frag<TA, 8>(ta, wm * 64 + tm * 16, lane);
#pragma unroll
      for (int tn = 0; tn < 4; ++tn) acc[tm][tn] = mma(bf[tn], af, acc[tm][tn]);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
  for (int ks = 0; ks < nk; ks += 2) {
    step(std::integral_constant<int, 0>(), ks);
    if (ks + 1 < nk) step(std::integral_constant<int, 1>(), ks + 1);
  }
  // each wave stages its rows in its 16 KiB of the idle stages
  uint8_t* stage_w = wave == 0 ? la0 : wave == 1 ? lb0 : wave == 2 ? la1 : lb1;
  mid_store<ODT>(stage_w, lane, m0 + wm * 64, n0 + wn * 64, g.M, g.N, g.y, g.ldy, g.vec_out, [](int) { return 0; },
                 [&](int tm, int tn, int) { return acc[tm][tn]; });
}

// every instance explicitly: the host stubs of implicitly instantiated ones
// are not all emitted here (ROCm 7.2 hipcc)
#define NTLB_BF16_CASES(X) X(1, 1, 8, 2) X(1, 2, 4, 3) X(2, 2, 4, 3) X(2, 4, 4, 3) X(4, 4, 4, 2) X(4, 4, 2, 2)
#define NTLB_BF16_INST(MB, NB, WK, NS)                                              \
  template __global__ void gemm_bf16_small_kernel<true, MB, NB, WK, NS>(Bf16Args);  \
  template __global__ void gemm_bf16_small_kernel<false, MB, NB, WK, NS>(Bf16Args);
NTLB_BF16_CASES(NTLB_BF16_INST)
#undef NTLB_BF16_INST
template __global__ void gemm_bf16_mid_kernel<true, DT_F32>(Bf16Args);
template __global__ void gemm_bf16_mid_kernel<true, DT_BF16>(Bf16Args);
template __global__ void gemm_bf16_mid_kernel<true, DT_F16>(Bf16Args);
template __global__ void gemm_bf16_mid_kernel<false, DT_BF16>(Bf16Args);

template <bool TA>
static int launch(const char* fn, const Bf16Plan& p, const Bf16Args& g, hipStream_t st) {
  if (p.mb == 8) {
    const dim3 grd((unsigned)(cdiv(g.M, MID) * cdiv(g.N, MID))), blk(256);
    if (g.y_dtype == DT_BF16) {
      gemm_bf16_mid_kernel<TA, DT_BF16><<<grd, blk, 0, st>>>(g);
      return check_launch(fn);
    }
    if constexpr (TA) {
      if (g.y_dtype == DT_F32)
        gemm_bf16_mid_kernel<TA, DT_F32><<<grd, blk, 0, st>>>(g);
      else
        gemm_bf16_mid_kernel<TA, DT_F16><<<grd, blk, 0, st>>>(g);
      return check_launch(fn);
    }
  }
  const dim3 grd((unsigned)cdiv(g.N, 16 * p.nb), (unsigned)cdiv(g.M, 16 * p.mb)), blk(64 * p.wk);
#define NTLB_BF16_CASE(MB, NB, WK, NS)                                              \
  if (p.mb == MB && p.nb == NB && p.wk == WK && p.ns == NS) {                       \
    gemm_bf16_small_kernel<TA, MB, NB, WK, NS><<<grd, blk, 0, st>>>(g);             \
    return check_launch(fn);                                                        \
  }
  NTLB_BF16_CASES(NTLB_BF16_CASE)
#undef NTLB_BF16_CASE
  return fail(NTLB_EUNSUPPORTED, "%s: no kernel for a %d x %d tile", fn, 16 * p.mb, 16 * p.nb);
}

}  // namespace bfs

// The tile: the smallest one whose workgroups all run at once, as the
// blockwise products choose it.  Measured (both operands transposed, bf16 out,
// in a graph, us; this kernel / 256x256 tiles): 1000 x K 1003: 4.9 / 25 at 64
// rows, 7.8 / 25 at 512, 9.9 / 26 at 1003, 13.7 / 26 at 1541, 19 / 27 at 4096;
// 2048 x K 2048: 7.7 / 44 at 128 rows, 12.4 / 44 at 512, 21 / 46 at 1003, 33 / 45
// at 2048, 36 / 46 at 4096.
//
// 128x128 tiles run two to a compute unit, and up to two of them for each unit
// they beat unsplit 256x256 tiles at every K: 512 tiles (4096 x 2048) 6.7 / 7.8 at K
// 64, 21.5 / 27 at 1024, 36 / 47 at 2048, 129 / 162 at 8192, while 529 tiles (2880 x
// 2880), a second round of them, take 8.6 / 8.1, 37 / 27, 65 / 46 and 239 / 161.
// Where the 256x256 tiles would split their tail (big_split), an estimate
// decides: 1.05 us a K step here, 1.4 / split there and 30 us for the exchange.
Bf16Plan bf16_small_plan(int64_t M, int64_t N, int64_t Kc, bool big_split) {
  const int64_t cus = split_device_cus();
  const int nk = (int)(Kc / bfs::KSTEP);
  auto wgs = [&](int64_t rows, int64_t cols) { return cdiv(M, rows) * cdiv(N, cols); };
  if (wgs(16, 16) <= cus) return {1, 1, 8, 2};
  if (wgs(16, 32) <= cus || M <= 16) return {1, 2, 4, 3};
  if (wgs(32, 32) <= cus) return {2, 2, 4, 3};
  if (wgs(32, 64) <= cus) return {2, 4, 4, 3};
  if (wgs(64, 64) <= cus) return {4, 4, 4, 2};
  if (wgs(64, 64) <= 2 * cus) return {4, 4, 2, 2};
  if (wgs(MID, MID) <= 2 * cus) {
    const int split = big_split ? split_plan(wgs(256, 256), nk, DQ_SPLIT_MIN_STEPS).s : 1;
    if (split == 1 || 1.05 * nk + 3 < 1.4 * nk / split + 30) return {8, 8, 4, 2};
  }
  return {0, 0, 0, 0};
}

int bf16_small_launch(const char* fn, const Bf16Plan& p, const Bf16Args& g, hipStream_t st) {
  return g.a.tr ? bfs::launch<true>(fn, p, g, st) : bfs::launch<false>(fn, p, g, st);
}

}  // namespace ntlb
