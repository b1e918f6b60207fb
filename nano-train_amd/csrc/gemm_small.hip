// Blockwise-scaled GEMM of few rows or few output tiles (the products that
// leave most of the chip idle on 256x256 tiles): same operands, scales and
// promotion as gemm.hip, output tiles of 16*MB x 16*NB.
//
// A workgroup of WK waves owns one tile and each wave multiplies the whole
// tile over its own range of K blocks, so no wave waits for another before
// the end; the WK partial tiles are summed in wave order through LDS.  A wave
// copies its operand rows global -> LDS (16 bytes per lane, eight consecutive
// lanes on one 128-byte row of a K block: reading the fragments straight from
// global memory puts neighbouring lanes on different rows and costs four
// times the address cycles), NS stages deep, into LDS that it alone reads, so
// the K loop has no barrier: a stage is waited for with vmcnt.
//
// What bounds it: with few rows the weight codes' stream (every code is read
// once, N / (16 NB) workgroups of 8 waves); with more rows the operands'
// re-reads from L2 (each tile reads 16 (MB + NB) rows of K bytes).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "ntlb_gemm_tile.h"
#include "ntlb_host.h"
#include "ntlb_small_tile.h"
#include "ntlb_splitk.h"

namespace ntlb {

// One wave's copies of a 16*MB-row A and 16*NB-row B K block into LDS: copy t
// moves rows 8t .. 8t+7 (lane i: row i/8, physical chunk i%8, which holds the
// logical chunk (i%8) ^ swz_perm(row); bit 3 of the row is t & 1).  Rows past
// the matrix lie beyond the resource and read zero.
template <int MB, int NB>
struct WaveCopy {
  static constexpr int COPIES = 2 * (MB + NB);
  static constexpr int BYTES = (MB + NB) * 16 * BK;
  __amdgpu_buffer_rsrc_t ra, rb;
  uint32_t a0, a1, b0, b1;  // byte offsets of this lane's chunk for even and odd copies
  uint32_t a16, b16;        // 16 rows in bytes
  __device__ __forceinline__ void init(const GemmArgs& g, int64_t m0, int64_t n0, int lane) {
    const int r = lane >> 3, c = lane & 7;
    ra = __builtin_amdgcn_make_buffer_rsrc((void*)g.a, (short)0, (int)(g.M * g.lda), 0x00020000);
    rb = __builtin_amdgcn_make_buffer_rsrc((void*)g.b, (short)0, (int)(g.N * g.ldb), 0x00020000);
    a0 = (uint32_t)((m0 + r) * g.lda + ((c ^ swz_perm(r)) << 4));
    a1 = (uint32_t)((m0 + 8 + r) * g.lda + ((c ^ swz_perm(8 + r)) << 4));
    b0 = (uint32_t)((n0 + r) * g.ldb + ((c ^ swz_perm(r)) << 4));
    b1 = (uint32_t)((n0 + 8 + r) * g.ldb + ((c ^ swz_perm(8 + r)) << 4));
    a16 = (uint32_t)(16 * g.lda);
    b16 = (uint32_t)(16 * g.ldb);
  }
  // A rows at lds, B rows after them
  __device__ __forceinline__ void issue(uint8_t* lds, int kb) const {
    const uint32_t k = (uint32_t)kb * BK;
#pragma unroll
    for (int t = 0; t < 2 * MB; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(lds + t * 8 * BK), 16, (t & 1) ? a1 : a0,
                                               k + (t >> 1) * a16, 0, 0);
#pragma unroll
    for (int t = 0; t < 2 * NB; ++t)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(lds + (16 * MB + t * 8) * BK), 16,
                                               (t & 1) ? b1 : b0, k + (t >> 1) * b16, 0, 0);
  }
};

// The K loop of one wave over blocks [kb0, kb1), kb0 < kb1: acc += the
// promoted partials.  s0 / s1 / s2 are this wave's stages (distinct LDS
// objects, so that the copies in flight are seen not to alias the reads).
template <int GRID, bool B_UNIFORM, int MB, int NB, int NS>
__device__ __forceinline__ void small_k_loop(const GemmArgs& g, const WaveCopy<MB, NB>& cp, int64_t m0, int64_t n0,
                                             int kb0, int kb1, uint8_t* s0, uint8_t* s1, uint8_t* s2, int lane,
                                             v4f (&acc)[MB][NB]) {
  const int li = lane & 15, gq = lane >> 4;
  const float* sap[MB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
    sap[mb] = g.sa + (min<int64_t>(m0 + mb * 16 + li, g.M - 1) >> g.a_shift) * g.sa_row;
  // B's scale: one per block for 128x128 blocks and tensor scales, else one
  // per column (this lane's columns 4*gq .. 4*gq+3 of each 16)
  const float* sbu = g.sb + (n0 >> g.b_shift) * g.sb_row;
  float sam[NS][MB];
  float sb1[NS];
  v4f sbv[NS][B_UNIFORM ? 1 : NB];
  auto stage = [&](int i) { return i == 0 ? s0 : i == 1 ? s1 : s2; };
  auto issue = [&](auto ic, int kb) {
    constexpr int I = decltype(ic)::value;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) sam[I][mb] = sap[mb][(int64_t)kb * g.sa_col];
    if constexpr (B_UNIFORM) {
      sb1[I] = sbu[(int64_t)kb * g.sb_col];
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          sbv[I][nb][q] = g.sb[(min<int64_t>(n0 + nb * 16 + gq * 4 + q, g.N - 1) >> g.b_shift) * g.sb_row +
                               (int64_t)kb * g.sb_col];
    }
    cp.issue(stage(I), kb);
  };
  auto compute = [&](auto ic) {
    constexpr int I = decltype(ic)::value;
    const uint8_t* ta = stage(I);
    const uint8_t* tb = ta + 16 * MB * BK;
    // the scales become visible here: a product of them moved up to an
    // earlier step would wait for loads younger than that step's copies
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) asm volatile("" : "+v"(sam[I][mb]));
    if constexpr (B_UNIFORM) {
      asm volatile("" : "+v"(sb1[I]));
    } else {
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) asm volatile("" : "+v"(sbv[I][nb]));
    }
    v8i bf[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) bf[nb] = load_frag(tb, nb * 16, lane);
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
      const v8i af = load_frag(ta, mb * 16, lane);
      raw_t<GRID> d[NB];
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) d[nb] = mma_raw<GRID>(bf[nb], af);
#pragma unroll
      for (int nb = 0; nb < NB; ++nb) {
        if constexpr (B_UNIFORM) {
          const float s = sam[I][mb] * sb1[I];
          acc[mb][nb] += raw_f32<GRID>(d[nb]) * s;
        } else {
          acc[mb][nb] += (raw_f32<GRID>(d[nb]) * sbv[I][nb]) * sam[I][mb];
        }
      }
    }
  };
  auto each = [](auto f) {
    f(std::integral_constant<int, 0>());
    f(std::integral_constant<int, 1>());
    if constexpr (NS > 2) f(std::integral_constant<int, 2>());
  };
  // the first NS - 1 blocks (past the end: the last block again, never read)
  each([&](auto ic) {
    if constexpr (decltype(ic)::value < NS - 1) issue(ic, min(kb0 + decltype(ic)::value, kb1 - 1));
  });
  auto step = [&](auto ic, int kb) {
    constexpr int I = decltype(ic)::value;
    // this wave's reads of the stage refilled now are done (lgkmcnt(0))
    __builtin_amdgcn_s_waitcnt(0xC07F);
    asm volatile("" ::: "memory");
    issue(std::integral_constant<int, (I + NS - 1) % NS>(), min(kb + NS - 1, kb1 - 1));
    // loads return in order: with at most the younger stages' copies
    // outstanding, this stage has landed
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * WaveCopy<MB, NB>::COPIES));
    asm volatile("" ::: "memory");
    compute(ic);
  };
  int kb = kb0;
  for (; kb + NS <= kb1; kb += NS) each([&](auto ic) { step(ic, kb + decltype(ic)::value); });
  each([&](auto ic) {
    if (kb + decltype(ic)::value < kb1) step(ic, kb + decltype(ic)::value);
  });
  // nothing of this wave is in flight into LDS past here
  __builtin_amdgcn_s_waitcnt(0);
  asm volatile("" ::: "memory");
}

// Row m, columns n .. n+3 of the output (bias, NaN flags, output type)
__device__ __forceinline__ void small_store4(const GemmArgs& g, int64_t m, int64_t n, v4f v, const int32_t* nan_b) {
  if (g.bias) {
#pragma unroll
    for (int q = 0; q < 4; ++q) v[q] += load_elem(g.bias, g.bias_dtype, min<int64_t>(n + q, g.N - 1));
  }
  const float qnan = __uint_as_float(0x7FC00000u);
  if (g.nan_a && g.nan_a[m]) v = (v4f){qnan, qnan, qnan, qnan};
  if (nan_b) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (nan_b[min<int64_t>(n + q, g.N - 1)]) v[q] = qnan;
  }
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

template <int GRID, bool B_UNIFORM, int MB, int NB, int WK, int NS>
__global__ void __launch_bounds__(64 * WK) gemm_small_kernel(GemmArgs g) {
  constexpr int WB = WaveCopy<MB, NB>::BYTES;
  static_assert(MB * NB * 1024 <= WB, "the partial tiles fit the first stage");
  __shared__ __attribute__((aligned(16))) uint8_t st0[WK * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st1[WK * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st2[NS > 2 ? WK * WB : 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = (int64_t)blockIdx.x * (16 * NB), m0 = (int64_t)blockIdx.y * (16 * MB);
  const int nk = (int)(g.Kp / BK);
  const int kb0 = (int)((int64_t)wave * nk / WK), kb1 = (int)((int64_t)(wave + 1) * nk / WK);
  v4f acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = (v4f){0.f, 0.f, 0.f, 0.f};
  if (kb0 < kb1) {
    WaveCopy<MB, NB> cp;
    cp.init(g, m0, n0, lane);
    small_k_loop<GRID, B_UNIFORM, MB, NB, NS>(g, cp, m0, n0, kb0, kb1, st0 + wave * WB, st1 + wave * WB,
                                              st2 + (NS > 2 ? wave * WB : 0), lane, acc);
  }
  sum_partials<MB, NB, WK>(reinterpret_cast<v4f*>(st0), acc, wave, lane, m0, n0, g.M, g.N,
                           [&](int64_t m, int64_t n, v4f v) { small_store4(g, m, n, v, g.nan_b); });
}

// ---------------------------------------------------------------------------
// 128x128 tiles: four waves as 2 (M) x 2 (N), each 64x64, both operands of a K
// block staged once per workgroup (32 KiB, double buffered), two workgroups
// per compute unit.  For products whose 256x256 tiles do not fill the chip
// (or leave a last wave of tiles mostly empty) but which are too large for
// 64x64 tiles: per 16x16x128 MFMA a wave reads 1 KiB of LDS (0.75 on the
// 256x256 tiles' 128x64 waves), which at the MFMA rate is the LDS bandwidth.
// ---------------------------------------------------------------------------
constexpr int MID_TILE = MID * BK;  // 16 KiB per operand stage

template <int GRID, bool B_UNIFORM, int ODT>
__global__ void __launch_bounds__(256, 2) gemm_mid_kernel(GemmArgs g) {
  __shared__ __attribute__((aligned(16))) uint8_t la0[MID_TILE];
  __shared__ __attribute__((aligned(16))) uint8_t lb0[MID_TILE];
  __shared__ __attribute__((aligned(16))) uint8_t la1[MID_TILE];
  __shared__ __attribute__((aligned(16))) uint8_t lb1[MID_TILE];
  __shared__ float ls0[2 * MID], ls1[2 * MID];  // A row scales, then B row scales
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  int64_t m0, n0;
  mid_tile(g.M, g.N, m0, n0);
  const bool own_a = tid < MID;
  const int64_t srow = own_a ? min<int64_t>(m0 + tid, g.M - 1) : min<int64_t>(n0 + tid - MID, g.N - 1);
  const float* s_src = own_a ? g.sa + (srow >> g.a_shift) * g.sa_row : g.sb + (srow >> g.b_shift) * g.sb_row;
  const int64_t s_step = own_a ? g.sa_col : g.sb_col;
  // wave w copies the 8-row groups w, w+4, w+8, w+12 of each operand (bit 3 of
  // their rows is w & 1, so a lane's chunk is the same in all four)
  const __amdgpu_buffer_rsrc_t ra =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.a, (short)0, (int)(g.M * g.lda), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb =
      __builtin_amdgcn_make_buffer_rsrc((void*)g.b, (short)0, (int)(g.N * g.ldb), 0x00020000);
  const int cr = wave * 8 + (lane >> 3), cc = (lane & 7) ^ swz_perm(cr);
  const uint32_t a_off = (uint32_t)((m0 + cr) * g.lda + cc * 16), b_off = (uint32_t)((n0 + cr) * g.ldb + cc * 16);
  const uint32_t a_grp = (uint32_t)(32 * g.lda), b_grp = (uint32_t)(32 * g.ldb);
  auto issue = [&](uint8_t* la, uint8_t* lb, int kt, int j) {
    const uint32_t k = (uint32_t)kt * BK;
    const int r0 = (wave + 4 * j) * 8;
    __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_ptr_t)(la + r0 * BK), 16, a_off, k + j * a_grp, 0, 0);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (lds_ptr_t)(lb + r0 * BK), 16, b_off, k + j * b_grp, 0, 0);
  };
  const int nk = (int)(g.Kp / BK);
  v4f acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 4; ++j) issue(la0, lb0, 0, j);
  ls0[tid] = s_src[0];
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  auto step = [&](auto bufc, int kt) {
    constexpr int BUF = decltype(bufc)::value;
    const uint8_t* ta = BUF ? la1 : la0;
    const uint8_t* tb = BUF ? lb1 : lb0;
    const float* s_cur = BUF ? ls1 : ls0;
    // the last block copies itself into the idle stage: one basic block
    const int kn = min(kt + 1, nk - 1);
    const float s_next = s_src[(int64_t)kn * s_step];
#pragma unroll
    for (int j = 0; j < 4; ++j) issue(BUF ? la0 : la1, BUF ? lb0 : lb1, kn, j);
    v8i bf[4];
#pragma unroll
    for (int tn = 0; tn < 4; ++tn) bf[tn] = load_frag(tb, wn * 64 + tn * 16, lane);
    float sam[4], sbu = 0.f;
    v4f sbv[B_UNIFORM ? 1 : 4];
#pragma unroll
    for (int tm = 0; tm < 4; ++tm) sam[tm] = s_cur[wm * 64 + tm * 16 + (lane & 15)];
    if constexpr (B_UNIFORM) {
      sbu = s_cur[MID + wn * 64];
    } else {
#pragma unroll
      for (int tn = 0; tn < 4; ++tn)
#pragma unroll
        for (int q = 0; q < 4; ++q) sbv[tn][q] = s_cur[MID + wn * 64 + tn * 16 + (lane >> 4) * 4 + q];
    }
    // as the 256x256 kernel: group tm's MFMAs are issued before group tm-1's
    // results are promoted
    raw_t<GRID> dp[4];
#pragma unroll
    for (int tm = 0; tm < 5; ++tm) {
      raw_t<GRID> d[4];
      if (tm < 4) {
        const v8i af = load_frag(ta, wm * 64 + tm * 16, lane);
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) d[tn] = mma_raw<GRID>(bf[tn], af);
      }
      if (tm > 0) {
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) {
          if constexpr (B_UNIFORM)
            acc[tm - 1][tn] += raw_f32<GRID>(dp[tn]) * (sam[tm - 1] * sbu);
          else
            acc[tm - 1][tn] += (raw_f32<GRID>(dp[tn]) * sbv[tn]) * sam[tm - 1];
        }
      }
      if (tm < 4) {
#pragma unroll
        for (int tn = 0; tn < 4; ++tn) dp[tn] = d[tn];
      }
    }
    (BUF ? ls0 : ls1)[tid] = s_next;
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
  };
  for (int kt = 0; kt < nk; kt += 2) {
    step(std::integral_constant<int, 0>(), kt);
    if (kt + 1 < nk) step(std::integral_constant<int, 1>(), kt + 1);
  }

  // each wave stages its rows in its 16 KiB of the idle stages
  uint8_t* stage_w = wave == 0 ? la0 : wave == 1 ? lb0 : wave == 2 ? la1 : lb1;
  const float qnan = __uint_as_float(0x7FC00000u);
  const int64_t mw = m0 + wm * 64, nw = n0 + wn * 64;
  mid_store<ODT>(
      stage_w, lane, mw, nw, g.M, g.N, g.y, g.ldy, g.vec_out,
      [&](int tm) { return g.nan_a && g.nan_a[min<int64_t>(mw + tm * 16 + (lane & 15), g.M - 1)] != 0; },
      [&](int tm, int tn, bool nan_m) {
        v4f v = acc[tm][tn];
        const int64_t n = nw + tn * 16 + (lane >> 4) * 4;
        if (g.bias) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] += load_elem(g.bias, g.bias_dtype, min<int64_t>(n + q, g.N - 1));
        }
        if (g.nan_b) {
#pragma unroll
          for (int q = 0; q < 4; ++q) v[q] = g.nan_b[min<int64_t>(n + q, g.N - 1)] ? qnan : v[q];
        }
        if (nan_m) v = (v4f){qnan, qnan, qnan, qnan};
        return v;
      });
}

struct SmallPlan {
  int mb, nb, wk, ns;
};

// Which kernel a dense product takes (mb = 8: 128x128 tiles; mb = 0: the
// 256x256 tiles of gemm.hip).  The smallest tile whose workgroups all run at
// once (one per compute unit, or two of the 64 KiB ones): a smaller one re-reads
// the operands more often, a larger one leaves compute units idle.  Measured
// (e4m3, bf16 out, in a graph, us; this kernel / 256x256 tiles):
//   N = K = 4096: 5.8 / 30 at 16 rows, 7 / 31 at 48, 9.4 / 33 at 128, 12.6 / 37 at
//   256, 21 / 41 at 512, 36 / 48 at 1003 (128x128 tiles), 42 / 61 at 2048, 85 /
//   63 at 4096; N 1541, K 1000: 3.6 / 15 at 16 rows, 14.5 / 28 at 1003, 19 / 29
//   at 2048, 26 / 34 at 4096; N 18432, K 7168: 30 / 64 at 16 rows, 41 / 64 at 48,
//   79 / 67 at 128.
// Between 128x128 and 256x256 tiles the two estimates decide: 1.3 us a K block
// for a chip full of 128x128 tiles, 1.75 us for 256x256 tiles plus 10 us around
// the loop, or 30 us where a split-K tail exchanges partial tiles.
static SmallPlan small_plan(int64_t M, int64_t N, int nk) {
  const int64_t cus = split_device_cus();
  auto wgs = [&](int64_t rows, int64_t cols) { return cdiv(M, rows) * cdiv(N, cols); };
  // up to four K blocks there is nothing to divide among waves: one wave per
  // tile, its blocks in order (N 4096, K 256: 3.0 / 9.0 at 16 rows, 4.2 / 9.2 at
  // 128, 6.6 / 10.2 at 300; N 1541, K 384: 10.3 / 22 at 1003 rows, where
  // 128x128 tiles take 14)
  if (nk <= 4 && wgs(16, 16) <= 24 * cus) return {1, 1, 1, 3};
  if (wgs(16, 16) <= cus) return {1, 1, 8, 2};
  if (wgs(16, 32) <= cus || M <= 16) return {1, 2, 4, 3};
  if (wgs(32, 32) <= cus) return {2, 2, 4, 3};
  if (wgs(32, 64) <= cus) return {2, 4, 4, 3};
  if (wgs(64, 64) <= cus) return {4, 4, 4, 2};
  if (wgs(64, 64) <= 2 * cus) return {4, 4, 2, 2};
  if (wgs(MID, MID) <= 2 * cus) {
    const SplitPlan sp = split_plan(wgs(256, 256), nk, SPLIT_MIN_BLOCKS);
    const double mid = 1.3 * nk + 4, big = 1.75 * nk / sp.s + (sp.s > 1 ? 30 : 10);
    if (mid < big) return {8, 8, 4, 2};
  }
  return {0, 0, 0, 0};
}

bool small_gemm_fits(int64_t M, int64_t N, int64_t Kp) { return small_plan(M, N, (int)(Kp / BK)).mb != 0; }

template <int GRID, bool B_UNIFORM>
static int small_launch(const char* fn, const SmallPlan& p, const GemmArgs& g, hipStream_t st) {
  if (p.mb == 8) {
    const dim3 grd((unsigned)(cdiv(g.M, MID) * cdiv(g.N, MID))), blk(256);
    if (g.y_dtype == DT_F32)
      gemm_mid_kernel<GRID, B_UNIFORM, DT_F32><<<grd, blk, 0, st>>>(g);
    else if (g.y_dtype == DT_F16)
      gemm_mid_kernel<GRID, B_UNIFORM, DT_F16><<<grd, blk, 0, st>>>(g);
    else
      gemm_mid_kernel<GRID, B_UNIFORM, DT_BF16><<<grd, blk, 0, st>>>(g);
    return check_launch(fn);
  }
  const dim3 grd((unsigned)cdiv(g.N, 16 * p.nb), (unsigned)cdiv(g.M, 16 * p.mb)), blk(64 * p.wk);
#define NTLB_SMALL_CASE(MB, NB, WK, NS)                                                      \
  if (p.mb == MB && p.nb == NB && p.wk == WK && p.ns == NS) {                                \
    gemm_small_kernel<GRID, B_UNIFORM, MB, NB, WK, NS><<<grd, blk, 0, st>>>(g);              \
    return check_launch(fn);                                                                 \
  }
  NTLB_SMALL_CASE(1, 1, 1, 3)
  NTLB_SMALL_CASE(1, 1, 8, 2)
  NTLB_SMALL_CASE(1, 2, 4, 3)
  NTLB_SMALL_CASE(2, 2, 4, 3)
  NTLB_SMALL_CASE(2, 4, 4, 3)
  NTLB_SMALL_CASE(4, 4, 4, 2)
  NTLB_SMALL_CASE(4, 4, 2, 2)
#undef NTLB_SMALL_CASE
  return fail(NTLB_EUNSUPPORTED, "%s: no kernel for a %d x %d tile", fn, 16 * p.mb, 16 * p.nb);
}

int small_gemm_launch(const char* fn, int grid, bool b_uniform, const GemmArgs& g, hipStream_t st) {
  const SmallPlan p = small_plan(g.M, g.N, (int)(g.Kp / BK));
  if (grid == GRID_E4M3)
    return b_uniform ? small_launch<GRID_E4M3, true>(fn, p, g, st) : small_launch<GRID_E4M3, false>(fn, p, g, st);
  return b_uniform ? small_launch<GRID_INT, true>(fn, p, g, st) : small_launch<GRID_INT, false>(fn, p, g, st);
}

// ---------------------------------------------------------------------------
// Per-expert products of few rows each (the expert loop while generating, or
// at small batches).  The 256x256-tile kernels give an expert's 8 rows a whole
// tile: 31/32 of the matrix work is padding and two rounds of tiles of 56 K
// blocks set the time, at 45% of the memory rate the weights could stream at.
// Here a wave owns 16*MB rows by 16*NB columns of one expert over all of K (the
// sums are those of the 256x256 tiles, bit for bit) and streams its weight
// rows through NS LDS stages of its own.
// ---------------------------------------------------------------------------

// Row tile `pid` of experts in order, `rows` rows each: the expert, its first
// row in the tile and its end.  Wave-uniform; false past the last tile.
__device__ __forceinline__ bool expert_tile(const int32_t* offsets, int n_experts, int rows, int pid, int lane, int& e,
                                            int& m0, int& hi) {
  int before = 0;
  for (int base = 0; base < n_experts; base += 64) {
    const int i = base + lane;
    const int lo = i < n_experts ? offsets[i] : 0, end = i < n_experts ? offsets[i + 1] : 0;
    const int tiles = (end - lo + rows - 1) / rows;
    int incl = tiles;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int t = __shfl_up(incl, d);
      if (lane >= d) incl += t;
    }
    const uint64_t hit = __ballot(before + incl > pid);
    if (hit) {
      const int l = __builtin_ctzll(hit);
      e = __builtin_amdgcn_readfirstlane(base + l);
      const int first = before + __shfl(incl, l) - __shfl(tiles, l);
      m0 = __builtin_amdgcn_readfirstlane(__shfl(lo, l) + (pid - first) * rows);
      hi = __builtin_amdgcn_readfirstlane(__shfl(end, l));
      return true;
    }
    before += __shfl(incl, 63);
  }
  return false;
}

__device__ __forceinline__ void take_expert(GemmArgs& g, int e, int hi) {
  g.M = hi;  // rows at or past the expert's end read zero and are not stored
  g.b += (int64_t)e * g.b_estride;
  g.sb += (int64_t)e * g.sb_estride;
  if (g.nan_b) g.nan_b += (int64_t)e * g.N;
}

template <int GRID, int MB, int NB, int NS>
__global__ void __launch_bounds__(256) gemm_small_grouped_kernel(GemmArgs g) {
  constexpr int WB = WaveCopy<MB, NB>::BYTES;
  __shared__ __attribute__((aligned(16))) uint8_t st0[4 * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st1[4 * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st2[NS > 2 ? 4 * WB : 16];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t n0 = ((int64_t)blockIdx.x * 4 + wave) * (16 * NB);
  int e, m0, hi;
  if (n0 >= g.N || !expert_tile(g.offsets, g.n_experts, 16 * MB, (int)blockIdx.y, lane, e, m0, hi)) return;
  take_expert(g, e, hi);
  v4f acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = (v4f){0.f, 0.f, 0.f, 0.f};
  WaveCopy<MB, NB> cp;
  cp.init(g, m0, n0, lane);
  small_k_loop<GRID, true, MB, NB, NS>(g, cp, m0, n0, 0, (int)(g.Kp / BK), st0 + wave * WB, st1 + wave * WB,
                                            st2 + (NS > 2 ? wave * WB : 0), lane, acc);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
      const int64_t m = m0 + mb * 16 + (lane & 15), n = n0 + nb * 16 + (lane >> 4) * 4;
      if (m < g.M && n < g.N) small_store4(g, m, n, acc[mb][nb], g.nan_b);
    }
}

// The gate/up projection with the SwiGLU and h's 1x128 quantization: eight
// waves of 32 columns make the 128 gate and 128 up columns of one h tile; the
// bf16 projections meet in LDS and 16 lanes finish an h tile of a row (the
// arithmetic of gemm.hip's swiglu_quant_rows).
template <int GRID, int MB, int NS, bool SR>
__global__ void __launch_bounds__(512) gemm_small_grouped_swiglu_kernel(GemmArgs g) {
#pragma clang fp contract(off)
  constexpr int WB = WaveCopy<MB, 2>::BYTES;
  static_assert(16 * MB * 512 <= 8 * WB, "the projections fit the first stage");
  __shared__ __attribute__((aligned(16))) uint8_t st0[8 * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st1[8 * WB];
  __shared__ __attribute__((aligned(16))) uint8_t st2[NS > 2 ? 8 * WB : 16];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int e, m0, hi;
  if (!expert_tile(g.offsets, g.n_experts, 16 * MB, (int)blockIdx.y, lane, e, m0, hi)) return;
  take_expert(g, e, hi);
  const int64_t n0 = (int64_t)blockIdx.x * 256, nw = n0 + wave * 32;
  v4f acc[MB][2];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) acc[mb][0] = acc[mb][1] = (v4f){0.f, 0.f, 0.f, 0.f};
  WaveCopy<MB, 2> cp;
  cp.init(g, m0, nw, lane);
  small_k_loop<GRID, true, MB, 2, NS>(g, cp, m0, nw, 0, (int)(g.Kp / BK), st0 + wave * WB, st1 + wave * WB,
                                      st2 + (NS > 2 ? wave * WB : 0), lane, acc);
  __syncthreads();  // every wave is done with its stages
  const float qnan = __uint_as_float(0x7FC00000u);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int r = mb * 16 + (lane & 15);
    const bool nan_m = g.nan_a && g.nan_a[min<int64_t>(m0 + r, g.M - 1)] != 0;
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int c = wave * 32 + nb * 16 + (lane >> 4) * 4;
      float v[4];
#pragma unroll
      for (int q = 0; q < 4; ++q)
        v[q] = nan_m || (g.nan_b && g.nan_b[n0 + c + q] != 0) ? qnan : acc[mb][nb][q];
      // 512-byte rows, 16-byte units swizzled by row
      *reinterpret_cast<uint2*>(st0 + r * 512 + (((c >> 3) ^ (r & 15)) << 4) + (c & 4) * 2) =
          make_uint2((uint32_t)f32_to_bf16_bits(v[0]) | ((uint32_t)f32_to_bf16_bits(v[1]) << 16),
                     (uint32_t)f32_to_bf16_bits(v[2]) | ((uint32_t)f32_to_bf16_bits(v[3]) << 16));
    }
  }
  __syncthreads();
  for (int r = tid >> 4; r < 16 * MB; r += 32) {
    const int64_t m = m0 + r;
    if (m >= g.M) break;  // uniform over the row's 16 lanes
    const int u = tid & 15;  // h columns 8u .. 8u+7 of the tile
    const uint4 gw = *reinterpret_cast<const uint4*>(st0 + r * 512 + ((u ^ (r & 15)) << 4));
    const uint4 uw = *reinterpret_cast<const uint4*>(st0 + r * 512 + (((16 + u) ^ (r & 15)) << 4));
    if (g.gu) {
      uint16_t* gup = g.gu + m * g.ldgu + n0 + u * 8;
      *reinterpret_cast<uint4*>(gup) = gw;
      *reinterpret_cast<uint4*>(gup + 128) = uw;
    }
    const uint32_t gg[4] = {gw.x, gw.y, gw.z, gw.w}, uu[4] = {uw.x, uw.y, uw.z, uw.w};
    float hv[8];
    uint32_t hb[4], amax = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const float gv = bf16_bits_to_f32((gg[q >> 1] >> (16 * (q & 1))) & 0xFFFFu);
      const float uv = bf16_bits_to_f32((uu[q >> 1] >> (16 * (q & 1))) & 0xFFFFu);
      const float sg = bf16_bits_to_f32(f32_to_bf16_bits(gv / (1.0f + expf(-gv))));
      const uint32_t h = f32_to_bf16_bits(sg * uv);
      amax = max(amax, (h & 0x7FFFu) << 16);
      hv[q] = bf16_bits_to_f32(h);
      hb[q >> 1] = (q & 1) ? (hb[q >> 1] | (h << 16)) : h;
    }
    amax = row16_max_u32(amax);
    const float s = scale_from_amax_bits(amax, g.h_qmaxf, g.h_scale_rule);
    const float rs = fast_div_ok<SR>(amax) ? 1.0f / s : 1.0f;
    const int64_t j0 = n0 / 2 + u * 8;
    uint32_t rb[8], lo, hi32;
    float q8[8];
    sr_words<SR>((uint64_t)(m * g.I + j0), g.h_seed, g.h_offset, rb);
    const bool nan = quant8_tile_rs<GRID, SR, false>(hv, amax, s, rs, g.h_qmaxf, rb, lo, hi32, q8);
    *reinterpret_cast<uint2*>(g.hc + m * g.ldhc + j0) = make_uint2(lo, hi32);
    if (g.h) *reinterpret_cast<uint4*>(g.h + m * g.ldh + j0) = make_uint4(hb[0], hb[1], hb[2], hb[3]);
    if (u == 0) {
      g.hs[m * g.hs_row + (n0 / 256) * g.hs_col] = s;
      if (nan && g.h_nan) atomicOr(g.h_nan + m, 1);
    }
  }
}

// Row blocks of 16 per tile for R rows over E experts of N weight rows each, 0
// for the 256x256 tiles.  The rows of each expert are known on the device only,
// so the average decides: skewed counts cost more tiles of one weight, which
// its XCDs' L2 hold.  us, 256x256 tiles | MB 1 | MB 2, rows routed unevenly:
//   gate/up 32 experts 4096 x 7168   average 1: 124 |  86 |  87   4: 224 | 141 | 150   8: 228 | 186 | 166
//     (8 rows: 5.6 TB/s of codes)            16: 230 | 218 | 205  32: 234 | 259 | 237  64: 247 | 406 | 299
//   down 32 experts 7168 x 2048      average 1:  56 |  46 |  46   4: 105 |  88 |  89   8: 135 | 103 |  95
//                                            16: 135 | 118 | 111  32: 137 | 159 | 129  64: 140 | 250 | 187
//   gate/up 8 experts 2048 x 2048            1:  40 |  20 |  19  32:  40 |  19 |  21  64:  47 |  27 |  20  128: 46 | 38 | 35
//   down 8 experts 2048 x 1024               1:  17 |  10 |  10  32:  17 |  10 |  12  64:  19 |  16 |  12  128: 19 | 22 | 21
// So up to 24 rows each, and up to 64 where the 256x256 tiles leave half of
// the chip's 256 compute units without a tile.  The counts themselves would
// move the line only where a few experts get every row: the whole loop at H
// 7168, I 2048, 32 experts, top 8 takes, 256x256 tiles | here, at 24 rows each 417 |
// 313 evenly, 418 | 371 by Zipf(1.2), 186 | 198 with all rows on 8 experts (16
// rows each: 181 | 136).
static int grouped_mb(int64_t R, int64_t E, int64_t N) {
  if (E > 16384) return 0;  // the row tiles are the grid's y
  if (R <= 4 * E) return 1;
  const bool few = (cdiv(R, 256) + E) * cdiv(N, 256) <= 128;
  return R <= (few ? 64 : 24) * E ? 2 : 0;
}

bool small_grouped_fits(int64_t R, int64_t E, int64_t N) { return grouped_mb(R, E, N) != 0; }

template <int GRID>
static void grouped_launch(const GemmArgs& g, hipStream_t st) {
  const int mb = grouped_mb(g.M, g.n_experts, g.N);
  // no more row tiles than rows, and one ragged tile per expert
  const int64_t tiles = std::min<int64_t>(g.M, cdiv(g.M, 16 * mb) + g.n_experts);
  // column workgroups in whole rounds over the XCDs: an expert's row tiles then
  // read the same weight rows through the same L2
  const dim3 grd((unsigned)(cdiv(g.N, 4 * 64) + 7) / 8 * 8, (unsigned)tiles);
  if (mb == 1)
    gemm_small_grouped_kernel<GRID, 1, 4, 3><<<grd, 256, 0, st>>>(g);
  else
    gemm_small_grouped_kernel<GRID, 2, 4, 2><<<grd, 256, 0, st>>>(g);
}

void small_grouped_launch(int grid, const GemmArgs& g, hipStream_t st) {
  if (grid == GRID_E4M3)
    grouped_launch<GRID_E4M3>(g, st);
  else
    grouped_launch<GRID_INT>(g, st);
}

template <int GRID, bool SR>
static void grouped_swiglu_launch(const GemmArgs& g, hipStream_t st) {
  const int mb = grouped_mb(g.M, g.n_experts, g.N);
  const int64_t tiles = std::min<int64_t>(g.M, cdiv(g.M, 16 * mb) + g.n_experts);
  const dim3 grd((unsigned)(g.N / 256), (unsigned)tiles);
  if (mb == 1)
    gemm_small_grouped_swiglu_kernel<GRID, 1, 3, SR><<<grd, 512, 0, st>>>(g);
  else
    gemm_small_grouped_swiglu_kernel<GRID, 2, 2, SR><<<grd, 512, 0, st>>>(g);
}

void small_grouped_swiglu_launch(int grid, const GemmArgs& g, hipStream_t st) {
  if (grid == GRID_E4M3) {
    if (g.h_sr)
      grouped_swiglu_launch<GRID_E4M3, true>(g, st);
    else
      grouped_swiglu_launch<GRID_E4M3, false>(g, st);
  } else {
    if (g.h_sr)
      grouped_swiglu_launch<GRID_INT, true>(g, st);
    else
      grouped_swiglu_launch<GRID_INT, false>(g, st);
  }
}

}  // namespace ntlb
