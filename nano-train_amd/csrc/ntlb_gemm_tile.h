// What the blockwise-scaled GEMM kernels share (gemm.hip: 256x256 tiles;
// gemm_small.hip: 16x16 to 128x128 tiles): the launch arguments, the swizzled
// LDS tile layout with its fragment reads, and the MFMA of one 128-wide K
// block.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "ntlb_device.h"
#include "ntlb_quant8.h"

namespace ntlb {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v2bf __attribute__((ext_vector_type(2)));

struct GemmArgs {
  const uint8_t* a;
  int64_t lda;
  const float* sa;
  int64_t sa_row, sa_col;
  int a_shift;
  const uint8_t* b;
  int64_t ldb;
  const float* sb;
  int64_t sb_row, sb_col;
  int b_shift;
  int64_t M, N, Kp;
  const void* bias;
  int bias_dtype;
  void* y;
  int y_dtype;
  int64_t ldy;
  const int32_t* nan_a;
  const int32_t* nan_b;
  int vec_out;  // y 16-byte aligned with 16-byte row pitch
  // grouped (per-expert) mode: rows of A sorted by expert, expert e owns rows
  // [offsets[e], offsets[e+1]) and multiplies B + e*b_estride (codes) with
  // scales sb + e*sb_estride
  const int32_t* offsets;
  int n_experts;
  int64_t b_estride, sb_estride;
  // SwiGLU epilogue (EPI_SWIGLU): B's rows come in 128-row blocks alternating
  // gate block t and up block t, so output tile columns [0,128) are gate and
  // [128,256) up for h columns n0/2 + [0,128).  h = bf16(silu(bf16(gate)) *
  // bf16(up)) is quantized per 1x128 tile (one tile per output tile row).
  uint16_t* h;    // optional bf16 h [M, I], row stride ldh
  int64_t ldh;
  uint8_t* hc;    // h codes [M, ldhc]
  int64_t ldhc;
  float* hs;      // h scales: hs[row * hs_row + tile * hs_col]
  int64_t hs_row, hs_col;
  int32_t* h_nan;  // optional per-row NaN flags of h
  uint16_t* gu;   // optional bf16 gate / up outputs [M, 2I] in B's interleaved column order, row stride ldgu
  int64_t ldgu;
  float h_qmaxf;
  int h_sr, h_scale_rule;
  uint64_t h_seed, h_offset;
  int64_t I;  // width of h = N / 2
  // Split-K tail (dense, EPI_STORE): workgroups at or past split_base take K
  // chunk (q % split_s) of tile split_base + q / split_s, q = pid - split_base;
  // the chunks' fp32 partials meet in ws and the last one to finish sums them
  // in chunk order and stores the tile.
  int split_base, split_s;
  float* ws;             // [tail tiles][split_s][NTHREADS * 128] fp32
  uint32_t* ws_count;    // per tail tile; zero between calls (the kernel resets it)
};

// Epilogues: store the tile as bf16 (EPI_STORE), fp32 or fp16, or the
// SwiGLU + 1x128 quantization of the expert MLP.  The output dtype is part of
// the kernel so that each kernel holds one straight-line store path.
constexpr int EPI_STORE = 0, EPI_SWIGLU = 1, EPI_STORE_F32 = 2, EPI_STORE_F16 = 3;

constexpr int BK = 128;  // K block: one scale block

typedef __attribute__((address_space(3))) void* lds_ptr_t;

// Byte offset of 16-byte chunk c of row r inside a swizzled [rows][128] tile.
// A fragment read has 16 lanes read 16 consecutive rows at one logical chunk;
// the permutation f(r) = (r & 7) ^ bit3(r) gives rows 0-7 eight distinct
// chunks (conflict-free in 8-lane phases over 128 bytes of banks) and gives
// every 16-row window distinct (row parity, chunk) pairs (conflict-free in
// 16-lane phases over 256 bytes of banks).
__device__ __forceinline__ int swz_perm(int r) { return (r & 7) ^ ((r >> 3) & 1); }
__device__ __forceinline__ int swz(int r, int c) { return r * BK + ((c ^ swz_perm(r)) << 4); }

// MFMA fragment of 16 rows: row = lane%16, 32 K bytes of group lane/16.
// Both operands use the same (lane group, byte) -> K mapping, so the products pair up.
__device__ __forceinline__ v8i load_frag(const uint8_t* tile, int row0, int lane) {
  const int r = row0 + (lane & 15);
  const int g = lane >> 4;
  const uint4 lo = *reinterpret_cast<const uint4*>(tile + swz(r, 2 * g));
  const uint4 hi = *reinterpret_cast<const uint4*>(tile + swz(r, 2 * g + 1));
  v8i f;
  f[0] = (int)lo.x; f[1] = (int)lo.y; f[2] = (int)lo.z; f[3] = (int)lo.w;
  f[4] = (int)hi.x; f[5] = (int)hi.y; f[6] = (int)hi.z; f[7] = (int)hi.w;
  return f;
}

// D[i][j] = sum_k P[i][k] Q[j][k] for a 16x16 tile; lane l holds D[4*(l/16)+r][l%16]
template <int GRID>
__device__ __forceinline__ v4f mma_block(const v8i& p, const v8i& q) {
  if constexpr (GRID == GRID_E4M3) {
    v4f z = {0.f, 0.f, 0.f, 0.f};
    // fmt 0 = e4m3 for both operands.  Zero scale operands select the
    // unscaled encoding (v_mfma_f32_16x16x128_f8f6f4, no v_mfma_ld_scale
    // prefix); its products equal those of unit e8m0 scales (127) bit for bit
    // over the whole config-2 output, and the c2 GEMM runs 1.5% faster.
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(p, q, z, 0, 0, 0, 0, 0, 0);
  } else {
    v4i z = {0, 0, 0, 0};
    v4i p0 = {p[0], p[1], p[2], p[3]}, p1 = {p[4], p[5], p[6], p[7]};
    v4i q0 = {q[0], q[1], q[2], q[3]}, q1 = {q[4], q[5], q[6], q[7]};
    v4i s = __builtin_amdgcn_mfma_i32_16x16x64_i8(p0, q0, z, 0, 0, 0);
    s = __builtin_amdgcn_mfma_i32_16x16x64_i8(p1, q1, s, 0, 0, 0);
    v4f f = {(float)s[0], (float)s[1], (float)s[2], (float)s[3]};
    return f;
  }
}

// The raw MFMA result of one 16x16 block over one K block (fp32 for e4m3,
// int32 for the int grid: at most 128 * 127^2 in magnitude, exact in fp32)
// and its conversion, so that a pipelined promotion can keep the raw form
// until it is consumed.
template <int GRID>
using raw_t = typename std::conditional<GRID == GRID_E4M3, v4f, v4i>::type;

template <int GRID>
__device__ __forceinline__ raw_t<GRID> mma_raw(const v8i& p, const v8i& q) {
  if constexpr (GRID == GRID_E4M3) {
    return mma_block<GRID>(p, q);
  } else {
    v4i z = {0, 0, 0, 0};
    v4i p0 = {p[0], p[1], p[2], p[3]}, p1 = {p[4], p[5], p[6], p[7]};
    v4i q0 = {q[0], q[1], q[2], q[3]}, q1 = {q[4], q[5], q[6], q[7]};
    v4i s = __builtin_amdgcn_mfma_i32_16x16x64_i8(p0, q0, z, 0, 0, 0);
    return __builtin_amdgcn_mfma_i32_16x16x64_i8(p1, q1, s, 0, 0, 0);
  }
}

template <int GRID>
__device__ __forceinline__ v4f raw_f32(const raw_t<GRID>& r) {
  if constexpr (GRID == GRID_E4M3) {
    return r;
  } else {
    return (v4f){(float)r[0], (float)r[1], (float)r[2], (float)r[3]};
  }
}

// the split-K tail's minimum K blocks per range (K 1024, 8 blocks: 25 us
// split, 16 unsplit)
constexpr int SPLIT_MIN_BLOCKS = 9;

// host side (gemm_small.hip): launch the few-row / few-tile kernels when they
// are the better choice for the shape; false leaves the product to the
// 256x256-tile kernel
bool small_gemm_fits(int64_t M, int64_t N, int64_t Kp);
int small_gemm_launch(const char* fn, int grid, bool b_uniform, const GemmArgs& g, hipStream_t st);

// the same for per-expert products: M_total rows over n_experts experts of N
// weight rows, B's scale uniform over a wave's columns
bool small_grouped_fits(int64_t M_total, int64_t n_experts, int64_t N);
void small_grouped_launch(int grid, const GemmArgs& g, hipStream_t st);
void small_grouped_swiglu_launch(int grid, const GemmArgs& g, hipStream_t st);

}  // namespace ntlb
