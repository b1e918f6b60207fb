// What the GEMMs on tiles below 256x256 share (gemm_small.hip: quantized codes;
// gemm_bf16.hip: bf16 operands): the wait for copies in flight, the sum of a
// workgroup's partial tiles, and the raster and the stores of 128x128 tiles.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "ntlb_device.h"

namespace ntlb {

// s_waitcnt with only vmcnt set
constexpr int vmcnt_imm(int n) { return (n & 15) | (7 << 4) | (15 << 8) | ((n >> 4) << 14); }

// The WK waves' partial tiles of 16*MB x 16*NB (acc[mb][nb]: lane l holds row
// 16*mb + l%16, columns 16*nb + 4*(l/16) + 0..3) meet in red and are summed in
// wave order; store(m, n, v) gets row m, columns n .. n+3 of the result.  Every
// thread of the workgroup must call it, with nothing in flight into red.
template <int MB, int NB, int WK, typename V4, typename Store>
__device__ __forceinline__ void sum_partials(V4* red, const V4 (&acc)[MB][NB], int wave, int lane, int64_t m0,
                                             int64_t n0, int64_t M, int64_t N, Store store) {
  __syncthreads();  // every wave is done with its stages: the partials go where the first one was
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) red[(wave * MB * NB + mb * NB + nb) * 64 + lane] = acc[mb][nb];
  __syncthreads();
  for (int q = threadIdx.x; q < MB * NB * 64; q += 64 * WK) {
    const int b = q >> 6, l = q & 63;
    V4 v = red[q];
#pragma unroll
    for (int w = 1; w < WK; ++w) v += red[w * MB * NB * 64 + q];
    const int64_t m = m0 + (b / NB) * 16 + (l & 15);
    const int64_t n = n0 + (b % NB) * 16 + (l >> 4) * 4;
    if (m < M && n < N) store(m, n, v);
  }
}

constexpr int MID = 128;  // rows and columns of the tiles below: four waves as 2 x 2, each 64x64

// The tile of this workgroup: each XCD walks a contiguous range of a raster of
// four row tiles
__device__ __forceinline__ void mid_tile(int64_t M, int64_t N, int64_t& m0, int64_t& n0) {
  const int num_n = (int)((N + MID - 1) / MID), num_m = (int)((M + MID - 1) / MID);
  const int nwg = (int)gridDim.x, xcd = (int)blockIdx.x & 7, local = (int)blockIdx.x >> 3;
  const int per = nwg >> 3, extra = nwg & 7;
  const int pid = xcd * per + min(xcd, extra) + local;
  constexpr int GROUP_M = 4;
  const int group = pid / (GROUP_M * num_n);
  const int gsize = min(num_m - group * GROUP_M, GROUP_M);
  const int in_group = pid - group * GROUP_M * num_n;
  m0 = (int64_t)(group * GROUP_M + in_group % gsize) * MID;
  n0 = (int64_t)(in_group / gsize) * MID;
}

// Stores a wave's 64x64 part of the tile, at row m0 and column n0: 32 of its
// rows at a time staged in the wave's 16 KiB of LDS and stored as whole 128-byte
// (fp32: 256-byte) row segments.  value(tm, tn, row(tm)) gives the block (tm, tn).
template <int ODT, typename Row, typename Value>
__device__ __forceinline__ void mid_store(uint8_t* stage_w, int lane, int64_t m0, int64_t n0, int64_t M, int64_t N,
                                          void* y, int64_t ldy, int vec_out, Row row, Value value) {
  typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
  constexpr int esz = ODT == DT_F32 ? 4 : 2, pitch = 64 * esz + 16, cpr = 64 * esz / 16, epc = 16 / esz;
  static_assert(32 * pitch <= MID * 128, "staged rows fit a stage");
#pragma unroll
  for (int part = 0; part < 2; ++part) {
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const auto of_row = row(part * 2 + t);
#pragma unroll
      for (int tn = 0; tn < 4; ++tn) {
        const auto v = value(part * 2 + t, tn, of_row);
        uint8_t* dst = stage_w + (t * 16 + (lane & 15)) * pitch + (tn * 16 + (lane >> 4) * 4) * esz;
        if constexpr (ODT == DT_F32) {
          *reinterpret_cast<std::remove_const_t<decltype(v)>*>(dst) = v;
        } else if constexpr (ODT == DT_BF16) {
          const v2bf p0 = {(__bf16)v[0], (__bf16)v[1]}, p1 = {(__bf16)v[2], (__bf16)v[3]};
          *reinterpret_cast<uint2*>(dst) =
              make_uint2(__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1));
        } else {
          const __half h[4] = {f32_to_f16(v[0]), f32_to_f16(v[1]), f32_to_f16(v[2]), f32_to_f16(v[3])};
          *reinterpret_cast<uint2*>(dst) = *reinterpret_cast<const uint2*>(h);
        }
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): this wave's staging writes are done
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < cpr / 2; ++j) {
      const int q = lane + 64 * j, r = q / cpr, c = q % cpr;
      const int64_t m = m0 + part * 32 + r, n = n0 + c * epc;
      const uint8_t* src = stage_w + r * pitch + c * 16;
      if (m >= M || n >= N) continue;
      uint8_t* ydst = reinterpret_cast<uint8_t*>(y) + (m * ldy + n) * esz;
      if (vec_out && n + epc <= N) {
        store16_nt(ydst, src);
      } else {
        using E = std::conditional_t<esz == 4, uint32_t, uint16_t>;
#pragma nounroll
        for (int e = 0; e < epc && n + e < N; ++e)
          reinterpret_cast<E*>(ydst)[e] = reinterpret_cast<const E*>(src)[e];
      }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // the re-reads are done before the next part overwrites
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace ntlb
