// Matrix-core products of activation rows against row-major weights, shared by
// the kernels that take more than a few token rows.
//
// A "unit" is 16 bytes of one row: 8 bf16 or 4 float. A k-step is 4 units of
// every row of a 16-row operand: lane l holds unit 4 step + l / 16 of row
// l % 16, so both operands of a product are plain 16-byte loads of row-major
// memory and no operand is rearranged. A bf16 step is one 16x16x32 MFMA; a
// float step is four 16x16x4 MFMAs, the i-th on element i of every lane's unit
// (the same four k on both sides). Results: row 4 (l / 16) + i of the first
// operand, row l % 16 of the second.
#pragma once

#include "common.h"

// element i (0..VE-1) of a 16-byte unit as float, and back
template <typename T> struct Chunk;
template <> struct Chunk<bf16_t> {
  static constexpr int VE = 8;
  __device__ __forceinline__ static float get(const uint4& c, int i) {
    const unsigned w = i < 2 ? c.x : i < 4 ? c.y : i < 6 ? c.z : c.w;
    return __uint_as_float((i & 1) ? (w & 0xffff0000u) : (w << 16));
  }
  __device__ __forceinline__ static uint4 pack(const float* v) {
    return make_uint4(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                      pack_bf16x2(v[6], v[7]));
  }
};
template <> struct Chunk<float> {
  static constexpr int VE = 4;
  __device__ __forceinline__ static float get(const uint4& c, int i) {
    return __uint_as_float(i == 0 ? c.x : i == 1 ? c.y : i == 2 ? c.z : c.w);
  }
  __device__ __forceinline__ static uint4 pack(const float* v) {
    return make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
  }
};

// The accumulators of one 16x16 result. Float products are summed in blocks:
// block() closes one (four partial sums of the block's steps, then their total
// onto the running sum), so that no sum is a long serial chain. bf16 products
// carry their 8-bit operands' error and take the chain.
template <typename T> struct RowAcc;
template <> struct RowAcc<bf16_t> {
  f32x4_t c = {0.f, 0.f, 0.f, 0.f};
  __device__ __forceinline__ void step(const uint4& a, const uint4& b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0,
                                                0, 0);
  }
  __device__ __forceinline__ void block() {}
  __device__ __forceinline__ f32x4_t sum() const { return c; }
};
template <> struct RowAcc<float> {
  f32x4_t total = {0.f, 0.f, 0.f, 0.f};
  f32x4_t c[4] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  __device__ __forceinline__ void step(const uint4& a, const uint4& b) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      c[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(Chunk<float>::get(a, i), Chunk<float>::get(b, i), c[i], 0, 0, 0);
  }
  __device__ __forceinline__ void block() {
    total += (c[0] + c[1]) + (c[2] + c[3]);
#pragma unroll
    for (int i = 0; i < 4; ++i) c[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ f32x4_t sum() const { return total + ((c[0] + c[1]) + (c[2] + c[3])); }
};

// 16 rows of 64 units (rows[r]: unit `lane` of row r, so that each load was 1 KB
// of one row) as the operands of 16 k-steps, through a wave's own LDS; no
// barrier, the wave reads what it wrote. Loads in the operand's own shape (16
// rows x 64 bytes) measured well below loads of whole lines: the many-row
// hyper-connection product (bf16, 2000 rows) took 46 us with them at any number
// of workgroups and 33 with lines through LDS; the mix of 14 rows 12.3 and 10.9.
constexpr int ROW_US = 65;         // LDS row stride in units: 64 and one of padding
__device__ __forceinline__ void to_frags(uint4* lds, const u32x4_t (&rows)[16], int lane, int r16, int g4,
                                         u32x4_t (&f)[16]) {
#pragma unroll
  for (int r = 0; r < 16; ++r) *reinterpret_cast<u32x4_t*>(lds + r * ROW_US + lane) = rows[r];
#pragma unroll
  for (int i = 0; i < 16; ++i) f[i] = *reinterpret_cast<const u32x4_t*>(lds + r16 * ROW_US + 4 * i + g4);
}

// 4 consecutive activations as float, and back
__device__ __forceinline__ void load_act4(const bf16_t* p, float (&v)[4]) {
  const uint2 u = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(u.x << 16); v[1] = __uint_as_float(u.x & 0xffff0000u);
  v[2] = __uint_as_float(u.y << 16); v[3] = __uint_as_float(u.y & 0xffff0000u);
}
__device__ __forceinline__ void load_act4(const float* p, float (&v)[4]) {
  const float4 u = *reinterpret_cast<const float4*>(p);
  v[0] = u.x; v[1] = u.y; v[2] = u.z; v[3] = u.w;
}
__device__ __forceinline__ void store_act4(bf16_t* p, const float (&v)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
}
__device__ __forceinline__ void store_act4(float* p, const float (&v)[4]) {
  *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
}
