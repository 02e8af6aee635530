// Weight units of the kernels that fetch 16 rows x 256 columns along the rows and pass each lane
// whole pieces of one row through LDS (gguf_gemv_rows.hip, gguf_gemm_rows.hip): every encoding's
// fetch, piece layout, codes and scales.
#pragma once

#include "gguf_common.h"
#include "gguf_launch.h"

namespace tensor_gguf {
namespace {

typedef float float4v __attribute__((ext_vector_type(4)));

// Bytes 0 and 1 of c as the fp16 subnormal pair (c0, c1) * 2^-24; bytes 2 and 3 likewise.
__device__ __forceinline__ uint32_t sub01(uint32_t c) { return __builtin_amdgcn_perm(0u, c, 0x0C010C00u); }
__device__ __forceinline__ uint32_t sub23(uint32_t c) { return __builtin_amdgcn_perm(0u, c, 0x0C030C02u); }

// The eight byte codes of two dwords less OFFSET as an MFMA operand, times 2^-9.  The subnormals are
// made normal (exact: v_pk_fma_f16, or v_pk_mul_f16 without an offset) since the MFMA aligns a
// product by its operands' exponent fields: with the codes left at 2^-24 its sums lost as many bits
// as the codes have leading zeros (8192 x 2560 fp32 sums against fp64: Q2_K 8.9e-6, Q4_1 4.9e-6, Q8_0 3.4e-7;
// normal, all encodings: 0.7e-7 to 1.0e-7, for 3-4% of a Q4_K layer's time).
template <int OFFSET>
__device__ __forceinline__ half8_t operand(uint32_t lo, uint32_t hi) {
  uint32_t v[4] = {sub01(lo), sub23(lo), sub01(hi), sub23(hi)};
  const half2_t up = {(_Float16)32768.0f, (_Float16)32768.0f};
  const half2_t off = {(_Float16)(-OFFSET / 512.0f), (_Float16)(-OFFSET / 512.0f)};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const half2_t c = as_half2(v[i]);
    v[i] = __builtin_bit_cast(uint32_t, OFFSET != 0 ? __builtin_elementwise_fma(c, up, off) : c * up);
  }
  return __builtin_bit_cast(half8_t, make_uint4(v[0], v[1], v[2], v[3]));
}

constexpr float kTwo9 = 512.0f;  // the codes' 2^-9 is taken out in the scales

// What differs between encodings.  ELEMS: elements of a unit (two blocks, or a quarter super-block); SUB: elements that share a scale;
// MIN: whether w = scale * code + low with low != 0; chunk t of a unit is 8 elements, at chunk_at(t)
// from the unit's first element.
template <int TYPE>
struct Unit {
  static constexpr bool BLOCK32 = Block<TYPE>::QK == 32;
  static constexpr int ELEMS = 64;
  static constexpr int SUB = TYPE == kQ2_K || TYPE == kQ3_K || TYPE == kQ6_K ? 16 : 32;
  static constexpr bool MIN = TYPE == kQ4_1 || TYPE == kQ5_1 || TYPE == kQ4_K || TYPE == kQ5_K || TYPE == kQ2_K;
  static constexpr int WORDS = TYPE == kQ8_0 ? 16 : TYPE == kQ5_K || TYPE == kQ6_K || TYPE == kQ3_K ? 16 : 8;
  // A step of four units is BYTES bytes of each row (eight blocks, or a super-block), fetched as PIECES
  // 16-byte pieces that take ROW bytes of LDS, an odd multiple of 16 so that the lanes of a read
  // (16 rows) start in different banks.
  static constexpr int BYTES = BLOCK32 ? 8 * Block<TYPE>::BYTES : Block<TYPE>::BYTES;
  static constexpr int PIECES = (BYTES + 15) / 16;
  static constexpr int ROW = 16 * (PIECES | 1);
  static constexpr int LOADS = (16 * PIECES + 63) / 64;  // of 16 bytes a lane, for one 16-row tile
  uint32_t q[WORDS];  // code bytes (Q5_K, Q6_K, Q3_K: low parts, then the 8 dwords of high bits)
  uint32_t h[4];      // scales, fifth bits and factors

  // Element offset in LDS of the unit that lane group g takes of a step, from the step's first.
  static __device__ __forceinline__ int lane_at(int g) {
    return TYPE == kQ6_K ? 128 * (g >> 1) + 32 * (g & 1) : ELEMS * g;
  }
  static constexpr int chunk_at(int t) { return TYPE == kQ6_K && t >= 4 ? 64 + 8 * (t - 4) : 8 * t; }

  // Read lane group g's unit from its row's pieces in LDS.
  __device__ __forceinline__ void read(const uint8_t* row, int g) {
    if constexpr (BLOCK32) {
      constexpr int B = Block<TYPE>::BYTES, W = B / 2;  // dwords of two blocks
      const uint32_t* p = reinterpret_cast<const uint32_t*>(row + 2 * B * g);
      uint32_t v[W];
#pragma unroll
      for (int i = 0; i < W; ++i) v[i] = p[i];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        // dword at byte i of block b: B is even, so a block starts at byte 0 or 2 of a dword
        auto at = [&](int i) {
          const int byte = b * B + i;
          return byte % 4 ? __builtin_amdgcn_alignbyte(v[byte / 4 + 1], v[byte / 4], 2) : v[byte / 4];
        };
        constexpr int qs = TYPE == kQ5_1 ? 8 : TYPE == kQ5_0 ? 6 : TYPE == kQ4_1 ? 4 : 2;
        h[b] = b * B % 4 ? v[b * B / 4] >> 16 : v[b * B / 4];
        if constexpr (MIN) h[b] = at(0);
        if constexpr (TYPE == kQ5_0 || TYPE == kQ5_1) h[2 + b] = at(qs - 4);
#pragma unroll
        for (int i = 0; i < WORDS / 2; ++i) q[WORDS / 2 * b + i] = at(qs + 4 * i);
      }
    } else {
      const uint8_t* p = row;
      const int part = g;
      const uint8_t* lo;
      const uint8_t* hi = nullptr;
      if constexpr (TYPE == kQ4_K || TYPE == kQ5_K) {
        const uint4 head = *reinterpret_cast<const uint4*>(p);
        h[0] = head.x, h[1] = head.y, h[2] = head.z, h[3] = head.w;
        lo = p + (TYPE == kQ4_K ? 16 : 48) + 32 * part;
        hi = p + 16;
      } else if constexpr (TYPE == kQ6_K) {
        lo = p + 32 * part;  // 64 h + 32 c
        hi = p + 128 + 32 * (part >> 1);
        const uint2 s = *reinterpret_cast<const uint2*>(p + 192 + 8 * (part >> 1));
        h[0] = s.x, h[1] = s.y, h[2] = *reinterpret_cast<const uint16_t*>(p + 208);
      } else if constexpr (TYPE == kQ2_K) {
        lo = p + 16 + 32 * (part >> 1);
        h[0] = *reinterpret_cast<const uint32_t*>(p + 4 * part);
        h[2] = *reinterpret_cast<const uint32_t*>(p + 80);
      } else {
        lo = p + 32 + 32 * (part >> 1);
        hi = p;
        const uint4 s = *reinterpret_cast<const uint4*>(p + 96);  // 12 scale bytes, d
        h[0] = s.x, h[1] = s.y, h[2] = s.z, h[3] = s.w & 0xFFFFu;
      }
      const uint4 a = *reinterpret_cast<const uint4*>(lo), b = *reinterpret_cast<const uint4*>(lo + 16);
      q[0] = a.x, q[1] = a.y, q[2] = a.z, q[3] = a.w, q[4] = b.x, q[5] = b.y, q[6] = b.z, q[7] = b.w;
      if constexpr (WORDS == 16) {
        const uint4 e = *reinterpret_cast<const uint4*>(hi), f = *reinterpret_cast<const uint4*>(hi + 16);
        q[8] = e.x, q[9] = e.y, q[10] = e.z, q[11] = e.w, q[12] = f.x, q[13] = f.y, q[14] = f.z, q[15] = f.w;
      }
    }
  }

  // MFMA operand of chunk t; part: the unit's index in its super-block (the lane group).
  template <int T>
  __device__ __forceinline__ half8_t chunk(int part) const {
    if constexpr (TYPE == kQ8_0) {
      return operand<128>(q[2 * T] ^ 0x80808080u, q[2 * T + 1] ^ 0x80808080u);
    } else if constexpr (BLOCK32) {
      constexpr int b = T >> 2, w = 4 * b + 2 * (T & 1);
      constexpr int shift = (T & 2) ? 4 : 0;
      uint32_t lo = (q[w] >> shift) & 0x0F0F0F0Fu, hi = (q[w + 1] >> shift) & 0x0F0F0F0Fu;
      if constexpr (TYPE == kQ5_0 || TYPE == kQ5_1) {
        constexpr int bit = 8 * (T & 3);  // chunk T is elements 8 (T & 3) of the block
        lo |= fifth_bits(h[2 + b] >> bit);
        hi |= fifth_bits(h[2 + b] >> (bit + 4));
      }
      return operand<TYPE == kQ4_0 ? 8 : TYPE == kQ5_0 ? 16 : 0>(lo, hi);
    } else if constexpr (TYPE == kQ2_K) {
      constexpr int w = 2 * (T & 3);
      const int shift = 4 * (part & 1) + 2 * (T >> 2);  // plane 2 c + T / 4 of half h, part = 2 h + c
      return operand<0>((q[w] >> shift) & 0x03030303u, (q[w + 1] >> shift) & 0x03030303u);
    } else if constexpr (TYPE == kQ3_K) {
      constexpr int w = 2 * (T & 3);
      const int shift = 4 * (part & 1) + 2 * (T >> 2), bit = 2 * part + (T >> 2);
      const uint32_t lo = ((q[w] >> shift) & 0x03030303u) | (((q[8 + w] >> bit) & 0x01010101u) << 2);
      const uint32_t hi = ((q[w + 1] >> shift) & 0x03030303u) | (((q[9 + w] >> bit) & 0x01010101u) << 2);
      return operand<4>(lo, hi);
    } else {  // Q4_K, Q5_K, Q6_K: low nibbles, then high nibbles
      constexpr int w = 2 * (T & 3), high = T >> 2;
      uint32_t lo = (q[w] >> (4 * high)) & 0x0F0F0F0Fu, hi = (q[w + 1] >> (4 * high)) & 0x0F0F0F0Fu;
      if constexpr (TYPE == kQ5_K) {
        const int bit = 2 * part + high;
        lo |= ((q[8 + w] >> bit) & 0x01010101u) << 4;
        hi |= ((q[9 + w] >> bit) & 0x01010101u) << 4;
      }
      if constexpr (TYPE == kQ6_K) {
        const int bit = 2 * (part & 1) + 4 * high;
        lo |= ((q[8 + w] >> bit) & 0x03030303u) << 4;
        hi |= ((q[9 + w] >> bit) & 0x03030303u) << 4;
      }
      return operand<TYPE == kQ6_K ? 32 : 0>(lo, hi);
    }
  }

  // Scale (times 2^9) and low value of sub-block s of the unit, zero where the unit (or the
  // second block of one) lies past the row's end.
  template <int S>
  __device__ __forceinline__ void scale(int part, bool valid, bool valid2, float& sc, float& low) const {
    low = 0.0f;
    if constexpr (BLOCK32) {
      const bool in = S == 0 ? valid : valid2;
      const uint32_t head = in ? h[S] : 0u;
      sc = half_bits_to_float(head) * kTwo9;
      if constexpr (MIN) low = half_bits_to_float(head >> 16);
    } else if constexpr (TYPE == kQ4_K || TYPE == kQ5_K) {
      const uint32_t dd = valid ? h[0] : 0u;
      int sc_lo, mn_lo, sc_hi, mn_hi;
      q4k_scale_pair(h[1], h[2], h[3], part, sc_lo, mn_lo, sc_hi, mn_hi);
      sc = half_bits_to_float(dd) * (kTwo9 * (float)(S ? sc_hi : sc_lo));
      low = -half_bits_to_float(dd >> 16) * (float)(S ? mn_hi : mn_lo);
    } else if constexpr (TYPE == kQ6_K) {
      // bytes 2 c, 2 c + 1 (sub-blocks 0, 1) and 2 c + 4, 2 c + 5 (2, 3) of the half's eight
      const uint32_t pair = (S < 2 ? h[0] : h[1]) >> (16 * (part & 1));
      const float d = half_bits_to_float(valid ? h[2] : 0u);
      sc = d * (kTwo9 * (float)(int8_t)((pair >> (8 * (S & 1))) & 0xFFu));
    } else if constexpr (TYPE == kQ2_K) {
      const uint32_t dd = valid ? h[2] : 0u;
      const uint32_t byte = h[0] >> (8 * S);
      sc = half_bits_to_float(dd) * (kTwo9 * (float)(byte & 15u));
      low = -half_bits_to_float(dd >> 16) * (float)((byte >> 4) & 15u);
    } else {  // Q3_K: sub-block 4 part + S of the super-block
      const float d = half_bits_to_float(valid ? h[3] : 0u);
      const uint32_t nib = ((part & 1 ? h[1] : h[0]) >> (8 * S)) >> (4 * (part >> 1));
      const uint32_t top = (h[2] >> (8 * S)) >> (2 * part);
      sc = d * (kTwo9 * (float)((int)((nib & 15u) | ((top & 3u) << 4)) - 32));
    }
  }
};

// v shifted down by d bytes, zeros in from above.
__device__ __forceinline__ uint4 shift_bytes(uint4 v, uint32_t d) {
  if (d & 8) v = make_uint4(v.z, v.w, 0u, 0u);
  if (d & 4) v = make_uint4(v.y, v.z, v.w, 0u);
  const uint32_t b = d & 3u;
  v = make_uint4(__builtin_amdgcn_alignbyte(v.y, v.x, b), __builtin_amdgcn_alignbyte(v.z, v.y, b),
                 __builtin_amdgcn_alignbyte(v.w, v.z, b), __builtin_amdgcn_alignbyte(0u, v.w, b));
  return d < 16u ? v : make_uint4(0u, 0u, 0u, 0u);
}

// A wave's fetch of one step of a 16-row tile: 16-byte pieces, consecutive lanes along a row.
template <int TYPE>
struct Fetch {
  using U = Unit<TYPE>;
  static constexpr int PIECES = U::PIECES;
  const uint8_t* w;          // the tile's first row
  uint32_t last_from;        // the largest byte offset of a piece in step 0
  uint32_t end;              // bytes from there to the end of the matrix
  uint32_t from[U::LOADS];   // byte offsets of the lane's pieces in step 0
  uint32_t step_at;          // byte offset of the step in v from step 0
  bool ragged;               // whether a piece of that step may pass the matrix's end (wave-uniform)
  uint4 v[U::LOADS];

  __device__ __forceinline__ void init(const uint8_t* matrix, int row0, int n, uint32_t row_bytes, int lane) {
    w = matrix + (size_t)row0 * row_bytes;
    end = (uint32_t)min((size_t)(n - row0) * row_bytes, (size_t)0xFFFFFFF0u);
    last_from = (uint32_t)min(15, n - 1 - row0) * row_bytes + (uint32_t)(16 * (PIECES - 1));
#pragma unroll
    for (int i = 0; i < U::LOADS; ++i) {
      const int piece = min(i * 64 + lane, 16 * PIECES - 1);
      const int r = piece / PIECES, c = piece - r * PIECES;
      from[i] = (uint32_t)min(r, n - 1 - row0) * row_bytes + (uint32_t)(16 * c);
    }
  }
  // A piece that would pass the end of the matrix is read as the matrix's last 16 bytes and moved
  // into place when it is stored (only the last tile has such pieces).
  __device__ __forceinline__ void load(int step) {
    step_at = (uint32_t)(step * U::BYTES);
    ragged = last_from + step_at + 16u > end;
#pragma unroll
    for (int i = 0; i < U::LOADS; ++i) v[i] = load16(w + min(from[i] + step_at, end - 16u));
  }
  __device__ __forceinline__ void store(uint8_t* lds, int lane) {
    if (ragged) {
#pragma unroll
      for (int i = 0; i < U::LOADS; ++i) {
        const uint32_t at = from[i] + step_at;
        v[i] = shift_bytes(v[i], at - min(at, end - 16u));
      }
    }
#pragma unroll
    for (int i = 0; i < U::LOADS; ++i) {
      const int piece = i * 64 + lane;
      const int r = piece / PIECES, c = piece - r * PIECES;
      if ((i + 1) * 64 <= 16 * PIECES || piece < 16 * PIECES) *reinterpret_cast<uint4*>(lds + r * U::ROW + 16 * c) = v[i];
    }
  }
};

// a / b for 0 <= a < 2^20 from inv = 1 / b (v_rcp_f32): an integer division costs tens of dependent
// instructions, several of which in a row were a third of a small launch.
__device__ __forceinline__ float inverse(int b) { return __builtin_amdgcn_rcpf((float)b); }
__device__ __forceinline__ int quotient(int a, float inv) { return (int)(((float)a + 0.5f) * inv); }
__device__ __forceinline__ int scalar(int v) { return __builtin_amdgcn_readfirstlane(v); }

}  // namespace
}  // namespace tensor_gguf
