// The pipelined fused dequant-GEMM kernel of gguf_gemm_pipe.hip and the launch of one tile, shared by
// its translation units (one for the encodings with plans, one for the others: they compile in
// parallel).
#pragma once

#include <algorithm>

#include "gguf_common.h"
#include "gguf_launch.h"

namespace tensor_gguf {
namespace pipe {

constexpr int BK = 64, ROW = 80;  // halves per LDS row (16-byte aligned, padded)
constexpr float kTwo24 = 16777216.0f, kTwo20 = 1048576.0f;

// fp16(scale * q + bias) for four codes q < 1024 given as fp16 subnormal pairs
// p02 = (q0, q2) * 2^-24 and p13 = (q1, q3) * 2^-24 (a code masked into the low
// bits of a half is that subnormal exactly). With scale24 = scale * 2^24 each
// product is exactly scale * q and the fma rounds once to fp32 as fmaf(scale, q,
// bias) does (one fp32-result v_fma_mix per element); each pair is then rounded to
// fp16 by one packed conversion, so the fp16 weight is the cast of the fp32 value.
__device__ __forceinline__ uint2 affine4(uint32_t p02, uint32_t p13, float scale24, float bias) {
  const half2_t a = as_half2(p02), b = as_half2(p13);
  return make_uint2(half2_from_fp32(fmaf((float)a[0], scale24, bias), fmaf((float)b[0], scale24, bias)),
                    half2_from_fp32(fmaf((float)a[1], scale24, bias), fmaf((float)b[1], scale24, bias)));
}

template <int TYPE, int TPR>
struct Geometry;

// Q4_K: TPR threads per weight row share the 32 quant bytes of the step's pair.
template <int TPR>
struct Geometry<kQ4_K, TPR> {
  static constexpr int QB = 32 / TPR;  // quant bytes per thread
  static constexpr int W0 = QB / 4, W1 = 4;  // dwords: quants, header
};

// Q5_K: Q4_K's slices plus the fifth-bit bytes at the same positions of the 32-byte qh run.
template <int TPR>
struct Geometry<kQ5_K, TPR> {
  static constexpr int QB = 32 / TPR;
  static constexpr int W0 = QB / 4, W1 = 4 + QB / 4;  // dwords: quants; header, then fifth bits
};

// Q6_K: TPR threads per weight row, each EPT = 64 / TPR consecutive elements.
template <int TPR>
struct Geometry<kQ6_K, TPR> {
  static constexpr int EPT = 64 / TPR;
  static constexpr int W0 = EPT / 4, W1 = EPT / 4 + 2;  // ql dwords; qh dwords + scales + d
};

// Q8_0 / Q4_0: a step is two 32-element blocks (68 / 36 bytes).  TPR threads per weight row
// share the step's quant bytes (64 / 32): thread p takes QB of them, all in block
// QB p / QPB at byte QB p % QPB (QPB = quant bytes per block), and that block's fp16 d.
template <int TPR>
struct Geometry<kQ8_0, TPR> {
  static constexpr int QPB = 32, QB = 2 * QPB / TPR;
  static constexpr int W0 = QB / 4, W1 = 2;  // dwords: quants; d (low half), unused
};
template <int TPR>
struct Geometry<kQ4_0, TPR> {
  static constexpr int QPB = 16, QB = 2 * QPB / TPR;
  static constexpr int W0 = QB / 4, W1 = 2;
};
// Q4_1, Q5_0, Q5_1: Q4_0's plan with a minimum beside d (Q4_1, Q5_1) and the block's 32 fifth bits.
template <int TPR>
struct Geometry<kQ4_1, TPR> : Geometry<kQ4_0, TPR> {};
template <int TPR>
struct Geometry<kQ5_0, TPR> : Geometry<kQ4_0, TPR> {};
template <int TPR>
struct Geometry<kQ5_1, TPR> : Geometry<kQ4_0, TPR> {};

// Q2_K / Q3_K: a step is two 2-bit planes of a half super-block, 32 bytes whose TPR threads take QB
// each: two elements a byte, 32 apart.
template <int TPR>
struct Geometry<kQ2_K, TPR> {
  static constexpr int QB = 32 / TPR;
  static constexpr int W0 = QB / 4, W1 = 2;  // dwords: quants; four scale bytes, d and dmin
};
template <int TPR>
struct Geometry<kQ3_K, TPR> {
  static constexpr int QB = 32 / TPR;
  static constexpr int W0 = QB / 4, W1 = 3 + QB / 4;  // quants; scale bytes (two dwords), d, third bits
};

// fp16(scale * (q - OFFSET)) for the four byte codes of q: the offset comes off the subnormal codes
// exactly (v_pk_add_f16), so an infinite scale stays infinite as in scale * (q - OFFSET).
template <int OFFSET>
__device__ __forceinline__ uint2 scaled4(uint32_t q, float scale24, float bias) {
  uint32_t p02 = q & 0x00FF00FFu, p13 = (q >> 8) & 0x00FF00FFu;
  if constexpr (OFFSET != 0) {
    const half2_t off = as_half2(0x80008000u | (uint32_t)OFFSET | ((uint32_t)OFFSET << 16));
    p02 = __builtin_bit_cast(uint32_t, as_half2(p02) + off);
    p13 = __builtin_bit_cast(uint32_t, as_half2(p13) + off);
  }
  return affine4(p02, p13, scale24, bias);
}

// Raw bytes of one step in vector registers (vector values stay in VGPRs; arrays of
// several sets were demoted to the stack). x: XL 16-byte activation chunks; a / b: the
// quant and header dwords of each of the thread's P weight parts.
template <int XL, int W0, int W1, int P>
struct Raw {
  typedef uint32_t XV __attribute__((ext_vector_type(4 * XL)));
  typedef uint32_t AV __attribute__((ext_vector_type(W0)));
  typedef uint32_t BV __attribute__((ext_vector_type(W1)));
  XV x;
  AV a[P];
  BV b[P];
};

}  // namespace pipe

// KS groups of WM x WN waves split K: each takes a run of steps (equal but for a unit of two or four)
// with its own LDS staging buffers; the KS partial tiles are summed in LDS at the end
// (KS = 1: the whole K range in one group).
//
// One launch covers the matrices of a GemmJob (they share x and K): blockIdx.x runs over the
// BN-wide column tiles of all of them in order.  With job.splits > 1, blockIdx.z also splits
// K across workgroups: workgroup z takes its split's range of steps and stores its fp32
// partial tile to job.partial, and gemm_reduce adds the splits in order.
//
// XT = float: fp32 activations (the packed call form), rounded to fp16 as they are loaded, so
// the staged tile is fp16(x) as in the reference's prefill numerics (benchmark.py:473-477).
template <int TYPE, int BM, int BN, int WM, int WN, int KS, typename OutT, typename XT = _Float16, bool XDMA = false>
__global__ __launch_bounds__(WM * WN * 64 * KS) void gemm_pipe(const XT* __restrict__ x, const GemmJob job,
                                                               int M, int K) {
  using namespace pipe;
  constexpr int THREADS = WM * WN * 64;  // per K group
  constexpr int MT = BM / WM / 16, NT = BN / WN / 16;
  constexpr int XL = XDMA ? 1 : BM * 8 / THREADS;  // 16-byte activation chunks per thread per step
  static_assert(!XDMA || (KS == 1 && sizeof(XT) == 2), "x by LDS DMA: fp16 x, one K group");
  constexpr int XS = BM * BK;                  // halves per DMA'd x buffer (128-byte rows, swizzled)
  constexpr int XPW = BM * BK * 2 / 1024 / (WM * WN);  // 1 KB DMA blocks per wave per step
  // TPR parts per weight row (a part: the row's step bytes one thread decodes).  Where BN
  // divides the threads, every thread takes one part of one row; otherwise (BN = 96, 192)
  // rows take 4 parts and thread t the parts t, t + THREADS, ... below BN * 4, so a wave
  // either has a part at a given index or has none (the test is wave-uniform).
  constexpr int TPR = THREADS % BN == 0 ? THREADS / BN : 4;
  constexpr int PARTS = (BN * TPR + THREADS - 1) / THREADS;
  static_assert((XDMA || XL * THREADS == BM * 8) && (TPR == 1 || TPR == 2 || TPR == 4) && PARTS <= 2 &&
                    (BN * TPR) % 64 == 0, "tile shape");
  using G = Geometry<TYPE, TPR>;
  using RawT = Raw<XL, G::W0, G::W1, PARTS>;
  constexpr int QK = Block<TYPE>::QK, BYTES = Block<TYPE>::BYTES;
  constexpr bool KQ = TYPE == kQ4_K || TYPE == kQ5_K;  // Q4_K's header and nibble layout
  constexpr bool B32 = Block<TYPE>::QK == 32;           // 32-element blocks, two per step
  constexpr bool PLANES = TYPE == kQ2_K || TYPE == kQ3_K;
  constexpr int STAGE = XDMA ? 3 * XS + 2 * BN * ROW : 2 * (BM + BN) * ROW;  // halves of one group's tiles
  __shared__ __attribute__((aligned(1024))) _Float16 stage[KS * STAGE];
  // wave-uniform (THREADS is a multiple of 64): keeps the step counter and the
  // addressing derived from it in scalar registers
  const int group = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / THREADS);
  _Float16* const xs0 = stage + group * STAGE;
  _Float16* const xs1 = xs0 + (XDMA ? XS : BM * ROW);
  _Float16* const ws0 = XDMA ? xs0 + 3 * XS : xs1 + BM * ROW;
  _Float16* const ws1 = ws0 + BN * ROW;

  // the wave index in a scalar register: the wave's tile offsets then take no vector registers
  const int tid = threadIdx.x % THREADS, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave / WN) * (16 * MT), wn = (wave % WN) * (16 * NT);
  // the matrix of this column tile (workgroup-uniform)
  const int tile = blockIdx.x;
  const int mi = tile < job.tile_end[0] ? 0 : tile < job.tile_end[1] ? 1 : 2;
  const int N = job.n[mi];
  const int m0 = blockIdx.y * BM, n0 = (tile - (mi ? job.tile_end[mi - 1] : 0)) * BN;
  int wrow[PARTS], wpart[PARTS];
  bool has[PARTS];
  // weight rows as 32-bit byte offsets from the matrix base (matrices stay under 4 GiB)
  const uint8_t* const wmat = job.w[mi];
  uint32_t wbase[PARTS];
#pragma unroll
  for (int p = 0; p < PARTS; ++p) {
    const int part = tid + p * THREADS;
    has[p] = part < BN * TPR;
    wrow[p] = has[p] ? part / TPR : 0;
    wpart[p] = part % TPR;
    wbase[p] = (uint32_t)min(n0 + wrow[p], N - 1) * (uint32_t)((K / QK) * BYTES);
  }
  // this group's steps of this split, in units of two (a super-block's four for the 256-element
  // encodings), which the first groups take one more of where they don't divide evenly; the host
  // guarantees whole units and one for every group
  constexpr int UNIT = B32 ? 2 : 4;
  const int split_steps = K / BK / job.splits, units = split_steps / UNIT, more = units % KS;
  const int steps = UNIT * (units / KS + (group < more ? 1 : 0));
  const int first = blockIdx.z * split_steps + UNIT * (group * (units / KS) + min(group, more));

  // XDMA: DMA source rows of this lane.  Block b = XPW wave + i of the x tile (1 KB, 8 rows of
  // 128 B) goes to LDS lane-linear: lane l writes 16 B at 16 l, row 8 b + l / 8, slot l % 8, which
  // holds chunk (l % 8) ^ ((row >> 1) & 7) of the row, so a 16-row fragment read hits 16 bank groups
  // as 32-bit byte offsets from the tile's first row (M * K * 2 stays under 4 GiB)
  const uint8_t* const xtile = reinterpret_cast<const uint8_t*>(x + (size_t)m0 * K);
  uint32_t xsrc[XDMA ? XPW : 1];
  if constexpr (XDMA) {
#pragma unroll
    for (int i = 0; i < XPW; ++i) {
      const int r = 8 * (XPW * wave + i) + (lane >> 3);
      const int cch = (lane & 7) ^ ((r >> 1) & 7);
      xsrc[i] = 2u * ((uint32_t)(min(m0 + r, M - 1) - m0) * (uint32_t)K + 8 * cch);
    }
  }
  auto dma = [&](int step, _Float16* xbuf) {
    if constexpr (XDMA) {
#pragma unroll
      for (int i = 0; i < XPW; ++i)
        __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(xtile + (xsrc[i] + (uint32_t)(2 * step * BK))),
                                         (void __attribute__((address_space(3)))*)(xbuf + (XPW * wave + i) * 512),
                                         16, 0, 0);
    }
  };
  auto load = [&](RawT& r, int step) {
    const int k0 = step * BK;
#pragma unroll
    for (int i = 0; i < (XDMA ? 0 : XL); ++i) {
      const int c = i * THREADS + tid, row = c >> 3, c8 = (c & 7) * 8;
      // rows past M reload row M - 1: their products land in output rows that are never stored
      const XT* src = x + (size_t)min(m0 + row, M - 1) * K + k0 + c8;
      if constexpr (sizeof(XT) == 4) {
        const uint4 lo = load16(reinterpret_cast<const uint8_t*>(src));
        const uint4 hi = load16(reinterpret_cast<const uint8_t*>(src + 4));
        r.x[4 * i] = half2_from_fp32(__builtin_bit_cast(float, lo.x), __builtin_bit_cast(float, lo.y));
        r.x[4 * i + 1] = half2_from_fp32(__builtin_bit_cast(float, lo.z), __builtin_bit_cast(float, lo.w));
        r.x[4 * i + 2] = half2_from_fp32(__builtin_bit_cast(float, hi.x), __builtin_bit_cast(float, hi.y));
        r.x[4 * i + 3] = half2_from_fp32(__builtin_bit_cast(float, hi.z), __builtin_bit_cast(float, hi.w));
      } else {
        const uint4 v = *reinterpret_cast<const uint4*>(src);
        r.x[4 * i] = v.x; r.x[4 * i + 1] = v.y; r.x[4 * i + 2] = v.z; r.x[4 * i + 3] = v.w;
      }
    }
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      if (!has[p]) continue;
      const uint8_t* blk = wmat + (wbase[p] + (uint32_t)((k0 / QK) * BYTES));
      typename RawT::AV& ra = r.a[p];
      typename RawT::BV& rb = r.b[p];
      if constexpr (B32) {
        constexpr int QPB = G::QPB, QB = G::QB;
        const uint8_t* b = blk + (QB * wpart[p] / QPB) * BYTES;  // this part's block: fp16 d, quants
        constexpr int HEAD = TYPE == kQ5_1 ? 8 : TYPE == kQ5_0 ? 6 : TYPE == kQ4_1 ? 4 : 2;
        const uint8_t* q = b + HEAD + QB * wpart[p] % QPB;
        if constexpr (G::W0 % 4 == 0) {
#pragma unroll
          for (int i = 0; i < G::W0; i += 4) {
            const uint4 v = load16(q + 4 * i);
            ra[i] = v.x; ra[i + 1] = v.y; ra[i + 2] = v.z; ra[i + 3] = v.w;
          }
        } else {
          const uint2 v = load8(q);
          ra[0] = v.x; ra[1] = v.y;
        }
        rb[0] = load4(b);
        rb[1] = TYPE == kQ5_0 || TYPE == kQ5_1 ? load4(b + HEAD - 4) : 0;
      } else if constexpr (PLANES) {
        const int half = (step & 3) >> 1, l0 = G::QB * wpart[p];
        const uint8_t* q = blk + (TYPE == kQ2_K ? 16 : 32) + 32 * half + l0;
#pragma unroll
        for (int i = 0; i < G::W0; ++i) ra[i] = load4(q + 4 * i);
        if constexpr (TYPE == kQ2_K) {
          rb[0] = load4(blk + 4 * (step & 3));
          rb[1] = load4(blk + 80);
        } else {
          rb[0] = load4(blk + 96 + 4 * (step & 1));
          rb[1] = load4(blk + 104);
          rb[2] = load4(blk + 106);  // high half: d
#pragma unroll
          for (int i = 0; i < G::W0; ++i) rb[3 + i] = load4(blk + l0 + 4 * i);
        }
      } else if constexpr (KQ) {
        const uint4 hd = load16(blk);
        rb[0] = hd.x; rb[1] = hd.y; rb[2] = hd.z; rb[3] = hd.w;
        const uint8_t* q = blk + (TYPE == kQ5_K ? 48 : 16) + 32 * (step & 3) + G::QB * wpart[p];
#pragma unroll
        for (int i = 0; i < G::W0; ++i) ra[i] = load4(q + 4 * i);
        if constexpr (TYPE == kQ5_K) {
#pragma unroll
          for (int i = 0; i < G::W0; ++i) rb[4 + i] = load4(blk + 16 + G::QB * wpart[p] + 4 * i);
        }
      } else {
        const int h = (step & 3) >> 1, e0 = G::EPT * wpart[p];  // element offset inside the step
        const int quarter = 2 * (step & 1) + (e0 >> 5), l0 = e0 & 31;
        const uint8_t* ql = blk + 64 * h + e0;
        const uint8_t* qh = blk + 128 + 32 * h + l0;
#pragma unroll
        for (int i = 0; i < G::W0; ++i) {
          ra[i] = load4(ql + 4 * i);
          rb[i] = load4(qh + 4 * i);
        }
        rb[G::W0] = load4(blk + 192 + 8 * h + 2 * quarter);  // scales 2q .. 2q+3 of this half
        rb[G::W0 + 1] = load4(blk + 206);                    // high half: d
      }
    }
  };

  auto store = [&](const RawT& r, _Float16* xs, _Float16* ws, int step) {
#pragma unroll
    for (int i = 0; i < (XDMA ? 0 : XL); ++i) {
      const int c = i * THREADS + tid, row = c >> 3, c8 = (c & 7) * 8;
      *reinterpret_cast<uint4*>(&xs[row * ROW + c8]) = make_uint4(r.x[4 * i], r.x[4 * i + 1], r.x[4 * i + 2], r.x[4 * i + 3]);
    }
#pragma unroll
    for (int p = 0; p < PARTS; ++p) {
      if (!has[p]) continue;
      const typename RawT::AV& ra = r.a[p];
      const typename RawT::BV& rb = r.b[p];
      if constexpr (B32) {
        constexpr int QPB = G::QPB, QB = G::QB;
        const float d = half_bits_to_float(rb[0]);
        // element e of block b (32 b + e in the step) sits at ws[wrow[p]][32 b + e]
        _Float16* dst = &ws[wrow[p] * ROW + 32 * (QB * wpart[p] / QPB) + QB * wpart[p] % QPB];
        if constexpr (TYPE == kQ8_0) {
          // d * q for the int8 code q, as the fp16 subnormal code q + 128 (byte ^ 0x80) times
          // d 2^24 plus -128 d: the product and the sum (q d) are exact, so is the fp32 value
          const float d24 = d * kTwo24, bias = -128.0f * d;
#pragma unroll
          for (int i = 0; i < G::W0; ++i) {
            const uint32_t u = ra[i] ^ 0x80808080u;
            *reinterpret_cast<uint2*>(dst + 4 * i) = affine4(u & 0x00FF00FFu, (u >> 8) & 0x00FF00FFu, d24, bias);
          }
        } else if constexpr (TYPE == kQ4_1 || TYPE == kQ5_0 || TYPE == kQ5_1) {
          // q * d + m, or (q - 16) * d; bit j of the fifth bits is element j's, bit j + 16 the high nibble's
          constexpr int OFFSET = TYPE == kQ5_0 ? 16 : 0;
          const float d24 = d * kTwo24, m = TYPE == kQ5_0 ? 0.0f : half_bits_to_float(rb[0] >> 16);
          const int j0 = QB * wpart[p] % QPB;
#pragma unroll
          for (int i = 0; i < G::W0; ++i) {
            uint32_t lo = ra[i] & 0x0F0F0F0Fu, hi = (ra[i] >> 4) & 0x0F0F0F0Fu;
            if constexpr (TYPE != kQ4_1) {
              const uint32_t fifth = rb[1] >> (j0 + 4 * i);
              lo |= fifth_bits(fifth);
              hi |= fifth_bits(fifth >> 16);
            }
            *reinterpret_cast<uint2*>(dst + 4 * i) = scaled4<OFFSET>(lo, d24, m);
            *reinterpret_cast<uint2*>(dst + 16 + 4 * i) = scaled4<OFFSET>(hi, d24, m);
          }
        } else {
          // (q - 8) * d: byte j's low nibble is element j, its high nibble element j + 16 (left in
          // bits 4-7 of its half, 16 q * 2^-24, against d 2^20)
          const float d24 = d * kTwo24, d20 = d * kTwo20, bias = -8.0f * d;
#pragma unroll
          for (int i = 0; i < G::W0; ++i) {
            const uint32_t q = ra[i], q8 = q >> 8;
            *reinterpret_cast<uint2*>(dst + 4 * i) = affine4(q & 0x000F000Fu, q8 & 0x000F000Fu, d24, bias);
            *reinterpret_cast<uint2*>(dst + 16 + 4 * i) = affine4(q & 0x00F000F0u, q8 & 0x00F000F0u, d20, bias);
          }
        }
      } else if constexpr (PLANES) {
        // planes 2 (step % 2) and the next: byte l holds element l of both; their 16-element scales are
        // bytes run and run + 2 of the step's four, run = l / 16
        const int l0 = G::QB * wpart[p], run = l0 >> 4;
        _Float16* dst = &ws[wrow[p] * ROW + l0];
        if constexpr (TYPE == kQ2_K) {
          const uint32_t sa = rb[0] >> (8 * run), sb = sa >> 16;
          const float d = half_bits_to_float(rb[1]), dmin = half_bits_to_float(rb[1] >> 16);
          // the upper plane stays two bits up in its byte: its scale takes 2^22
          const float da = d * (float)(sa & 15u) * kTwo24, db = d * (float)(sb & 15u) * (kTwo24 / 4);
          const float ma = -(dmin * (float)((sa >> 4) & 15u)), mb = -(dmin * (float)((sb >> 4) & 15u));
#pragma unroll
          for (int i = 0; i < G::W0; ++i) {
            const uint32_t q = ra[i] >> (4 * (step & 1));
            *reinterpret_cast<uint2*>(dst + 4 * i) = affine4(q & 0x00030003u, (q >> 8) & 0x00030003u, da, ma);
            *reinterpret_cast<uint2*>(dst + 32 + 4 * i) = affine4(q & 0x000C000Cu, (q >> 8) & 0x000C000Cu, db, mb);
          }
        } else {
          const int half = (step & 3) >> 1;
          const uint32_t codes = ((rb[0] >> (4 * half)) & 0x0F0F0F0Fu) | (((rb[1] >> (2 * (step & 3))) & 0x03030303u) << 4);
          const uint32_t sa = codes >> (8 * run), sb = sa >> 16;
          const float d = half_bits_to_float(rb[2] >> 16);
          const float da = d * (float)((int)(sa & 63u) - 32) * kTwo24, db = d * (float)((int)(sb & 63u) - 32) * kTwo24;
#pragma unroll
          for (int i = 0; i < G::W0; ++i) {
            const uint32_t q = ra[i] >> (4 * (step & 1)), h = rb[3 + i] >> (2 * (step & 3));
            *reinterpret_cast<uint2*>(dst + 4 * i) = scaled4<4>((q & 0x03030303u) | ((h & 0x01010101u) << 2), da, 0.0f);
            *reinterpret_cast<uint2*>(dst + 32 + 4 * i) =
                scaled4<4>(((q >> 2) & 0x03030303u) | ((h << 1) & 0x04040404u), db, 0.0f);
          }
        }
      } else if constexpr (KQ) {
        // d*sc*q - dmin*m: the product is exact, the subtraction rounds once; high nibbles stay in
        // bits 4-7 of their halves (16 q * 2^-24), so their scale takes 2^20
        float ds_lo, dm_lo, ds_hi, dm_hi;
        if constexpr (TPR == 4) {
          // the four lanes of a row (a DPP quad) each decode one of the step's four factors,
          // lane f: f & 2 picks sub-block 2j + 1, f & 1 the min, and share them by broadcasts
          const int f = lane & 3, jj = step & 3, t8 = 16 * (jj & 1) + 8 * (f >> 1);
          // the scale bytes (rb[1]) or the min bytes (rb[2]) by one byte permute
          const uint32_t word = __builtin_amdgcn_perm(rb[2], rb[1], f & 1 ? 0x07060504u : 0x03020100u);
          const uint32_t low6 = __builtin_amdgcn_ubfe(word, t8, 6);  // sub-blocks 0-3
          const uint32_t split = __builtin_amdgcn_ubfe(rb[3], t8 + 4 * (f & 1), 4) |
                                 (__builtin_amdgcn_ubfe(word, t8 + 6, 2) << 4);
          const uint32_t code = jj < 2 ? low6 : split;
          const float lane_scale = f & 1 ? -1.0f : (f & 2 ? kTwo20 : kTwo24);
          const float v = half_bits_to_float(rb[0] >> (16 * (f & 1))) * lane_scale * (float)code;
          const int vi = __builtin_bit_cast(int, v);
          ds_lo = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(vi, 0x00, 0xF, 0xF, false));
          dm_lo = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(vi, 0x55, 0xF, 0xF, false));
          ds_hi = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(vi, 0xAA, 0xF, 0xF, false));
          dm_hi = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(vi, 0xFF, 0xF, 0xF, false));
        } else if constexpr (TPR == 2) {
          // the two lanes of a row each decode the scale and min of one sub-block (lane f: 2j + f)
          // and take the other lane's by pair broadcasts within the DPP quad
          const int f = lane & 1, jj = step & 3, t8 = 16 * (jj & 1) + 8 * f;
          const uint32_t sc = jj < 2 ? __builtin_amdgcn_ubfe(rb[1], t8, 6)
                                     : __builtin_amdgcn_ubfe(rb[3], t8, 4) | (__builtin_amdgcn_ubfe(rb[1], t8 + 6, 2) << 4);
          const uint32_t mn = jj < 2 ? __builtin_amdgcn_ubfe(rb[2], t8, 6)
                                     : __builtin_amdgcn_ubfe(rb[3], t8 + 4, 4) | (__builtin_amdgcn_ubfe(rb[2], t8 + 6, 2) << 4);
          const float d = half_bits_to_float(rb[0]), dmin = half_bits_to_float(rb[0] >> 16);
          const int ds = __builtin_bit_cast(int, d * (f ? kTwo20 : kTwo24) * (float)sc);
          const int dm = __builtin_bit_cast(int, -(dmin * (float)mn));
          ds_lo = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(ds, 0xA0, 0xF, 0xF, false));  // lanes 0, 2
          dm_lo = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(dm, 0xA0, 0xF, 0xF, false));
          ds_hi = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(ds, 0xF5, 0xF, 0xF, false));  // lanes 1, 3
          dm_hi = __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(dm, 0xF5, 0xF, 0xF, false));
        } else {
          int sc_lo, mn_lo, sc_hi, mn_hi;
          q4k_scale_pair(rb[1], rb[2], rb[3], step & 3, sc_lo, mn_lo, sc_hi, mn_hi);
          const float d = half_bits_to_float(rb[0]), dmin = half_bits_to_float(rb[0] >> 16);
          ds_lo = d * (float)sc_lo * kTwo24;
          dm_lo = -(dmin * (float)mn_lo);
          ds_hi = d * (float)sc_hi * kTwo20;
          dm_hi = -(dmin * (float)mn_hi);
        }
        _Float16* dst = &ws[wrow[p] * ROW + G::QB * wpart[p]];
#pragma unroll
        for (int i = 0; i < G::W0; ++i) {
          const uint32_t q = ra[i];  // low nibbles: sub-block 2j, high nibbles: 2j+1
          const uint32_t q8 = q >> 8;
          uint32_t lo02 = q & 0x000F000Fu, lo13 = q8 & 0x000F000Fu;
          uint32_t hi02 = q & 0x00F000F0u, hi13 = q8 & 0x00F000F0u;
          if constexpr (TYPE == kQ5_K) {
            // fifth bits: bit 2j (sub-block 2j) and 2j+1 of the qh byte at the quant byte's position
            const uint32_t h = rb[4 + i] >> (2 * (step & 3));
            lo02 |= (h & 0x00010001u) << 4;
            lo13 |= ((h >> 8) & 0x00010001u) << 4;
            hi02 |= ((h >> 1) & 0x00010001u) << 8;
            hi13 |= ((h >> 9) & 0x00010001u) << 8;
          }
          *reinterpret_cast<uint2*>(dst + 4 * i) = affine4(lo02, lo13, ds_lo, dm_lo);
          *reinterpret_cast<uint2*>(dst + 32 + 4 * i) = affine4(hi02, hi13, ds_hi, dm_hi);
        }
      } else {
        const int e0 = G::EPT * wpart[p];
        const int quarter = 2 * (step & 1) + (e0 >> 5), l0 = e0 & 31;
        const float d = half_bits_to_float(rb[G::W0 + 1] >> 16);
        _Float16* dst = &ws[wrow[p] * ROW + e0];
#pragma unroll
        for (int i = 0; i < G::W0; ++i) {
          // 6-bit codes of elements l0 + 4i .. + 3 of this quarter
          const uint32_t lo = (ra[i] >> (4 * (step & 1))) & 0x0F0F0F0Fu;
          const uint32_t hi = ((rb[i] >> (2 * quarter)) & 0x03030303u) << 4;
          const uint32_t q = lo | hi;
          // scale index 8h + 2 quarter + l / 16: byte l / 16 of the dword loaded at 2 quarter
          const float sc = (float)(int8_t)(rb[G::W0] >> (8 * ((l0 + 4 * i) >> 4)));
          // (q - 32) * sc * d == q * (sc d) - 32 (sc d): exact, one fused rounding
          const float scd = sc * d;
          *reinterpret_cast<uint2*>(dst + 4 * i) =
              affine4(q & 0x003F003Fu, (q >> 8) & 0x003F003Fu, scd * kTwo24, -32.0f * scd);
        }
      }
    }
  };

  float4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};

  // fragments of one 32-wide half kk of the step staged in (xs, ws)
  auto fragments = [&](half8_t (&a)[MT], half8_t (&b)[NT], const _Float16* xs, const _Float16* ws, int kk) {
    const int koff = 32 * kk + 8 * (lane >> 4);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int row = wm + 16 * i + (lane & 15);
      if constexpr (XDMA)
        a[i] = *reinterpret_cast<const half8_t*>(&xs[row * BK + 8 * ((4 * kk + (lane >> 4)) ^ ((row >> 1) & 7))]);
      else
        a[i] = *reinterpret_cast<const half8_t*>(&xs[row * ROW + koff]);
    }
#pragma unroll
    for (int j = 0; j < NT; ++j)
      b[j] = *reinterpret_cast<const half8_t*>(&ws[(wn + 16 * j + (lane & 15)) * ROW + koff]);
  };
  auto multiply = [&](const half8_t (&a)[MT], const half8_t (&b)[NT]) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int j = 0; j < NT; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b[j], acc[i][j], 0, 0, 0);
  };
  // XDMA: the fragments of the last step's second half, multiplied first in the next: the matrix
  // pipe has work while that step's fragments come from LDS (without it and with x through registers,
  // a 256 x 128 step took 2700 cycles for 1024 of MFMA work).  M = 2048: Q6_K 4096 x 12288
  // 274 -> 251 us, Q8_0 269 -> 219, Q4_K 4096 x 4096 80 -> 77, Q5_K 99 -> 81, Q3_K 143 -> 88; the
  // 256 x 192 tile 395 -> 389 (Q4_K 24576 x 4096).  Weights two steps ahead measured no faster.
  half8_t a1[MT], b1[NT];
  if constexpr (XDMA) {
#pragma unroll
    for (int i = 0; i < MT; ++i) a1[i] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < NT; ++j) b1[j] = half8_t{0, 0, 0, 0, 0, 0, 0, 0};
  }

  // one K step: fragment reads of (xs, ws), then MFMAs interleaved with the
  // staging of `staged` into (xn, wnext) and the prefetch of `fetch_step`
  auto step_body = [&](const _Float16* xs, const _Float16* ws, _Float16* xn, _Float16* wnext, const RawT& staged,
                       int staged_step, RawT& fetched, int fetch_step, _Float16* xdma = nullptr) {
    half8_t a[2][MT], b[2][NT];
    fragments(a[0], b[0], xs, ws, 0);
    if constexpr (XDMA) {
      // the x DMA of the fetched step is issued ahead of its weight loads and the order is pinned:
      // loads complete in order, so once a wave's dequant has waited on those weights (the next
      // step's store), its DMA'd x has landed too, before the barrier that follows.
      // Ping-pong: the upper half of the waves issue their MFMAs before they dequantize, the lower
      // half (in the 256 x 192 tile those with two weight parts, everywhere else each wave has one) after, so
      // the two waves that share a SIMD keep its matrix pipe and its VALU busy at the same time.
      auto mfma_all = [&]() {
        multiply(a1, b1);
        __builtin_amdgcn_sched_barrier(0);
        fragments(a1, b1, xs, ws, 1);
        multiply(a[0], b[0]);
      };
      const bool mfma_first = wave >= WM * WN / 2;
      if (mfma_first) {
        mfma_all();
        __builtin_amdgcn_sched_barrier(0);
      }
      store(staged, xn, wnext, staged_step);
      dma(fetch_step, xdma);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      load(fetched, fetch_step);
      if (!mfma_first) {
        __builtin_amdgcn_sched_barrier(0);
        mfma_all();
      }
      return;
    }
    fragments(a[1], b[1], xs, ws, 1);
    store(staged, xn, wnext, staged_step);
    load(fetched, fetch_step);
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[kk][i], b[kk][j], acc[i][j], 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 2 * MT * NT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one MFMA
      __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // two VALU
      if (i % 4 == 0) __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // an LDS store
      if (i % 4 == 2) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // a global load
    }
  };

  // two register sets of raw bytes: step s+1 is staged into LDS while step s+2 is fetched
  RawT ra, rb;
  const int last = first + steps - 1;
  if constexpr (XDMA) {
    // three x buffers: step s reads buffer s % 3 while the DMA of step s + 2 fills (s + 2) % 3;
    // the barrier between steps orders LDS only (this wave's DMA'd x of the next step has landed
    // by then), so the weight loads in flight stay in flight
    dma(first, xs0);
    asm volatile("" ::: "memory");
    dma(first + 1, xs1);
    asm volatile("" ::: "memory");
    load(ra, first);
    load(rb, first + 1);
    store(ra, xs0, ws0, first);
    __builtin_amdgcn_s_waitcnt(0);  // the first two x tiles have landed (every counter)
    __syncthreads();
    int cur = 0;
    for (int step = first; step < first + steps; step += 2) {
      const int c1 = cur == 2 ? 0 : cur + 1, c2 = c1 == 2 ? 0 : c1 + 1;
      step_body(xs0 + cur * XS, ws0, nullptr, ws1, rb, step + 1, ra, min(step + 2, last), xs0 + c2 * XS);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      const int c3 = c2 == 2 ? 0 : c2 + 1;
      step_body(xs0 + c1 * XS, ws1, nullptr, ws0, ra, min(step + 2, last), rb, min(step + 3, last), xs0 + c3 * XS);
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      cur = c2;
    }
    multiply(a1, b1);
  } else {
    load(ra, first);
    load(rb, first + 1);
    store(ra, xs0, ws0, first);
    __syncthreads();
    for (int step = first; step < first + steps; step += 2) {
      // the last step stages and fetches clamped copies that are never read
      step_body(xs0, ws0, xs1, ws1, rb, step + 1, ra, min(step + 2, last));
      __syncthreads();
      step_body(xs1, ws1, xs0, ws0, ra, min(step + 2, last), rb, min(step + 3, last));
      __syncthreads();
    }
    if constexpr (KS > 1) {
      // the barriers of the groups that took a unit more
      if (more > 0 && group >= more)
        for (int i = 0; i < UNIT; ++i) __syncthreads();
    }
  }
  if constexpr (KS > 1) {
    // partial tiles of groups 1 .. KS-1 -> LDS (over the staging buffers), summed by group 0
    float* red = reinterpret_cast<float*>(stage);
    static_assert((KS - 1) * MT * NT * 4 * THREADS * 4 <= KS * STAGE * 2, "reduction buffer");
    if (group > 0) {
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) red[(((group - 1) * MT + i) * NT + j) * 4 * THREADS + e * THREADS + tid] = acc[i][j][e];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < KS; ++g)
#pragma unroll
      for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] += red[(((g - 1) * MT + i) * NT + j) * 4 * THREADS + e * THREADS + tid];
  }
  const bool split = job.splits > 1;
  OutT* const out = static_cast<OutT*>(job.out[mi]);
  float* const part = split ? job.partial + (size_t)blockIdx.z * M * job.n_total + job.col0[mi] : nullptr;
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) {
      const int col = n0 + wn + 16 * j + (lane & 15);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = m0 + wm + 16 * i + 4 * (lane >> 4) + e;
        if (row < M && col < N) {
          if (split) part[(size_t)row * job.n_total + col] = acc[i][j][e];
          else store_out<OutT>(out, (size_t)row * N + col, acc[i][j][e]);
        }
      }
    }
}

// out_i[row, c] = the sum of the splits' partial sums, added in split order (so the result does
// not depend on which workgroup finished first), converted once to the output type.
// A thread takes four consecutive columns of one row (blockIdx.y strides over the rows): one
// 16-byte load per split when the row width is a multiple of 4 (every row then starts
// 16-byte aligned in each split's plane), and one 4-wide store when the four columns fall in
// one matrix at a 4-aligned offset.
template <typename OutT>
__global__ __launch_bounds__(256) void gemm_reduce(const GemmJob job, int M) {
  const int n = job.n_total;
  const size_t plane = (size_t)M * n;
  const int c = 4 * (blockIdx.x * 256 + threadIdx.x);
  if (c >= n) return;
  const bool wide = (n & 3) == 0;
  for (int row = blockIdx.y; row < M; row += gridDim.y) {
    const float* p = job.partial + (size_t)row * n + c;
    float s[4];
    if (wide) {
      float4 v = *reinterpret_cast<const float4*>(p);
      for (int z = 1; z < job.splits; ++z) {
        const float4 u = *reinterpret_cast<const float4*>(p + z * plane);
        v.x += u.x; v.y += u.y; v.z += u.z; v.w += u.w;
      }
      s[0] = v.x; s[1] = v.y; s[2] = v.z; s[3] = v.w;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = 0.f;
        if (c + i < n) {
          s[i] = p[i];
          for (int z = 1; z < job.splits; ++z) s[i] += p[z * plane + i];
        }
      }
    }
    const int mi = job.count > 1 && c >= job.col0[1] ? (job.count > 2 && c >= job.col0[2] ? 2 : 1) : 0;
    const int local = c - job.col0[mi];
    OutT* out = static_cast<OutT*>(job.out[mi]) + (size_t)row * job.n[mi];
    if (wide && local + 4 <= job.n[mi] && ((job.n[mi] | local) & 3) == 0) {
      if constexpr (sizeof(OutT) == 2) {
        *reinterpret_cast<uint2*>(out + local) = make_uint2(half2_from_fp32(s[0], s[1]), half2_from_fp32(s[2], s[3]));
      } else {
        *reinterpret_cast<float4*>(out + local) = make_float4(s[0], s[1], s[2], s[3]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int col = c + i;
        if (col >= n) break;
        const int m = job.count > 1 && col >= job.col0[1] ? (job.count > 2 && col >= job.col0[2] ? 2 : 1) : 0;
        store_out<OutT>(static_cast<OutT*>(job.out[m]), (size_t)row * job.n[m] + (col - job.col0[m]), s[i]);
      }
    }
  }
}

namespace {

// Workgroup tiles of the pipelined GEMM, by index: 0..3 without a K split inside the workgroup,
// 4..7 with two or four wave groups per workgroup (LDS holds one double-buffered stage per
// group, so 128 x 128 and 128 x 64 take KS <= 2 and 64 x 64 KS <= 4), 8 the 256 x 96 tile (8
// waves of 64 x 48), 9 the 256 x 192 tile (8 waves of 64 x 96, x by LDS DMA).
struct Tile {
  int bm, bn, ks;
};
constexpr int kTileCount = 10;
constexpr Tile kTiles[kTileCount] = {{256, 128, 1}, {128, 128, 1}, {128, 64, 1}, {64, 64, 1}, {128, 128, 2},
                                     {128, 64, 2},  {64, 64, 2},   {64, 64, 4},  {256, 96, 1}, {256, 192, 1}};
constexpr int kDmaTile = 9;  // x tile by LDS DMA: fp16 x only

// The 256 x 192 tile's 8 waves of 64 x 96 fit the register file only without the activation
// staging registers (x by LDS DMA); with Q5_K's fifth bits or Q6_K's layout they still spill.
template <int TYPE, typename XT>
constexpr bool dma_tile_type() {
  return sizeof(XT) == 2 && (TYPE == kQ4_K || TYPE == kQ8_0 || TYPE == kQ4_0);
}

long tile_count(const GemmGroupArgs& a, const Tile& t) {
  long columns = 0;
  for (int i = 0; i < a.count; ++i) columns += (a.n[i] + t.bn - 1) / t.bn;
  return (long)((a.m + t.bm - 1) / t.bm) * columns;
}

int total_columns(const GemmGroupArgs& a) {
  int n = 0;
  for (int i = 0; i < a.count; ++i) n += a.n[i];
  return n;
}

// The job of one launch: per-matrix column tiles and partial-sum columns.
GemmJob make_job(const GemmGroupArgs& a, const Tile& t, int splits, void* workspace) {
  GemmJob job{};
  int tiles = 0, col = 0;
  for (int i = 0; i < kGemmGroupMax; ++i) {
    if (i < a.count) {
      job.w[i] = static_cast<const uint8_t*>(a.w[i]);
      job.out[i] = a.out[i];
      job.n[i] = a.n[i];
      tiles += (a.n[i] + t.bn - 1) / t.bn;
      job.col0[i] = col;
      col += a.n[i];
    } else {
      job.col0[i] = col;  // past the last matrix: never selected
    }
    job.tile_end[i] = tiles;
  }
  job.count = a.count;
  job.n_total = col;
  job.splits = splits;
  job.partial = static_cast<float*>(workspace);
  return job;
}

template <int TYPE, int BM, int BN, int WM, int WN, int KS, typename OutT, typename XT, bool XDMA = false>
hipError_t launch_pipe(const GemmGroupArgs& a, int splits, void* workspace, hipStream_t stream) {
  const GemmJob job = make_job(a, Tile{BM, BN, KS}, splits, workspace);
  const dim3 grid(job.tile_end[kGemmGroupMax - 1], (a.m + BM - 1) / BM, splits), block(WM * WN * 64 * KS);
  hipLaunchKernelGGL((gemm_pipe<TYPE, BM, BN, WM, WN, KS, OutT, XT, XDMA>), grid, block, 0, stream,
                     static_cast<const XT*>(a.x), job, a.m, a.k);
  if (splits > 1) {
    // four columns per thread across x; rows over y (strided past 65535 rows)
    const unsigned cols = (unsigned)((job.n_total + 1023) / 1024), rows = (unsigned)std::min(a.m, 65535);
    hipLaunchKernelGGL((gemm_reduce<OutT>), dim3(cols, rows), dim3(256), 0, stream, job, a.m);
  }
  return hipGetLastError();
}

template <int TYPE, typename OutT, typename XT>
hipError_t launch_tile(const GemmGroupArgs& a, int tile, int splits, void* workspace, hipStream_t stream) {
  switch (tile) {
    case 0: return launch_pipe<TYPE, 256, 128, 4, 2, 1, OutT, XT, sizeof(XT) == 2>(a, splits, workspace, stream);
    case 1: return launch_pipe<TYPE, 128, 128, 2, 2, 1, OutT, XT>(a, splits, workspace, stream);
    case 2: return launch_pipe<TYPE, 128, 64, 2, 2, 1, OutT, XT>(a, splits, workspace, stream);
    case 3: return launch_pipe<TYPE, 64, 64, 1, 2, 1, OutT, XT>(a, splits, workspace, stream);
    case 4: return launch_pipe<TYPE, 128, 128, 2, 2, 2, OutT, XT>(a, splits, workspace, stream);
    case 5: return launch_pipe<TYPE, 128, 64, 2, 2, 2, OutT, XT>(a, splits, workspace, stream);
    case 6: return launch_pipe<TYPE, 64, 64, 1, 2, 2, OutT, XT>(a, splits, workspace, stream);
    case 7: return launch_pipe<TYPE, 64, 64, 1, 2, 4, OutT, XT>(a, splits, workspace, stream);
    case 8: return launch_pipe<TYPE, 256, 96, 4, 2, 1, OutT, XT>(a, splits, workspace, stream);
    case kDmaTile:
      if constexpr (dma_tile_type<TYPE, XT>())
        return launch_pipe<TYPE, 256, 192, 4, 2, 1, OutT, XT, true>(a, splits, workspace, stream);
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

template <int TYPE>
hipError_t launch_typed(const GemmGroupArgs& a, int tile, int splits, void* workspace, hipStream_t stream) {
  if (a.x_f32)
    return a.out_half ? launch_tile<TYPE, _Float16, float>(a, tile, splits, workspace, stream)
                      : launch_tile<TYPE, float, float>(a, tile, splits, workspace, stream);
  return a.out_half ? launch_tile<TYPE, _Float16, _Float16>(a, tile, splits, workspace, stream)
                    : launch_tile<TYPE, float, _Float16>(a, tile, splits, workspace, stream);
}


}  // namespace
}  // namespace tensor_gguf
