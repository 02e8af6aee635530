// Decode GEMV on matrix cores, every encoding, any K the encoding allows, 1 <= M <= 8 rows of
// fp16 activations: out[m, n] = sum_k x[m, k] * W[n, k], up to three matrices that share x in
// one launch, or a gate / up pair with the SwiGLU epilogue.
//
// Each lane owns whole pieces of one weight row (a unit of 64 elements: two 32-element
// blocks, or a quarter super-block), so that a piece's scale is a value of the lane's
// own and is applied once per 16 or 32 elements in fp32.  v_mfma_f32_16x16x32_f16 does the
// products all the same: its B operand takes 8 codes from every lane (lane n + 16 g: row n of a
// 16-row tile, piece g of four that follow each other), and its A operand holds the activations
// block-diagonally, row 4 g + m being x[m] over piece g and zero over the other three.  Result
// rows 4 g .. 4 g + 3 are then the four activation rows' sums over piece g alone, and they lie in
// just the lanes that own piece g.  Three quarters of the multiplies are by zero, which a decode
// GEMV can afford: at M <= 4 a SIMD spends 16 of its cycles per 512 weights on them, against the
// ~60 of the decode (M > 4 takes a second MFMA for rows 4..7), while a vector dot product
// would spend M / 2 instructions per weight pair and read M activations per weight from LDS.
//
// Codes enter the MFMA as fp16 code * 2^-9 (v_perm_b32 widens bytes with a zero high byte, one packed
// multiply, or a fma that subtracts a constant offset exactly, makes the subnormal normal), so
// nothing is biased and cancelled.  Minimums multiply the sums of x over their
// 16 or 32 elements, which come from an MFMA of the same activations with ones.
//
// A workgroup owns one or a few 16-row tiles and splits K over its waves; a wave fetches 16 rows x 256
// columns at a time in 16-byte pieces along the rows (lane-owned pieces read straight from memory
// touch a cache line per lane and stop at 2 TB/s), passes them to their owning lanes through an LDS
// area of its own, and requests the next ones before it multiplies.  The activations are staged
// in LDS in slices (all of K where it fits), padded with zeros to whole steps; the first are requested
// ahead of the first weights and waited for behind them.  Partial sums meet in LDS in range order.
//
// What bounds it: the stream at large shapes (Q8_0 12288 x 4096 at M = 4: 13.1 us, 4.1 TB/s;
// 22.9 on the vector kernel), below ~8 MB the chain from launch to store (x, weights, LDS, MFMAs,
// partial sums; ~2.5 us over an empty launch).  Instructions count there: integer divisions, branchy
// bounds checks and unrolled variants of this kernel that ran each instruction once cost up to 3 us
// in fetching them.  Microseconds per launch (graph replays, weights rotated), vector kernels ->
// here: Q6_K 4096 x 12288 22.3 -> 13.5 (M = 4), 64.0 -> 17.9 (M = 8); Q4_0 12288 x 4096 55.2 -> 11.3
// (M = 8); Q5_0 6912 x 2560 10.2 -> 6.8 (M = 2); Q3_K 2560 x 6912 10.4 -> 7.4 (M = 1); Q5_K SwiGLU
// pair 2 x 6912 x 2560 33.4 -> 9.0 (M = 1), 90.6 -> 11.3 (M = 8).  Measured and not kept: two
// row tiles per wave (spills), shares of the steps that cross tiles (code size), lanes
// without activations masked off instead of reading zeros (1-3% slower).
#include <algorithm>

#include "gguf_decode.h"
#include "gguf_rows.h"
#include "gguf_rows_plan.h"

namespace tensor_gguf {
namespace {

// What a group (SwiGLU: the up matrix) reads besides the leading arguments, which arrive in registers: a
// single matrix waits for no load of the argument block.  Nor does the kernel ask for its block size,
// which would add 256 bytes of hidden arguments to each launch: a pass of 28 launches on new buffers behind other
// work was submitted in 245 us with them (8.3 us a call), 180 us without (4.6).
struct RowsMore {
  const uint8_t* w[kGemvGroupMax - 1];  // matrices 1 and 2 (SwiGLU: up)
  void* out[kGemvGroupMax - 1];
  int n[kGemvGroupMax - 1];
  int first_block[kGemvGroupMax - 1];   // first workgroup of matrices 1 and 2
};
enum { kRowsHalf = 1, kRowsSwiglu = 2, kRowsGroup = 4 };  // flags

// The sum of v over lanes n, n + 16, n + 32 and n + 48, in each of them: the row swaps of v with
// itself leave rows {0, 0, 2, 2} and {1, 1, 3, 3}, then rows {0, 0} and {2, 2} of the pair sums.
__device__ __forceinline__ float sum_pieces(float v) {
  uint32_t b = __builtin_bit_cast(uint32_t, v);
  const auto rows = __builtin_amdgcn_permlane16_swap(b, b, false, false);
  const uint32_t r0 = rows[0], r1 = rows[1];
  b = __builtin_bit_cast(uint32_t, __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1));
  const auto halves = __builtin_amdgcn_permlane32_swap(b, b, false, false);
  const uint32_t h0 = halves[0], h1 = halves[1];
  return __builtin_bit_cast(float, h0) + __builtin_bit_cast(float, h1);
}

__device__ __forceinline__ bool is_finite(float v) {
  return (__builtin_bit_cast(uint32_t, v) & 0x7F800000u) != 0x7F800000u;
}

// A sum that is not finite: an infinity in x makes scale * (codes . x) + low * sum(x) infinity minus
// infinity, and one in a scale multiplies a sum of either sign, where x . W is defined by each
// element's product.  The encodings without a vector kernel that sums scale by scale (gemv_blocks
// multiplies elements) take such outputs again, element by element, a wave to an output: one
// infinite row of eight at 12288 x 4096 Q5_K 12.5 -> 109 us; the test of each sum costs finite calls 0 to 2%.
template <int TYPE>
constexpr bool by_element() {
  return TYPE == kQ4_1 || TYPE == kQ5_0 || TYPE == kQ5_1 || TYPE == kQ2_K || TYPE == kQ3_K || TYPE == kQ5_K;
}

// x . (one row of W) over the wave, in every lane.
template <int TYPE>
__device__ __forceinline__ float element_product(const uint8_t* __restrict__ row, const _Float16* __restrict__ x, int k, int lane) {
  float sum = 0.0f;
#pragma unroll 1
  for (int e = 8 * lane; e < k; e += 512) {
    float v[8];
    decode8<TYPE>(row + (size_t)(e / Block<TYPE>::QK) * Block<TYPE>::BYTES, e % Block<TYPE>::QK, v);
    const half8_t xv = *reinterpret_cast<const half8_t*>(x + e);
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = fmaf(v[i], (float)xv[i], sum);
  }
  return wave_sum(sum);
}

constexpr int kRowsZero = 256;  // bytes of zeros in LDS that inactive lanes read

// MR: activation rows a lane keeps sums of (1, 4 or 8).  The workgroup's waves are `per` row tiles
// times `split` ranges of K: wave t * split + q takes steps q, q + split, .. of tile t.
template <int TYPE, int MR>
__global__ __launch_bounds__(768) void gemv_rows(const _Float16* __restrict__ x, const uint8_t* __restrict__ w0,
                                                  void* __restrict__ out0, int n0, int k, int m_rows, int per,
                                                  int split, int slice_steps, int flags, const RowsMore more) {
  using U = Unit<TYPE>;
  constexpr int MG = MR > 4 ? 2 : 1;      // MFMA groups of four activation rows
  constexpr int LIVE = MR == 1 ? 1 : 4;   // rows kept per group
  constexpr int CHUNKS = U::ELEMS / 8, PER_SUB = U::SUB / 8, SUBS = U::ELEMS / U::SUB;
  constexpr int XCHUNKS = MR == 1 ? 1 : MR == 4 ? 2 : 4;  // 16-byte activation chunks a thread loads at a time
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, threads = 64 * per * split;
  const int wave = scalar(tid >> 6);
  const int col = lane & 15, g = lane >> 4;
  const bool pair = flags & kRowsSwiglu;

  // the workgroup's matrix, the wave's row tile (SwiGLU: gate and up tiles in turn) and K range
  const int block = blockIdx.x;
  int mat = 0, n = n0, first_block = 0;
  const uint8_t* w = w0;
  void* out = out0;
  if (flags & kRowsGroup) {
    mat = (block >= more.first_block[0]) + (block >= more.first_block[1]);
    if (mat) {
      w = more.w[mat - 1];
      out = more.out[mat - 1];
      n = more.n[mat - 1];
      first_block = more.first_block[mat - 1];
    }
  }
  const int tile_of_block = (block - first_block) * (pair ? per >> 1 : per);
  const int tile = scalar(quotient(wave, inverse(split))), range = wave - tile * split;
  const int blocks = k / Block<TYPE>::QK;  // of a row
  const int units = U::BLOCK32 ? (blocks + 1) / 2 : k / U::ELEMS;
  const int steps = (units + 3) / 4;
  Fetch<TYPE> fetch;

  // activation rows in LDS: a slice of columns each, 16 bytes past a multiple of 256 so that the
  // rows of a b128 read start in different banks
  const int row_lds = slice_steps * 4 * U::ELEMS * 2 + 16;
  const int zero_at = m_rows * row_lds;
  uint8_t* staged = lds + zero_at + kRowsZero + wave * (16 * U::ROW);  // the wave's own
  const int xm = col & 3;
  const bool mine = (col >> 2) == g;
  const bool active0 = mine && xm < m_rows, active1 = MG == 2 && mine && xm + 4 < m_rows;
  if (tid < kRowsZero / 16) *reinterpret_cast<uint4*>(lds + zero_at + 16 * tid) = make_uint4(0, 0, 0, 0);

  float acc[MG][LIVE] = {};
  half8_t ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = (_Float16)1.0f;

  for (int s0 = 0; s0 < steps; s0 += slice_steps) {
    const int last = min(s0 + slice_steps, steps);
    const int col0 = s0 * 4 * U::ELEMS;
    const int all16 = (last - s0) * (U::ELEMS / 2);  // 16-byte chunks of a row, with zeros to whole steps
    const int live16 = min(all16, (k - col0) >> 3);  // those that hold activations
    const int total = m_rows * all16;
    const float inv16 = inverse(all16);
    // The activations are requested first, XCHUNKS chunks a thread (past the last: the last again),
    // then the wave's first weights, and only then are the activations waited for.
    auto chunk_of = [&](int c, int& at, bool& live) {
      c = min(c, total - 1);
      const int m = quotient(c, inv16), e = c - m * all16;
      at = m * row_lds + 16 * e;
      live = e < live16;
      return x + ((size_t)m * k + (uint32_t)(col0 + 8 * min(e, live16 - 1)));
    };
    uint4 xr[XCHUNKS];
    int at[XCHUNKS];
    bool live[XCHUNKS];
#pragma unroll
    for (int i = 0; i < XCHUNKS; ++i) xr[i] = *reinterpret_cast<const uint4*>(chunk_of(tid + i * threads, at[i], live[i]));
    int s = s0 + range;
    if (s0 == 0)
      fetch.init(pair && (tile & 1) ? more.w[0] : w, min((tile_of_block + (pair ? tile >> 1 : tile)) * 16, n - 1), n,
                 (uint32_t)(blocks * Block<TYPE>::BYTES), lane);
    fetch.load(min(s, last - 1));
    asm volatile("" ::: "memory");
#pragma unroll
    for (int i = 0; i < XCHUNKS; ++i)
      *reinterpret_cast<uint4*>(lds + at[i]) = live[i] ? xr[i] : make_uint4(0, 0, 0, 0);
    for (int c = tid + XCHUNKS * threads; c - tid < total; c += XCHUNKS * threads) {
#pragma unroll
      for (int i = 0; i < XCHUNKS; ++i) xr[i] = *reinterpret_cast<const uint4*>(chunk_of(c + i * threads, at[i], live[i]));
#pragma unroll
      for (int i = 0; i < XCHUNKS; ++i)
        *reinterpret_cast<uint4*>(lds + at[i]) = live[i] ? xr[i] : make_uint4(0, 0, 0, 0);
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");

    for (; s < last; s += split) {
      const int xat = ((s - s0) * 4 * U::ELEMS + U::lane_at(g)) * 2;
      half8_t xv[CHUNKS][MG];
      const uint8_t* x0 = lds + (active0 ? xm * row_lds + xat : zero_at);
      const uint8_t* x1 = lds + (active1 ? (xm + 4) * row_lds + xat : zero_at);
#pragma unroll
      for (int t = 0; t < CHUNKS; ++t) {
        xv[t][0] = *reinterpret_cast<const half8_t*>(x0 + 2 * U::chunk_at(t));
        if constexpr (MG == 2) xv[t][MG - 1] = *reinterpret_cast<const half8_t*>(x1 + 2 * U::chunk_at(t));
      }
      U unit;
      fetch.store(staged, lane);
      if (s + split < last) fetch.load(s + split);
      asm volatile("" ::: "memory");  // a wave's LDS operations complete in order
      unit.read(staged + col * U::ROW, g);
      asm volatile("" ::: "memory");
      const int u = 4 * s + g;
      const bool valid = u < units, valid2 = !U::BLOCK32 || 2 * u + 1 < blocks;
      auto sub = [&](auto index) {
        constexpr int S = decltype(index)::value;
        float4v d[MG] = {}, sums[MG] = {};
        auto mul = [&](auto offset) {
          constexpr int T = S * PER_SUB + decltype(offset)::value;
          const half8_t b = unit.template chunk<T>(g);
#pragma unroll
          for (int i = 0; i < MG; ++i) d[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[T][i], b, d[i], 0, 0, 0);
          if constexpr (U::MIN) {
#pragma unroll
            for (int i = 0; i < MG; ++i) sums[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv[T][i], ones, sums[i], 0, 0, 0);
          }
        };
        mul(std::integral_constant<int, 0>{});
        mul(std::integral_constant<int, 1>{});
        if constexpr (PER_SUB == 4) {
          mul(std::integral_constant<int, 2>{});
          mul(std::integral_constant<int, 3>{});
        }
        float sc, low;
        unit.template scale<S>(g, valid, valid2, sc, low);
#pragma unroll
        for (int i = 0; i < MG; ++i)
#pragma unroll
          for (int r = 0; r < LIVE; ++r) {
            acc[i][r] = fmaf(sc, d[i][r], acc[i][r]);
            if constexpr (U::MIN) acc[i][r] = fmaf(low, sums[i][r], acc[i][r]);
          }
      };
      sub(std::integral_constant<int, 0>{});
      sub(std::integral_constant<int, 1>{});
      if constexpr (SUBS >= 4) {
        sub(std::integral_constant<int, 2>{});
        sub(std::integral_constant<int, 3>{});
      }
      asm volatile("" ::: "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the activations' place is free
  }

  // the four pieces' sums, then the waves' partial tiles [wave][m][16] over K in range order
  float* partial = reinterpret_cast<float*>(lds);
  const int tile_items = m_rows * 16;
#pragma unroll
  for (int i = 0; i < MG; ++i)
#pragma unroll
    for (int r = 0; r < LIVE; ++r) {
      const float v = sum_pieces(acc[i][r]);
      if (g == 0 && 4 * i + r < m_rows) partial[wave * tile_items + (4 * i + r) * 16 + col] = v;
    }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int step = pair ? 2 : 1, outputs = (pair ? per >> 1 : per) * tile_items;
  const float inv_items = inverse(tile_items);
  for (int first = 64 * wave; first < outputs; first += threads) {
    const int o = min(first + lane, outputs - 1);
    const int t = quotient(o, inv_items), in_tile = o - t * tile_items, m = in_tile >> 4;
    const float* p = partial + t * step * split * tile_items + in_tile;
    const int row = (tile_of_block + t) * 16 + (in_tile & 15);
    const bool live = first + lane < outputs && row < n;
    auto over_ranges = [&](const float* from) {  // in range order, four reads in flight
      float v = 0.0f;
      for (int q = 0; q < split; q += 4) {
        float r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) r[i] = from[min(q + i, split - 1) * tile_items];
#pragma unroll
        for (int i = 0; i < 4; ++i) v += q + i < split ? r[i] : 0.0f;
      }
      return v;
    };
    float v = over_ranges(p), up = 0.0f;
    if (pair) up = over_ranges(p + split * tile_items);
    if constexpr (by_element<TYPE>()) {
      uint64_t rest = __builtin_amdgcn_ballot_w64(live && !(is_finite(v) && is_finite(up)));
      for (; __builtin_expect(rest != 0, 0); rest &= rest - 1) {
        const int l = __builtin_ctzll(rest);
        const size_t at = (size_t)__builtin_amdgcn_readlane(row, l) * (size_t)(blocks * Block<TYPE>::BYTES);
        const _Float16* xm = x + (size_t)__builtin_amdgcn_readlane(m, l) * k;
        const float exact = element_product<TYPE>(w + at, xm, k, lane);
        const float exact_up = pair ? element_product<TYPE>(more.w[0] + at, xm, k, lane) : 0.0f;
        if (lane == l) v = exact, up = exact_up;
      }
    }
    if (pair) v = swiglu(v, up);
    if (!live) continue;
    const size_t index = (size_t)m * n + row;
    if (flags & kRowsHalf) store_out(static_cast<_Float16*>(out), index, v);
    else store_out(static_cast<float*>(out), index, v);
  }
}

struct RowsLaunch {
  const GemvArgs* g;
  RowsMore more;
  int per, split, slice_steps, flags, grid;
  size_t lds;
};

template <int TYPE, int MR>
hipError_t launch_rows(const RowsLaunch& l, hipStream_t stream) {
  const GemvArgs& g = l.g[0];
  hipLaunchKernelGGL((gemv_rows<TYPE, MR>), dim3(l.grid), dim3(64 * l.per * l.split), l.lds, stream,
                     static_cast<const _Float16*>(g.x), static_cast<const uint8_t*>(g.w), g.out, g.n, g.k, g.m, l.per,
                     l.split, l.slice_steps, l.flags, l.more);
  return hipGetLastError();
}

template <int TYPE>
hipError_t launch_rows_type(RowsLaunch& l, int count, hipStream_t stream) {
  using U = Unit<TYPE>;
  const int m = l.g[0].m, k = l.g[0].k;
  const int pair = l.flags & kRowsSwiglu ? 2 : 1;  // tiles that stay together
  int rows[kGemvGroupMax];
  for (int i = 0; i < count; ++i) rows[i] = l.g[i].n;
  const int steps = (k + 4 * U::ELEMS - 1) / (4 * U::ELEMS);
  const auto [groups, max_waves] = plan_gemv_rows(rows, count, m, pair > 1);
  l.per = groups * pair;
  const int most = std::max(1, std::min(max_waves / l.per, steps)), rounds = (steps + most - 1) / most;
  l.split = (steps + rounds - 1) / rounds;  // the fewest ranges of that many steps
  l.grid = 0;
  for (int i = 0; i < count; ++i) {
    l.grid += ((l.g[i].n + 15) / 16 + groups - 1) / groups;
    if (i < kGemvGroupMax - 1) l.more.first_block[i] = i + 1 < count ? l.grid : 0x7fffffff;
  }
  for (int i = count; i < kGemvGroupMax - 1; ++i) l.more.first_block[i] = 0x7fffffff;
  const int waves = l.per * l.split;
  const int max_lds = 156 * 1024;
  const int step_bytes = 4 * U::ELEMS * 2;
  const int fixed = kRowsZero + 16 * m + waves * 16 * U::ROW;
  l.slice_steps = std::max(1, std::min(steps, (max_lds - fixed) / (m * step_bytes)));
  l.lds = std::max((size_t)m * (l.slice_steps * step_bytes) + fixed, (size_t)waves * m * 16 * 4);
  if (m == 1) return launch_rows<TYPE, 1>(l, stream);
  if (m <= 4) return launch_rows<TYPE, 4>(l, stream);
  return launch_rows<TYPE, 8>(l, stream);
}

}  // namespace

bool gemv_rows_single(const GemvArgs& a) {
  if (a.x_f32 || a.m < 1 || a.m > kGemvMaxM || a.k > kRowsMaxK) return false;
  return gemv_rows_single_better(a.type, a.m, a.n, a.k);
}

bool gemv_rows_group(const GemvArgs* a, int count) {
  if (count < 2 || a[0].x_f32 || a[0].m < 1 || a[0].m > kGemvMaxM || a[0].k > kRowsMaxK) return false;
  int rows[kGemvGroupMax];
  for (int i = 0; i < count; ++i) rows[i] = a[i].n;
  return gemv_rows_group_better(rows, count, a[0].m, a[0].k);
}

bool gemv_rows_pair(const GemvArgs& a) {
  if (a.x_f32 || a.m < 1 || a.m > kGemvMaxM || a.k > kRowsMaxK) return false;
  return gemv_rows_pair_better(a.type, a.m, a.n, a.k);
}

hipError_t launch_gemv_rows(const GemvArgs* g, int count, const void* w_up, hipStream_t stream) {
  RowsLaunch l{};
  l.g = g;
  l.flags = (g[0].out_half ? kRowsHalf : 0) | (w_up ? kRowsSwiglu : 0) | (count > 1 ? kRowsGroup : 0);
  for (int i = 0; i < count; ++i) {
    if (i) l.more.out[i - 1] = g[i].out;
    if (i) l.more.w[i - 1] = static_cast<const uint8_t*>(g[i].w);
    if (i) l.more.n[i - 1] = g[i].n;
  }
  if (w_up) l.more.w[0] = static_cast<const uint8_t*>(w_up);
  switch (g[0].type) {
    case kQ4_0: return launch_rows_type<kQ4_0>(l, count, stream);
    case kQ4_1: return launch_rows_type<kQ4_1>(l, count, stream);
    case kQ5_0: return launch_rows_type<kQ5_0>(l, count, stream);
    case kQ5_1: return launch_rows_type<kQ5_1>(l, count, stream);
    case kQ8_0: return launch_rows_type<kQ8_0>(l, count, stream);
    case kQ2_K: return launch_rows_type<kQ2_K>(l, count, stream);
    case kQ3_K: return launch_rows_type<kQ3_K>(l, count, stream);
    case kQ4_K: return launch_rows_type<kQ4_K>(l, count, stream);
    case kQ5_K: return launch_rows_type<kQ5_K>(l, count, stream);
    case kQ6_K: return launch_rows_type<kQ6_K>(l, count, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tensor_gguf
