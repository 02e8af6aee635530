// Dequant-GEMM of 9 to 64 activation rows that streams the weights, every encoding and row length:
// out[m, n] = sum_k fp16(x[m, k]) * fp16(dequant(W)[n, k]), fp32 accumulate, up to three matrices
// that share x in one launch.
//
// The fetch of the matrix-core decode GEMV (gguf_gemv_rows.hip): a wave takes 16 rows x 256 columns at a
// time, 16-byte pieces along the rows, passed through LDS to the lanes that own them (lane n + 16 g:
// unit g of row n).  A lane turns each 8 codes of its unit into fp16 weights (one fp32 fma per code from
// its exact fp16 value, then the fp16 cast: the values every GEMM here stages) and they are
// the B operand of one MFMA per 16 activation rows as they are: the A operand's lane m + 16 g reads
// x[m] at the columns of unit g, so any assignment of columns to lane groups gives the same sum.
// Weights go through no LDS tile after decoding and are decoded once for all M.
//
// A workgroup owns up to twelve row tiles of 16, 32 or 64 activation rows and splits the columns of a
// slice over its remaining waves; slices of the activations are staged in LDS, the next one's loads in
// flight in registers.  No K split across workgroups: no workspace, no second launch.
//
// What bounds it: what a CU reads, weights and its workgroup's activations (64 KB a row tile at M = 32
// and K = 1024) through L2, hence the split of M over workgroups where the matrix is narrow.
// Microseconds per launch (graph replays, weights rotated), pipelined tiles with their reduce or the
// per-element small-M kernel -> here: Q4_K gate + up 2 x 12288 x 4096 at M = 9 / 32 / 64 42 / 44 / 46 -> 18 / 26
// / 39; q + k + v (4096, 1024, 1024) x 4096 at M = 32 Q4_K 18.3 -> 14.0, Q6_K 28.8 -> 16.0; Q6_K 4096 x 12288
// 36.1 -> 26.5; Q5_0 12288 x 4096 56.7 -> 19.1; packed form, fp32 x, 4096 x 4096 at M = 8 Q3_K 18.1 -> 8.5.
#include <algorithm>

#include "gguf_rows.h"
#include "gguf_rows_plan.h"

namespace tensor_gguf {
namespace {

struct GemmRowsMore {
  const uint8_t* w[kGemmGroupMax - 1];
  void* out[kGemmGroupMax];
  int n[kGemmGroupMax - 1];
  int first_block[kGemmGroupMax - 1];  // first workgroup of matrices 1 and 2
  int blocks;                          // workgroups of all matrices, for one set of activation rows
  bool out_half, group;
};

// XT = float: fp32 activations (the packed call form), rounded to fp16 as they are staged.
template <int TYPE, int MT, typename XT>
__global__ __launch_bounds__(64 * kRowsWaves) void gemm_rows(const XT* __restrict__ x, const uint8_t* __restrict__ w0, int n0,
                                                 int k, int m_all, int per, int split, int slice_steps, int m_splits,
                                                 const GemmRowsMore more) {
  using U = Unit<TYPE>;
  constexpr int CHUNKS = U::ELEMS / 8, PER_SUB = U::SUB / 8, SUBS = U::ELEMS / U::SUB;
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int threads = 64 * kRowsWaves;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = scalar(tid >> 6);
  const int col = lane & 15, g = lane >> 4;

  // The workgroups of one set of weight rows and different activation rows are 8 apart: on the same
  // XCD, whose L2 then reads the weights once.
  int block = blockIdx.x, m_split = 0;
  if (m_splits > 1) {
    const int set = (int)(blockIdx.x >> 3) / m_splits;
    m_split = (int)(blockIdx.x >> 3) - set * m_splits;
    block = set * 8 + (blockIdx.x & 7);
    if (block >= more.blocks) return;
  }
  const int m0 = m_split * (16 * MT), m_rows = min(16 * MT, m_all - m0);
  x += (size_t)m0 * k;
  int mat = 0, n = n0, first_block = 0;
  const uint8_t* w = w0;
  if (more.group) {
    mat = (block >= more.first_block[0]) + (block >= more.first_block[1]);
    if (mat) {
      w = more.w[mat - 1];
      n = more.n[mat - 1];
      first_block = more.first_block[mat - 1];
    }
  }
  const int tile0 = (block - first_block) * per;
  const int tile = scalar(quotient(wave, inverse(split))), range = wave - tile * split;
  const bool computes = wave < per * split;  // the other waves only help to stage activations
  const int blocks = k / Block<TYPE>::QK;
  const int units = U::BLOCK32 ? (blocks + 1) / 2 : k / U::ELEMS;
  const int steps = (units + 3) / 4;

  const int row_lds = slice_steps * 512 + 16;  // a slice's columns of one activation row, and 16 bytes
  uint8_t* staged = lds + m_rows * row_lds + wave * (16 * U::ROW);

  // 16-byte pieces of the slice at step s0, E activations each: all of a row's, with zeros to whole
  // steps, and those that hold activations
  constexpr int E = 16 / sizeof(XT);
  uint4 xr[kXRegs];
  auto pieces = [&](int s0, int& all, int& live, float& inv) {
    all = min(slice_steps, steps - s0) * (256 / E);
    live = min(all, (k - s0 * 256) / E);
    inv = inverse(all);
  };
  auto slice_load = [&](int s0) {
    int all, live;
    float inv;
    pieces(s0, all, live, inv);
#pragma unroll
    for (int i = 0; i < kXRegs; ++i) {
      const int c = min(tid + i * threads, m_rows * all - 1), m = quotient(c, inv), e = c - m * all;
      xr[i] = *reinterpret_cast<const uint4*>(x + ((size_t)m * k + (uint32_t)(s0 * 256 + E * min(e, live - 1))));
    }
  };
  auto slice_store = [&](int s0) {
    int all, live;
    float inv;
    pieces(s0, all, live, inv);
#pragma unroll
    for (int i = 0; i < kXRegs; ++i) {
      const int c = min(tid + i * threads, m_rows * all - 1), m = quotient(c, inv), e = c - m * all;
      const uint4 v = e < live ? xr[i] : make_uint4(0, 0, 0, 0);
      if constexpr (E == 8) {
        *reinterpret_cast<uint4*>(lds + m * row_lds + 16 * e) = v;
      } else {
        *reinterpret_cast<uint2*>(lds + m * row_lds + 8 * e) =
            make_uint2(half2_from_fp32(__builtin_bit_cast(float, v.x), __builtin_bit_cast(float, v.y)),
                       half2_from_fp32(__builtin_bit_cast(float, v.z), __builtin_bit_cast(float, v.w)));
      }
    }
  };

  slice_load(0);
  Fetch<TYPE> fetch;
  int s = range;
  if (computes) {
    fetch.init(w, min((tile0 + tile) * 16, n - 1), n, (uint32_t)(blocks * Block<TYPE>::BYTES), lane);
    fetch.load(min(s, steps - 1));
  }
  const uint8_t* xrow[MT];  // this lane's activation rows as the A operand (rows past M: the last again)
#pragma unroll
  for (int i = 0; i < MT; ++i) xrow[i] = lds + min(16 * i + col, m_rows - 1) * row_lds + 2 * U::lane_at(g);

  float4v acc[MT] = {};
  for (int s0 = 0; s0 < steps; s0 += slice_steps) {
    const int last = min(s0 + slice_steps, steps);
    slice_store(s0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (last < steps) slice_load(last);
    if (computes) {
      for (; s < last; s += split) {
        fetch.store(staged, lane);
        if (s + split < steps) fetch.load(s + split);
        asm volatile("" ::: "memory");  // a wave's LDS operations complete in order
        U unit;
        unit.read(staged + col * U::ROW, g);
        asm volatile("" ::: "memory");
        const int u = 4 * s + g;
        const bool valid = u < units, valid2 = !U::BLOCK32 || 2 * u + 1 < blocks;
        const int xat = (s - s0) * 512;
        auto sub = [&](auto index) {
          constexpr int S = decltype(index)::value;
          float sc, low;
          unit.template scale<S>(g, valid, valid2, sc, low);
          auto mul = [&](auto offset) {
            constexpr int T = S * PER_SUB + decltype(offset)::value;
            const half8_t q = unit.template chunk<T>(g);
            uint32_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i)
              v[i] = half2_from_fp32(fmaf((float)q[2 * i], sc, low), fmaf((float)q[2 * i + 1], sc, low));
            const half8_t b = __builtin_bit_cast(half8_t, make_uint4(v[0], v[1], v[2], v[3]));
#pragma unroll
            for (int i = 0; i < MT; ++i) {
              const half8_t xv = *reinterpret_cast<const half8_t*>(xrow[i] + xat + 2 * U::chunk_at(T));
              acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xv, b, acc[i], 0, 0, 0);
            }
          };
          mul(std::integral_constant<int, 0>{});
          mul(std::integral_constant<int, 1>{});
          if constexpr (PER_SUB == 4) {
            mul(std::integral_constant<int, 2>{});
            mul(std::integral_constant<int, 3>{});
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
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the slice's place is free
  }

  // partial tiles [wave][m][16] over the activations, then their sum in range order
  float* partial = reinterpret_cast<float*>(lds);
  const int tile_items = m_rows * 16;
  if (computes) {
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int m = 16 * i + 4 * g + r;
        if (m < m_rows) partial[wave * tile_items + m * 16 + col] = acc[i][r];
      }
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  const int outputs = per * tile_items;
  const float inv_items = inverse(tile_items);
  for (int o = tid; o < outputs; o += threads) {
    const int t = quotient(o, inv_items), in_tile = o - t * tile_items;
    const float* p = partial + t * split * tile_items + in_tile;
    float v = 0.0f;
    for (int q = 0; q < split; q += 4) {
      float r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = p[min(q + i, split - 1) * tile_items];
#pragma unroll
      for (int i = 0; i < 4; ++i) v += q + i < split ? r[i] : 0.0f;
    }
    const int row = (tile0 + t) * 16 + (in_tile & 15);
    if (row >= n) continue;
    const size_t index = (size_t)(m0 + (in_tile >> 4)) * n + row;
    if (more.out_half) store_out(static_cast<_Float16*>(more.out[mat]), index, v);
    else store_out(static_cast<float*>(more.out[mat]), index, v);
  }
}

struct GemmRowsLaunch {
  const GemmGroupArgs* a;
  GemmRowsMore more;
  int per, split, slice_steps, m_splits, grid;
  size_t lds;
};

template <int TYPE, int MT>
hipError_t launch_rows(const GemmRowsLaunch& l, hipStream_t stream) {
  const GemmGroupArgs& a = *l.a;
  const uint8_t* w = static_cast<const uint8_t*>(a.w[0]);
  if (a.x_f32)
    hipLaunchKernelGGL((gemm_rows<TYPE, MT, float>), dim3(l.grid), dim3(64 * kRowsWaves), l.lds, stream,
                       static_cast<const float*>(a.x), w, a.n[0], a.k, a.m, l.per, l.split, l.slice_steps, l.m_splits,
                       l.more);
  else
    hipLaunchKernelGGL((gemm_rows<TYPE, MT, _Float16>), dim3(l.grid), dim3(64 * kRowsWaves), l.lds, stream,
                       static_cast<const _Float16*>(a.x), w, a.n[0], a.k, a.m, l.per, l.split, l.slice_steps,
                       l.m_splits, l.more);
  return hipGetLastError();
}

template <int TYPE>
hipError_t launch_rows_type(GemmRowsLaunch& l, hipStream_t stream) {
  using U = Unit<TYPE>;
  const GemmGroupArgs& a = *l.a;
  const int steps = (a.k + 255) / 256;
  const GemmRowsPlan plan = plan_gemm_rows(a.n, a.count, a.m, a.k, (double)Block<TYPE>::BYTES / Block<TYPE>::QK,
                                           a.x_f32);
  l.m_splits = plan.m_splits;
  l.per = plan.per;
  const int m = std::min(a.m, 16 * plan.t);
  // the slice that the threads' registers and LDS hold
  const int lds_x = 158 * 1024 - kRowsWaves * 16 * U::ROW - 16 * m;
  l.slice_steps = std::min({steps, gemm_rows_slice(m, a.x_f32), lds_x / (m * 512)});
  if (l.slice_steps < 1) return hipErrorInvalidValue;
  l.split = std::max(1, std::min(kRowsWaves / l.per, l.slice_steps));
  if (l.slice_steps < steps) l.slice_steps = l.slice_steps / l.split * l.split;  // every wave a whole share
  l.grid = 0;
  for (int i = 0; i < a.count; ++i) {
    l.grid += ((a.n[i] + 15) / 16 + l.per - 1) / l.per;
    if (i < kGemmGroupMax - 1) l.more.first_block[i] = i + 1 < a.count ? l.grid : 0x7fffffff;
  }
  for (int i = a.count; i < kGemmGroupMax - 1; ++i) l.more.first_block[i] = 0x7fffffff;
  l.more.blocks = l.grid;
  if (l.m_splits > 1) l.grid = (l.grid + 7) / 8 * 8 * l.m_splits;
  l.lds = std::max((size_t)m * (l.slice_steps * 512 + 16) + (size_t)kRowsWaves * 16 * U::ROW,
                   (size_t)l.per * l.split * m * 64);
  switch (plan.t) {
    case 1: return launch_rows<TYPE, 1>(l, stream);
    case 2: return launch_rows<TYPE, 2>(l, stream);
    default: return launch_rows<TYPE, 4>(l, stream);
  }
}

}  // namespace

bool gemm_skinny_takes(const GemmGroupArgs& a) {
  return a.m <= kSkinnyMaxM && a.count == 1 && gemm_skinny_better(a.type, a.m, a.n[0], a.k, a.x_f32);
}

// M <= 64, but
//  * long rows with a K split across workgroups to take (a plan with a workspace) at M > 32, where every workgroup
//    stages 16 or 32 whole activation rows for its few weight rows: 4096 x 12288 Q4_K at M = 64 31.4
//    against 26.3 us, at M = 32 21.6 against 23.9;
//  * one matrix of short rows, where latency is all (gemm_skinny_better).
bool gemm_rows_takes(const GemmGroupArgs& a, const GemmPlan& plan) {
  if (a.m > 64 || a.k > kRowsMaxK) return false;
  if (a.m > 32 && a.k >= 8192 && plan.small_m && plan.splits > 1) return false;
  return !gemm_skinny_takes(a);
}

hipError_t launch_gemm_rows(const GemmGroupArgs& a, hipStream_t stream) {
  GemmRowsLaunch l{};
  l.a = &a;
  l.more.out_half = a.out_half;
  l.more.group = a.count > 1;
  for (int i = 0; i < a.count; ++i) {
    l.more.out[i] = a.out[i];
    if (i) l.more.w[i - 1] = static_cast<const uint8_t*>(a.w[i]);
    if (i) l.more.n[i - 1] = a.n[i];
  }
  switch (a.type) {
    case kQ4_0: return launch_rows_type<kQ4_0>(l, stream);
    case kQ4_1: return launch_rows_type<kQ4_1>(l, stream);
    case kQ5_0: return launch_rows_type<kQ5_0>(l, stream);
    case kQ5_1: return launch_rows_type<kQ5_1>(l, stream);
    case kQ8_0: return launch_rows_type<kQ8_0>(l, stream);
    case kQ2_K: return launch_rows_type<kQ2_K>(l, stream);
    case kQ3_K: return launch_rows_type<kQ3_K>(l, stream);
    case kQ4_K: return launch_rows_type<kQ4_K>(l, stream);
    case kQ5_K: return launch_rows_type<kQ5_K>(l, stream);
    case kQ6_K: return launch_rows_type<kQ6_K>(l, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace tensor_gguf
