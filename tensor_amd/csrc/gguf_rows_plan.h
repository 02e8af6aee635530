// Launch shapes of the kernels that stream 16-row tiles (gguf_gemv_rows.hip, gguf_gemm_rows.hip), and the
// lines between them and the kernels they stand beside: plain host code without HIP, so that a CPU
// test can compile it by itself.
#pragma once

#include <algorithm>

#include "gguf_types.h"

namespace tensor_gguf {

constexpr int kRowsMaxK = 1 << 22;  // 16 rows stay within the 32-bit offsets of a tile

// The streaming GEMM's launch: workgroups of `per` row tiles and 16 t activation rows, m_splits of
// which share a set of weight rows.
struct GemmRowsPlan {
  int t, per, m_splits;
};

constexpr int kRowsWaves = 12;  // waves of a streaming GEMM workgroup, one workgroup a CU

// Workgroups of one set of activation rows: row tiles are grouped within a matrix, so each
// matrix rounds up by itself.
inline long rows_blocks(const int* n, int count, int per) {
  long blocks = 0;
  for (int i = 0; i < count; ++i) blocks += ((n[i] + 15) / 16 + per - 1) / per;
  return blocks;
}

// Rounds of the 256 CUs that a launch takes: the sets of weight rows go round the eight XCDs in turn,
// each with its m_splits workgroups (32 CUs an XCD).
inline long gemm_rows_rounds(const int* n, int count, const GemmRowsPlan& plan) {
  return ((rows_blocks(n, count, plan.per) + 7) / 8 * plan.m_splits + 31) / 32;
}

// 256-column steps of an activation slice of `rows` rows that a workgroup's threads hold in registers.
constexpr int kXRegs = 8;  // 16-byte activation chunks of the next slice a thread holds
inline int gemm_rows_slice(int rows, bool x_f32) {
  return kXRegs * kRowsWaves * 64 * 16 / (rows * (x_f32 ? 1024 : 512));
}

// The (t, per) of least cost, rounds x what a workgroup takes: its start and end, and for each 256
// columns the decode, products and weights of its tiles (over fewer waves where a slice has fewer steps
// than a tile has waves) and the staging of its activations.  In units of ~15 ns, fitted to
// 420 shapes and row counts of Q4_K, Q6_K, Q8_0, Q5_0 and Q2_K timed at every (t, per): the choice is 0.7%
// slower than the best on average, 11% at the 99th percentile.  Counting tiles over all matrices
// instead of the workgroups launched, and reads without the decode, took a second round for four workgroups or
// decoded everything four times: q + k + v (4096, 1024, 1024) x 4096 Q4_K at M = 32 23.5 -> 14.0 us, at M =
// 64 34.9 -> 18.2; 3 x 4096 rows at M = 32 36.0 -> 19.0; 8192 columns, (8192, 1024, 1024), Q8_0 at M =
// 48 83.8 -> 42.9.
inline GemmRowsPlan plan_gemm_rows(const int* n, int count, int m, int k, double bytes_per_element, bool x_f32) {
  const int m16 = (m + 15) / 16, steps = (k + 255) / 256;
  GemmRowsPlan best{1, 1, m16};
  double least = 0;
  for (int t : {1, 2, 4}) {
    if (t > 1 && t >= 2 * m16) break;  // no more rows than M
    const int rows = std::min(m, 16 * t), slice = std::max(1, gemm_rows_slice(rows, x_f32));
    const double staging = rows * (rows > 48 && steps > slice ? 1.6 : 1.0);
    for (int per = 1; per <= kRowsWaves; ++per) {
      const GemmRowsPlan plan{t, per, (m16 + t - 1) / t};
      const long rounds = gemm_rows_rounds(n, count, plan);
      const int waves = kRowsWaves / per;  // of a tile
      const double idle = steps > slice && slice < waves ? (double)waves / slice : 1.0;
      const double cost = rounds * (150 + steps * (per * (7 + 2 * t + 7 * bytes_per_element) * idle + staging));
      if (least == 0 || cost < least) best = plan, least = cost;
      if (rounds == 1) break;  // more tiles only make that round longer
    }
  }
  return best;
}

// Whether one matrix is left to the per-element kernel (gemm_skinny): short rows, where latency is all and the streaming
// kernel starts and ends ~1 us later.  It decodes per element, so the encodings differ in how long a row may be; K of
// its 512-column passes counts against it, and for the streaming kernel whole rounds of 256-column steps over its waves (K = 512
// and 1024 are, 544 to 768 and 1792 leave waves idle), hence the exceptions.  From graph replays of both
// kernels, every encoding, M = 2 to 64, 320 to 20000 rows of 256 to 4096 columns, fp16 and fp32 x: the choice takes 0.2%
// more than the better one on average (6% at the 99th percentile), with lines on elements 3.0%.  us, per element /
// streaming, M = 16: Q2_K 8192 x 256 4.0 / 4.7, Q4_K 1024 x 1024 4.1 / 4.6 and 320 x 256 3.1 / 4.3, Q6_K 4096 x 512
// 5.2 / 5.0; Q5_1 4096 x 1056 at M = 48 5.1 / 6.8, Q4_K 2560 x 2560 at M = 32 10.0 / 7.1.
inline bool gemm_skinny_better(int type, int m, int n, int k, bool x_f32) {
  // how the decode per element compares: cheap, Q4_K, Q5_0, dear
  const int c = type == kQ4_K ? 1 : type == kQ5_0 ? 2 : type == kQ3_K || type == kQ5_K || type == kQ6_K ? 3 : 0;
  const bool idle = (k + 255) / 256 == 7;
  if (x_f32 && c == 0 && m > 16 && n > 1024 && k > 1056 && k <= 1536)  // 2560 x 1280 at M = 64: Q4_1 8.7 / 7.4 us,
    return type == kQ2_K && m > 32;                                     // Q2_K 6.8 / 7.5
  if (x_f32 && (type == kQ4_1 || type == kQ5_1) && m > 8 && m <= 32 && n <= 2048 && k > 1792 && k <= 2048)
    return true;  // the lightest decode, and a streaming slice of fp32 x ends here: 2048 x 2048 7.4 / 8.3 us, Q5_1
  if (n <= 4096) {
    if (m > 32 && n > 1024) {  // the streaming kernel spreads M over workgroups, each decoding again
      constexpr int longest[4] = {1280, 768, 1056, 768};
      return (k <= longest[c] && !(k == 1024 && (c >= 1 || x_f32))) || (idle && c == 0 && n >= 3072);
    }
    if (c == 1 && n > 1024 && (m > 16 || x_f32)) return k < 512 || (m <= 16 && k == 512);
    if (c == 2) return k <= 768 && k != 512 && (k < 512 || n <= 1024);
    return c == 0 ? k <= 1280 || (type == kQ5_1 && idle) : k <= (c == 1 ? 1024 : 511);
  }
  if (m <= 16) {
    if (n > 8192) return c == 0 && k <= 256 && n <= 10240;
    return c == 0 ? k <= 384 || (type != kQ4_0 && k % 256 != 0 && k <= 1056) : c <= 2 && k <= (c == 1 ? 384 : 256);
  }
  // beyond 4096 rows M's tiles stay in one workgroup, from 8192 with two tiles of W: one round of those only there
  if (n < 8192) return m > 32 && k <= 256 && type != kQ5_K;
  if (n == 8192) {
    if (c == 0) return (k <= 1056 && k != 1024) || ((idle || k == 1280) && type != kQ4_0 && type != kQ4_1);
    return k <= (type == kQ5_K ? 256 : c == 2 && m <= 32 ? 768 : 512);
  }
  return m <= 32 && (c == 0 ? (long long)n * k <= 13ll << 19 && k != 512 : c == 2 && k <= 256 && n <= 20480);
}

// The decode GEMV's workgroups: `groups` row tiles (or gate / up tile pairs) of one matrix and at most
// `waves` waves.
struct GemvRowsPlan {
  int groups, waves;
};

// One workgroup per CU where that holds all tiles, its 12 waves (the most that leave a lane 168
// registers) sharing their steps: 12288 x 4096 at M = 4 (768 tiles) Q4_0 9.4 us with three tiles against
// 10.0 with one tile and 8 waves.  The workgroups that are launched count, each matrix rounding up by
// itself: 3 x 4096 rows of 4096 columns take 258 of three tiles, so four tiles each: Q4_K at M = 4 / 8 17.4 /
// 22.2 -> 11.7 / 15.0 us, Q8_0 19.7 / 23.3 -> 13.9 / 15.7.  Up to six tiles (2 x 12288 rows, 20000
// rows: Q4_K at M = 2 / 8 16.7 / 28.0 -> 14.9 / 20.7 and 16.5 / 27.0 -> 14.2 / 18.8), eight where M > 4
// (2 x 14336 rows Q4_K at M = 6 27.3 -> 22.8, 32000 rows 29.1 -> 24.3).  Larger matrices go in workgroups of four
// tiles and 8 waves, two of which fit a CU beside the activations of four rows: 64000 x 4096 Q6_K at M = 4 45.6 us against 53.0 with 12 waves and 58.6 with one tile; 2 x 14336 rows
// Q4_K at M = 2 17.2 us against 18.6 with seven tiles.
inline GemvRowsPlan plan_gemv_rows(const int* n, int count, int m, bool pair) {
  for (int groups = 1; groups <= (pair ? 4 : m > 4 ? 8 : 6); ++groups)
    if (rows_blocks(n, count, groups) <= 256) return {groups, 12};
  return {4, 8};
}

// Whether a single matrix goes on this kernel rather than on the vector kernels, which reach their result sooner
// where latency is all (1024 x 1024 at M = 1: Q4_0 3.0 against 2.3 us).  A line for M = 1, 2, 3, 4, 5 to 6 and
// 7 to 8, in 2^20 elements times sqrt(n / 4096): few rows leave CUs without a tile, so of two matrices of one size the
// longer rows gain less (Q4_1 at M = 6: 1024 x 6912 9.5 us against 7.1 on the vector kernel, 4096 x 2048 5.4 against
// 6.2).  They lie where graph replays of both sides crossed, every encoding at 640 to 12288 rows of 512 to 6912 columns,
// weights in the caches and out of them: the choice takes 1.1% more than the better one on average and up to 14% near a
// line, where lines on elements alone took 3.3% and up to 34%.
// A band of row lengths moves a line: up to 2048 columns are one pass of the Q4_0 and Q8_0 vector kernels, of which shorter
// ones leave lanes idle (Q8_0 at M = 4: 3000 x 1536 4.1 us there, 4.5 here; 3000 x 2560 6.9 and 5.8), from M = 2 to
// 6 whole passes beyond too (Q4_0 5120 x 4096 at M = 2 5.5 and 6.3), and Q2_K's gain at up to 1024.  Q6_K's holds to one
// round of waves of long rows, 2048 rows at M = 3 (x 4096 5.5 and 6.2, 2560 x 4096 6.9 and 5.9).
inline bool gemv_rows_single_better(int type, int m, int n, int k) {
  const double millions = (double)n * k / (1 << 20), size2 = millions * millions * n / 4096;
  const int at = m <= 4 ? m - 1 : m <= 6 ? 4 : 5;
  const auto from = [&](const double (&lines)[6], double band = 1) {
    return size2 >= lines[at] * band * (lines[at] * band);
  };
  const bool whole_step = m == 1 && k % 4096 == 0 && k <= 16384;  // row lengths of the tuned M = 1 kernels
  const bool half_step = m == 1 && k % 2048 == 0 && k <= 16384;
  const bool whole = (k > 1024 && k <= 2048) || (k % 2048 == 0 && at >= 1 && at <= 4);
  const double one_pass = !whole ? 1 : m <= 2 ? 1.4 : 2.2;
  switch (type) {
    case kQ4_0: return !half_step && from({38, 18, 3.8, 2.5, 1, 0.5}, one_pass);
    case kQ4_1: return !half_step && from({28, 13.8, 8, 4.4, 3.6, 1.7});
    case kQ5_0: return !half_step && from({5.7, 4.4, 3.6, 1.6, 1.7, 0.75});
    case kQ5_1: return !half_step && from({18, 9.8, 5.7, 3.6, 3.6, 1.7});
    case kQ8_0: return !half_step && from({20.6, 16.8, 6.1, 2.7, 1.3, 0.7}, one_pass);
    case kQ2_K: return !whole_step && from({18, 4.7, 4.7, 1.6, 3.5, 0.75}, k > 1024 ? 1 : m == 2 && k > 512 ? 3 : 2);
    case kQ3_K: return !whole_step && from({3.5, 1.6, 1.1, 1.1, 2, 0.75}, k <= 1024 ? 1.3 : 1);
    case kQ5_K: return !whole_step && from({2, 1.6, 0.75, 0.55, 0.55, 0.55});
    case kQ6_K:
      if (k > 2048 && (m == 3 ? n <= 2048 && k <= 4096 : at == 4 && n <= 1024)) return false;
      return !(whole_step && k <= 12288) && from({13, 0.5, 0.5, 0.5, 0.5, 0.5});
    // M > 1: the plans of tensor_gguf_gemv_plan_v1.  M = 1: rows of 1024 columns are level, of 1536 and 2048 (one
    // pass there too) take 10 to 22% longer here, of 2560 to 6912 2 to 14% less.
    case kQ4_K: return m == 1 && !whole_step && k > 2048;
    default: return false;
  }
}

// The same for SwiGLU pairs, in 2^20 elements of both matrices, where the vector pair kernels (one wave per output row)
// crossed: 2 x 3072 x 1024 at M = 2 Q8_0 4.4 against 4.9 us, at M = 4 6.1 against 5.0; 2 x 6912 x
// 2560 at M = 1 15.4 against 11.3.  Where their rows are one pass the line lies half as high again at M = 1 and 4 (M =
// 1, 2 x 4096 x 2048: Q4_0 4.3 against 4.9, Q4_K 4.7 against 5.2; Q8_0 2 x 2000 x 1056 at M = 4 5.1 against 5.6).
// Q4_K and Q5_K at M = 1 keep their tuned row lengths; Q4_K at M > 1 always comes here (12288 x 4096 at M = 4 about
// 16 us, 18.5 on the sector kernel in pairs that this replaced).
inline bool gemv_rows_pair_better(int type, int m, int n, int k) {
  if ((type == kQ4_K || type == kQ5_K) && m == 1 && k % 4096 == 0 && k <= 16384) return false;
  if (type == kQ4_K && m >= 2) return true;
  const bool slow = type == kQ3_K || type == kQ5_K || type == kQ6_K;  // pairs costly to decode per lane
  const bool one_pass = (type == kQ4_0 || type == kQ8_0 || type == kQ4_K) && k > 1024 && k <= 2048 && (m == 1 || m == 4);
  const int millions = m >= 4 || slow ? 4 : m == 3 ? 8 : 16;
  return 2.0 * n * k >= (double)(millions << 20) * (one_pass ? 1.5 : 1);
}

// Whether a group of two or three matrices goes in one launch, which saves a launch per further matrix (q, k, v
// of 1024 + 2 x 128 rows and 1024 columns at M = 4: one launch of 3.4 us against three of 2.5 to 2.9).
// Matrices that the tuned M = 1 kernels stream faster each by itself keep them from 32 M elements (2 x 12288 x
// 4096 Q6_K: 18.4 against 18.9 us; 6144 x 4096 in three matrices, Q8_0: 12.4 against 8.3).  Wide Q4_K
// matrices at M > 4 are no exception: with the workgroups of plan_gemv_rows 2 x 12288 rows of 4096 columns take
// 20.7 us at M = 8 against 22.5 in two launches, 2 x 28672 x 8192 93 against 117, 2 x 12288 x 12288 57 against 90.
inline bool gemv_rows_group_better(const int* n, int count, int m, int k) {
  if (m > 1 || k % 2048 != 0) return true;
  long long elements = 0;
  for (int i = 0; i < count; ++i) elements += (long long)n[i] * k;
  return elements < 32ll << 20;
}

}  // namespace tensor_gguf
