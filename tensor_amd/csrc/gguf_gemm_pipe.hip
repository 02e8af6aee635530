// Pipelined fused dequant-GEMM on gfx950 (kernel in gguf_gemm_pipe.h; Q4_K, Q5_K, Q6_K, Q8_0 and Q4_0
// here, the other encodings in gguf_gemm_pipe_more.hip):
// out[m, n] = sum_k fp16(x[m, k]) * fp16(W[n, k]), fp32 accumulation
// (reference kernel: AKAS _packed, benchmarks/kernels/showcase/kernels.py:114-119;
//  Triton restatement triton_kernels.py:185-211).
//
// Same tile algorithm as the generic kernel in gguf_gemm.hip (BM x BN
// workgroup tile, BK = 64 steps, LDS-staged fp16 tiles, 16x16x32 fp16 MFMA
// with fp32 accumulators) with a deeper software pipeline:
//
//   * two register sets of raw bytes: step s+1 is dequantized into LDS while
//     step s+2 is in flight from HBM and step s is multiplied (a four-set ring
//     measured no faster: the steps are not bound by load latency);
//   * the LDS double buffer as two arrays, so the compiler may overlap the
//     staging stores of one buffer with the fragment reads of the other;
//   * each step is one straight-line region in which sched_group_barrier
//     interleaves every MFMA with dequant VALU work, an LDS store or a global
//     load, keeping the matrix pipe fed while the VALU decodes;
//   * XDMA (the 256 x 192 tile, and 256 x 128 with fp16 x): the activation tile
//     goes from global memory straight to LDS (global_load_lds_dwordx4, three
//     swizzled buffers), which frees the staging registers the wider tile needs;
//     half of its waves issue a step's MFMAs before their dequant and half after,
//     so the two waves of a SIMD overlap matrix and vector work (ping-pong), and
//     the MFMAs of a step's second half run under the next step's LDS reads;
//   * Q4_K / Q5_K with four (two) threads per weight row: the lanes of a row, a
//     DPP quad (pair), each decode one (two) of the step's four scale factors
//     and share them by broadcasts, instead of each decoding all four.
//
// Weights are dequantized with the reference's fp32 arithmetic (every product
// exact, one rounding) and converted to fp16 with round-to-nearest-even, so
// the staged tiles are bit-exact fp16(dequant(W)).
//   Q4_K (triton_kernels.py:143-162): a step is one 32-byte quant pair j of a
//     super-block, 64 codes: low nibbles = sub-block 2j, high = 2j+1.
//   Q6_K (triton_kernels.py:163-180): a step covers quarters 2(s%2), 2(s%2)+1
//     of half h = (s%4)/2: the 64 low-nibble bytes of ql for that half (nibble
//     s%2), the 32 qh bytes of the half (2 bits per quarter) and 4 scales.
//   Q8_0 / Q4_0 (triton_kernels.py:135-142 for Q4_0): a step is two whole
//     32-element blocks, d * q and (q - 8) * d.
#include "gguf_gemm_pipe.h"

namespace tensor_gguf {
namespace {

// The encodings with plans (K split across workgroups, plans named by the caller).
bool pipe_type(int type) {
  return type == kQ4_K || type == kQ5_K || type == kQ6_K || type == kQ8_0 || type == kQ4_0;
}

int block_bytes(int type) {
  switch (type) {
    case kQ4_0: return Block<kQ4_0>::BYTES;
    case kQ4_1: return Block<kQ4_1>::BYTES;
    case kQ5_0: return Block<kQ5_0>::BYTES;
    case kQ5_1: return Block<kQ5_1>::BYTES;
    case kQ8_0: return Block<kQ8_0>::BYTES;
    case kQ2_K: return Block<kQ2_K>::BYTES;
    case kQ3_K: return Block<kQ3_K>::BYTES;
    case kQ4_K: return Block<kQ4_K>::BYTES;
    case kQ5_K: return Block<kQ5_K>::BYTES;
    default: return Block<kQ6_K>::BYTES;
  }
}
bool block32(int type) { return type == kQ4_0 || type == kQ4_1 || type == kQ5_0 || type == kQ5_1 || type == kQ8_0; }

// The kernel addresses weights and the x tile by 32-bit offsets: every matrix stays under 4 GiB
// and a 256-row x tile under 2 GiB (K <= 2^22); larger shapes take the generic kernel.
bool offsets_fit(const GemmGroupArgs& a) {
  if (a.k > (1 << 22)) return false;
  const uint64_t row = (uint64_t)(a.k / (block32(a.type) ? 32 : 256)) * block_bytes(a.type);
  for (int i = 0; i < a.count; ++i)
    if ((uint64_t)a.n[i] * row >= (1ull << 32)) return false;
  return true;
}

// A tile and split count that fit the shape: K is whole 64-element steps, and the steps of a
// split divide evenly into the workgroup's wave groups, each taking an even number of them (the
// main loop runs two steps per pass) that starts on a super-block (4 steps) for the 256-element
// encodings.
// The LDS-DMA tile takes fp16 x and the encodings whose kernel fits the register file.
bool valid_plan(const GemmGroupArgs& a, int tile, int splits) {
  if (!offsets_fit(a)) return false;
  const int steps = a.k / pipe::BK, unit = block32(a.type) ? 2 : 4;
  if (tile == kDmaTile && (a.x_f32 || !(a.type == kQ4_K || a.type == kQ8_0 || a.type == kQ4_0))) return false;
  return tile >= 0 && tile < kTileCount && splits >= 1 && a.k % pipe::BK == 0 &&
         steps % (unit * kTiles[tile].ks * splits) == 0;
}

// Largest tile that still gives the 256 CUs work: the workgroup count of a tile must reach
// kMinBlocks, else a smaller tile is taken, and below 256 x 128 the K range is split over two
// or four wave groups of one workgroup so that every SIMD holds at least one wave (measured at
// M = 256: 1.4x to 4x faster than the unsplit tiles for the q/k/v/o, gate/up and down shapes).
constexpr long kMinBlocks = 160;

// A tile is taken only where M fills more than half its rows: 256-row tiles from M = 129,
// 128-row tiles from M = 65 (timing harness, Q4_K gate + up 2 x 12288 x 4096: M = 32 69.8 ->
// 39.8 us on 64 x 64 KS2, M = 128 72.3 -> 51.4 on 128 x 128 KS2; one 12288-row gate at M = 96 /
// 128 on 128 x 64 KS2 33.1 / 33.9 us; the Q6_K LM head at M = 32 414 -> 320 us).  At M <= 64
// the 64 x 64 tile splits K over 4 wave groups while its tiles stay within 256, else over 2.
//
// 256 x 96 against 256 x 128: per workgroup a 96-column step takes 0.84 of a 128-column one
// (timing harness, Q4_K M = 2048: 1.008 against 1.196 us per step), so the narrower tile wins
// where its extra workgroups still fit the rounds of the wider one: C4 at M = 512 and C5's gate
// + up at M = 256 (192 -> 256 workgroups, one round): 70.9 -> 64.9 us and 71.1 -> 64.6 us; Q6_K
// and Q8_0 at C4 M = 512 88.4 -> 79.9 and 79.2 -> 67.0 us; at M = 2048 (three rounds against
// four) the 128-column tile stays (229.7 against 257.4 us).
//
// (With x by LDS DMA in the 256 x 128 tile too its steps came down, Q4_K 4096 x 4096 at M = 2048
// from 1.25 to 1.20 us; the lines between the tiles stay where they were.)
//
// 256 x 192 (x by LDS DMA, ping-pong waves) steps take 1.3 of a 256 x 128 step and 1.5 of a
// 256 x 96 one (Q4_K, timing harness: 1.50-1.54 against 1.12 and 0.97-0.99 us per step at
// M = 1024 / 2048) for 1.5 and 2 times their columns; it wins where it needs fewer rounds: C4 at
// M = 2048 214.7 (256 x 128) -> 192.6 us, M = 1024 124.6 (256 x 96) -> 98.3 us, and at M = 1536
// (two rounds, the second half full, against three of 256 x 96) 200.2 -> 185.6 us; at M = 512
// (half a round) it takes 84 us against 63 on 256 x 96.
int wide_tile(const GemmGroupArgs& a) {
  const auto rounds = [&](int tile) { return (tile_count(a, kTiles[tile]) + 255) / 256; };
  const long cost0 = rounds(0) * 119, cost8 = rounds(8) * 99;  // rounds x step time (10 ns)
  const long cost9 = valid_plan(a, kDmaTile, 1) ? rounds(kDmaTile) * 145 : cost0 + 1;
  if (cost9 < cost0 && cost9 < cost8) return kDmaTile;
  return rounds(8) * 84 < rounds(0) * 100 ? 8 : 0;
}

// uneven: wave groups may take unequal shares of K.
int base_tile(const GemmGroupArgs& a, bool uneven = false) {
  const int steps = a.k / pipe::BK;  // even (whole 32-element block pairs or super-blocks)
  const int units = steps / (block32(a.type) ? 2 : 4);
  const bool ks2 = uneven ? units >= 2 : steps % 8 == 0, ks4 = uneven ? units >= 4 : steps % 16 == 0;
  if (a.m > 128 && tile_count(a, kTiles[0]) >= kMinBlocks) return wide_tile(a);
  if (a.m > 64) {
    const long wide = tile_count(a, kTiles[1]);
    if (wide >= 512) return 1;
    if (wide >= kMinBlocks) return ks2 ? 4 : 1;
    if (a.m <= 128 && tile_count(a, kTiles[2]) >= kMinBlocks) return ks2 ? 5 : 2;
  }
  if (ks4 && (a.m > 64 || tile_count(a, kTiles[3]) < 256)) return 7;
  if (ks2) return 6;
  if (tile_count(a, kTiles[2]) >= kMinBlocks) return 2;
  return 3;
}

}  // namespace

GemmPlan plan_gemm_group(const GemmGroupArgs& a, size_t workspace_bytes) {
  GemmPlan plan{base_tile(a), 1};
  if (!pipe_type(a.type)) return plan;
  // M <= 64 with every N <= 4096 (where one matrix alone takes the small-M kernel): 64 x 64
  // tiles with K over four wave groups, split across workgroups while the grid stays within
  // 256 workgroups and each split keeps >= 16 steps; taken when that grid reaches 128
  // workgroups, else each matrix keeps its small-M launch.  Timing harness at M = 32: q + k + v
  // (4096, 1024, 1024) x 4096 Q4_K 41.2 -> 16.5 us with 2 splits, down 4096 x 12288 Q4_K 40.7 ->
  // 22.5 us with 4, Q6_K 44.3 -> 34.5, Q8_0 37.7 -> 30.9, o 4096 x 4096 15.0 -> 13.6.
  bool narrow = a.m <= kSkinnyMaxM;
  for (int i = 0; i < a.count; ++i) narrow = narrow && a.n[i] <= 4096;
  if (narrow) {
    const long tiles = tile_count(a, kTiles[7]);
    int splits = 1;
    while (tiles * splits * 2 <= 256 && valid_plan(a, 7, splits * 2) && a.k / pipe::BK / (splits * 2) >= 16 &&
           (size_t)splits * 2 * a.m * total_columns(a) * sizeof(float) <= workspace_bytes)
      splits *= 2;
    if (valid_plan(a, 7, splits) && tiles * splits >= 128) return GemmPlan{7, splits, true};
    return plan;
  }
  // Split K across workgroups with the 256 x 128 tile when that tile alone leaves most CUs
  // idle and the small tiles are no better: when even 64 x 64 tiles need more than one round
  // of 256 workgroups, or K is long (>= 8192).  Measured at M = 256 (q + k + v grouped 68 ->
  // 34 us with 4 splits, the Q6_K down 4096 x 12288 90 -> 54 us with 8); the 4096 x 4096 o
  // projection stays on 64 x 64 tiles (25 us against 30 split).  From M = 65 (timing harness,
  // M = 96 / 128 / 160): the down 4096 x 12288 Q6_K 96 / 95 / 93 -> 46 / 48 / 50 us with 8
  // splits, Q8_0 85 / 89 / 85 -> 46 / 48 / 49, Q4_K 55 / 55 / 56 -> 40 / 41 / 43; q + k + v at
  // M = 160 40 -> 31 with 4.  Splits double while the grid stays within 256 workgroups and each
  // split keeps >= 8 steps (512 of K).
  const long tiles = tile_count(a, kTiles[0]);
  const bool big_tile = plan.tile != 3 && plan.tile != 6 && plan.tile != 7;  // already fills the CUs
  const bool crowded = tile_count(a, kTiles[3]) > 256 || a.k >= 8192;
  if (a.m <= kSkinnyMaxM || big_tile || !crowded) return plan;
  int splits = 1;
  while (tiles * splits * 2 <= 256 && valid_plan(a, 0, splits * 2) && a.k / pipe::BK / (splits * 2) >= 8 &&
         (size_t)splits * 2 * a.m * total_columns(a) * sizeof(float) <= workspace_bytes)
    splits *= 2;
  if (splits > 1) plan = GemmPlan{0, splits};
  return plan;
}

size_t gemm_group_workspace(const GemmGroupArgs& a, const GemmPlan& plan) {
  return plan.splits > 1 ? (size_t)plan.splits * a.m * total_columns(a) * sizeof(float) : 0;
}

hipError_t launch_gemm_group_plan(const GemmGroupArgs& a, const GemmPlan& plan, void* workspace,
                                  size_t workspace_bytes, hipStream_t stream) {
  if (!gemm_group_pipelined(a, plan) || a.count < 1 || a.count > kGemmGroupMax ||
      gemm_group_workspace(a, plan) > workspace_bytes || (plan.splits > 1 && !workspace))
    return hipErrorInvalidValue;
  switch (a.type) {
    case kQ4_K: return launch_typed<kQ4_K>(a, plan.tile, plan.splits, workspace, stream);
    case kQ5_K: return launch_typed<kQ5_K>(a, plan.tile, plan.splits, workspace, stream);
    case kQ6_K: return launch_typed<kQ6_K>(a, plan.tile, plan.splits, workspace, stream);
    case kQ8_0: return launch_typed<kQ8_0>(a, plan.tile, plan.splits, workspace, stream);
    default: return launch_typed<kQ4_0>(a, plan.tile, plan.splits, workspace, stream);
  }
}

bool gemm_tile_geometry(int tile, int* bm, int* bn, int* ks) {
  if (tile < 0 || tile >= kTileCount) return false;
  *bm = kTiles[tile].bm;
  *bn = kTiles[tile].bn;
  *ks = kTiles[tile].ks;
  return true;
}

bool gemm_group_pipelined(const GemmGroupArgs& a, const GemmPlan& plan) {
  return pipe_type(a.type) && valid_plan(a, plan.tile, plan.splits);
}

GemmGroupArgs gemm_single(const GemvArgs& a) {
  GemmGroupArgs g{};
  g.x = a.x;
  g.w[0] = a.w;
  g.out[0] = a.out;
  g.n[0] = a.n;
  g.count = 1;
  g.type = a.type;
  g.m = a.m;
  g.k = a.k;
  g.out_half = a.out_half;
  g.x_f32 = a.x_f32;
  return g;
}

hipError_t launch_gemm_pipe_config(const GemvArgs& a, hipStream_t stream, int config) {
  if (a.x_f32 || !pipe_type(a.type)) return hipErrorInvalidValue;
  return launch_gemm_group_plan(gemm_single(a), GemmPlan{config, 1}, nullptr, 0, stream);
}

// Q4_1, Q5_0, Q5_1, Q2_K and Q3_K with fp16 x, on the tile an unsplit plan would take: no K split across
// workgroups, so they need no workspace and no scratch.  Against the generic kernel (gemm_v2: one
// register set, per-element decoder; graph replays): 4096 x 4096 at M = 128 / 333 / 1024 Q3_K 147 / 157
// / 142 -> 32 / 63 / 71 us, Q5_0 158 / 154 / 136 -> 30 / 59 / 63; 12288 x 4096 at M = 512 Q4_1 146 -> 70,
// Q2_K 154 -> 73; 640 x 2560 at M = 333 Q5_1 85 -> 22.
bool gemm_more_type(int type) {
  return type == kQ4_1 || type == kQ5_0 || type == kQ5_1 || type == kQ2_K || type == kQ3_K;
}

// No plan names their tiles, so the wave groups of a workgroup may share K unevenly, which K = 2560 (40
// steps) and 6912 (108) otherwise rule out.  Q3_K at M = 333 on 64 x 64 tiles: 2560 x 6912 94 us in one
// group -> 56 in four, 2560 x 2560 24.3 in two -> 22.9 in four.
bool gemm_group_more(const GemmGroupArgs& a) {
  return gemm_more_type(a.type) && !a.x_f32 && valid_plan(a, 3, 1);  // base_tile picks no more groups than K has units
}

hipError_t launch_gemm_group_more(const GemmGroupArgs& a, hipStream_t stream) {
  if (!gemm_group_more(a) || a.count < 1 || a.count > kGemmGroupMax) return hipErrorInvalidValue;
  return launch_gemm_pipe_more(a, base_tile(a, true), stream);
}

bool gemm_pipe_supported(const GemvArgs& a) {
  const GemmGroupArgs g = gemm_single(a);
  return gemm_group_pipelined(g, plan_gemm_group(g, 0)) || gemm_group_more(g);
}

hipError_t launch_gemm_pipe(const GemvArgs& a, hipStream_t stream, bool* handled) {
  const GemmGroupArgs g = gemm_single(a);
  const GemmPlan plan = plan_gemm_group(g, 0);
  if (gemm_group_more(g)) {
    *handled = true;
    return launch_gemm_group_more(g, stream);
  }
  *handled = gemm_group_pipelined(g, plan);
  if (!*handled) return hipSuccess;
  return launch_gemm_group_plan(g, plan, nullptr, 0, stream);
}

}  // namespace tensor_gguf
