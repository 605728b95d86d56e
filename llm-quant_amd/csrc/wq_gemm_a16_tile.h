// Weight-only quantized GEMM for prompt-sized activations (M in the hundreds and thousands), gfx950:
// bf16 (or fp16) activations times int4 / int8 group-quantized weights on the 16-bit matrix core, with no dense
// copy of the weight anywhere. The text below describes the bf16 form; what differs for fp16 is said at kBiased.
//
//   out[m, n] = sum over g of  wscale[sr(n), g] * sum_k x[m, g*128 + k] * code[n, g, k]
//
// the weight-only branch of RealQuantLinear.forward (llmquant/quantizers/real.py:84-91): products of a
// bf16 value and a small integer are exact in fp32, the matrix core adds them in fp32, and the scale is
// applied once per group. (The reference's kernel mode dequantizes the whole weight to the activation
// dtype and calls the BLAS library for M > 4, llmquant/quantizers/kernel.py:68-79,88-91: nine times the
// int4 codes' bytes through HBM per call, and a second rounding per weight.)
//
// Shape. A workgroup of eight waves (two per SIMD) owns a 128 (m) x 256 (n) tile of the output; every wave owns
// 32 of the 256 columns and all 128 rows: 4 x 1 MFMA tiles of 32 x 32 (v_mfma_f32_32x32x16_bf16), eight
// k-steps of 16 per group. A lane converts the codes of one column only, and each converted operand feeds four
// MFMAs (with 64 x 64 per wave two waves converted the same codes: measured 3-4 % slower on the large shapes).
// Everything reaches LDS straight from global memory (buffer loads into LDS, 1 KB per wave instruction,
// XOR-swizzled by row so that the operand reads are conflict-free), three stages deep for int4, two for int8:
// the activation tile, the raw codes of the 256 weight rows, the activation-sum records and the group's scales.
// The workgroup meets once per group, when its last operands are in registers, and the next group's are read from LDS
// behind that barrier.
// What bounds it: issue, and power. Per group a wave issues 36 multiplications of 32 cycles (float16 32), 128 to 160 vector
// instructions of conversion and folding, 39 LDS reads, and the two waves of a SIMD share one matrix core: 2300 cycles if it never
// waited, 3100 measured (float16 3020), 224 workgroups. What counts is how evenly the rest lies between the multiplications: a
// step that carries more than six vector instructions is longer than its multiplication (independent multiplications on two
// waves a SIMD, cycles each with 0 / 4 / 6 / 8 / 12 / 16 vector instructions behind it: 33 / 35 / 35 / 44 / 56 / 67). Folds and
// conversions eight to sixteen a step and none elsewhere: 3316 (3190). Without folds 2460, without conversions 3100 (float16 2730),
// without transfers 2990 at a clock 10 to 17 % higher: on random codes the chip holds 1.6 to 1.9 GHz under this loop, on zeros 2.2,
// so that a cycle saved is half a cycle's time. Launches of 512 x 14336 x 4096 int4 us, the lumped loop / this, in turn on one
// card: bf16 with its preparation 77.7 / 75.4 (another card 72.5), fp16 68.8 / 66.6; 333 x 4096 x 14336 fp16 63.6 / 61.0 (another
// 56.2); 36 problems of both widths 2 % in the middle, 0 to 6. Launches of few narrow
// tiles on short rows pay 0.1 to 0.2 us for the result's way through LDS.
//
// Codes become bf16 without a conversion instruction: a nibble n = code + 8 placed in the mantissa of
// 16.0 (bits 0x4180 | n << 3) IS the bf16 value 16 + n, two nibbles per AND-OR (int8: code + 128 through
// v_cvt_f32_ubyte, whose upper half is the bf16 value). The matrix core therefore sums x * (code + B),
// B = 24 or 128, and B * sum_k x is taken out again per group by one more k-step in front of the eight: the
// group's activation sum, cut into three bf16 pieces, against the constant -B. The fp32 group sum is then
// folded into the fp32 total with one multiply-add by the group's weight scale.
//
// A bfloat16 activation is prepared once per call by act_prep_kernel: rows padded to whole tiles, within every
// 16-byte chunk the eight values reordered to (0, 4, 1, 5, 2, 6, 3, 7), the order in which the AND-OR above
// leaves the codes (a sum does not care about the order of its terms, as long as both operands agree), and
// the per-group sums written as records of bf16 pieces.
//
// Small N: a split of the reduction axis across workgroups, fp32 partial tiles in a workspace, added in a
// fixed order by a second launch (the result does not depend on which workgroup finished first).
#pragma once

#include <type_traits>

#include "llmq_device.h"

namespace {

using namespace llmq;

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));

// bfloat16: the matrix core sums x * (code + B) and B * sum x is taken out again (below). float16 has the mantissa
// to hold B + code as well, but the pieces of a group's activation sum do not fit its exponent range (128 values of
// up to 65504, and pieces of a small sum fall below its smallest step), so there the bias is taken off the
// operand itself, exactly, with one packed instruction per two codes, and there is no correction step (operand_words).
template <typename T> constexpr bool kBiased = std::is_same<T, bf16_t>::value;
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kGroup = 128;
constexpr int kRowBytes = kGroup * 2;          // one activation row of one group
template <int BITS> constexpr int kCodeRowBytes = BITS == 4 ? kGroup / 2 : kGroup;

// The workgroup's tile: BM activation rows x 32 COLS weight rows; a wave owns 32 of the columns, all the rows and
// one KH-th of every group's k-steps. Wide (128 x 256, eight waves, two per SIMD) is the throughput shape. Narrow
// (64 x 128) is for outputs that have too few wide tiles to occupy the chip (a 512-token prompt against a 3072-row
// weight: 48 wide tiles, 192 narrow ones): its eight waves are four column blocks times two halves of the group
// (still two waves per SIMD, so that one converts codes while the other multiplies), the halves' totals are added
// through LDS once, at the end, and the smaller stages leave LDS for four of them in flight. WGS: workgroups that
// share a CU (their stages share its LDS).
// CHUNK (the grouped tiles): four groups' scales at a time, see below.
template <int BM, int COLS, int KH, int WGS = 1, bool CHUNK = false> struct Shape {
  static constexpr bool kChunk = CHUNK;
  static constexpr int kBM = BM;                 // activation rows per workgroup
  static constexpr int kWaveM = BM;              // ... and per wave
  static constexpr int kWaveN = 32;              // weight rows (output columns) per wave
  static constexpr int kColWaves = COLS;         // column blocks
  static constexpr int kKH = KH;                 // waves that share a column block, each with 8 / KH k-steps of a group
  static constexpr int kWaves = COLS * KH;
  static constexpr int kBN = kWaveN * COLS;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kTileBytes = BM * kRowBytes;
  static constexpr int kMT = BM / 32, kNT = kWaveN / 32;
  static constexpr int kRecWaves = BM < 64 ? 1 : BM / 64;   // waves that fetch the activation-sum records (64 rows each)
  static constexpr int kRecTileBytes = kRecWaves * 64 * 16;
  static constexpr int kScaleTileBytes = CHUNK ? 0 : kBN * 4;         // (of a stage)
  static constexpr int kChunks = CHUNK ? (BM >= 64 ? 2 : 1) : 0;      // (beside the stages)
  static constexpr int kChunkBytes = kChunks * kBN * 16;
  static constexpr int kScaleWaves = CHUNK ? 0 : kBN / 64;   // ... and, after them, the scales (64 columns each)
  template <int BITS> static constexpr int kCodeTileBytes = kBN * kCodeRowBytes<BITS>;
  template <int BITS>
  static constexpr int kStageBytes = kTileBytes + kCodeTileBytes<BITS> + kRecTileBytes + kScaleTileBytes;
  // as many stages as fit the 160 KB of LDS, at most four: a group's transfers are requested kStages - 1 groups
  // before it is multiplied (wide: three for int4, 153 KB, two for int8; narrow: four)
  static constexpr int kWavesPerSimd = (kWaves * WGS + 3) / 4;
  template <int BITS>
  static constexpr int kFitting = (160 * 1024 / WGS - kChunkBytes) / kStageBytes<BITS>;
  template <int BITS> static constexpr int kStages = kFitting<BITS> >= 4 ? 4 : kFitting<BITS>;
  template <int BITS> static constexpr int kLdsBytes = kStages<BITS> * kStageBytes<BITS> + kChunkBytes;
  static constexpr bool kRowBlocks = kMT * KH == 4;   // the loop of wide and narrow tiles (the kernel's main loop has two forms)
};
using Wide = Shape<128, 8, 1>;
using Narrow = Shape<64, 4, 2>;
// (what the host side sizes for when it does not say which: the wide tile)
constexpr int kBM = Wide::kBM, kBN = Wide::kBN;


// ---- activation preparation -----------------------------------------------------------------------
// One lane per 16-byte chunk, 16 lanes per (row, group): `v` holds the chunk's eight bf16 values (zeros in a lane
// with nothing to do; a row of 16 lanes is active or idle as one). Writes the reordered chunk, and from the row's
// first lane the record of the group's sum.
template <typename T>
__device__ __forceinline__ void emit_prepared(const u32x4 v, const bool active, const bool first_of_row,
                                              u32x4* __restrict__ chunk_out, u32x4* __restrict__ record_out) {
  if constexpr (!kBiased<T>) {
    // (the operands are in the chunk's own order, and without a correction step the records, which stay part of the
    // layout, are read by nobody: a float16 activation in rows of its own needs no preparation)
    if (!active) return;
    *chunk_out = v;
    if (first_of_row) *record_out = u32x4{0u, 0u, 0u, 0u};
    return;
  }
  float f[8];
  Pack<bf16_t>::unpack(v, f);
  float s = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
  s = row16_sum(s);
  if (!active) return;
  // (x0 x1)(x2 x3)(x4 x5)(x6 x7) -> (x0 x4)(x1 x5)(x2 x6)(x3 x7)
  u32x4 o;
  o.x = __builtin_amdgcn_perm(v.z, v.x, 0x05040100u);
  o.y = __builtin_amdgcn_perm(v.z, v.x, 0x07060302u);
  o.z = __builtin_amdgcn_perm(v.w, v.y, 0x05040100u);
  o.w = __builtin_amdgcn_perm(v.w, v.y, 0x07060302u);
  *chunk_out = o;
  if (first_of_row) {
    // s = hi + mid + lo, each a bf16: 24 bits of the sum
    const uint32_t hi = bf16_bits_rne(s);
    const float r1 = s - __builtin_bit_cast(float, hi << 16);
    const uint32_t mid = bf16_bits_rne(r1);
    const float r2 = r1 - __builtin_bit_cast(float, mid << 16);
    const uint32_t lo = bf16_bits_rne(r2);
    *record_out = u32x4{hi | (mid << 16), lo, 0u, 0u};  // k' slots 0..2 of the correction step
  }
}

template <typename T>
__global__ __launch_bounds__(256) void act_prep_kernel(const u32x4* __restrict__ x, u32x4* __restrict__ xp,
                                                       u32x4* __restrict__ rec, const int64_t n_chunks) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const bool active = i < n_chunks;  // n_chunks is a multiple of 16: a row of 16 lanes is active or idle as one
  u32x4 v = {0u, 0u, 0u, 0u};
  if (active) v = x[i];
  emit_prepared<T>(v, active, (threadIdx.x & 15) == 0, xp + (active ? i : 0), rec + (active ? i >> 4 : 0));
}

// LlamaRMSNorm (optionally on x + delta, the residual add in front of it, which is stored as well) whose result
// goes straight into prepared form: what act_prep_kernel would make of llmq_add_rmsnorm's output, without that
// tensor and without the second launch. One workgroup per row, the arithmetic and rounding points of
// rmsnorm_kernel (csrc/prefill_ops.hip): out = w * bf16(x_f32 * rsqrt(mean(x_f32^2) + eps)), rounded to bf16.
// hidden is a multiple of 128, so the 16 lanes of a (row, group) are in the loop together.
constexpr int kNormThreads = 256;
template <typename T, bool ADD>
__global__ __launch_bounds__(kNormThreads) void rmsnorm_prep_kernel(const T* __restrict__ x,
                                                                   const T* __restrict__ delta,
                                                                   const T* __restrict__ w,
                                                                   T* __restrict__ sum_out, u32x4* __restrict__ xp,
                                                                   u32x4* __restrict__ rec, const int hidden,
                                                                   const float eps) {
  __shared__ float red[kNormThreads / kWave];
  const int64_t base = static_cast<int64_t>(blockIdx.x) * hidden;
  const T* row = x + base;
  const int tid = threadIdx.x;
  float ss = 0.0f;
  for (int i = tid * 8; i < hidden; i += kNormThreads * 8) {
    float f[8];
    Pack<T>::unpack(load16(row + i), f);
    if constexpr (ADD) {
      float d[8];
      Pack<T>::unpack(load16(delta + base + i), d);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = round_through<T>(f[e] + d[e]);
      store16(sum_out + base + i, Pack<T>::pack(f));
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) ss = fmaf(f[e], f[e], ss);
  }
  ss = wave_sum(ss);
  if ((tid & (kWave - 1)) == 0) red[tid / kWave] = ss;
  __syncthreads();
  float total = 0.0f;
#pragma unroll
  for (int k = 0; k < kNormThreads / kWave; ++k) total += red[k];
  const float inv_rms = rsqrtf(total / static_cast<float>(hidden) + eps);
  // (with ADD a thread reads back exactly the packets it stored above)
  const T* src = ADD ? sum_out + base : row;
  const int64_t chunk0 = base >> 3;   // the row's first chunk; 16 chunks a group
  for (int i = tid * 8; i < hidden; i += kNormThreads * 8) {
    float f[8], g[8];
    Pack<T>::unpack(load16(src + i), f);
    Pack<T>::unpack(load16(w + i), g);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = g[e] * round_through<T>(f[e] * inv_rms);
    const int64_t chunk = chunk0 + (i >> 3);
    emit_prepared<T>(Pack<T>::pack(f), true, (tid & 15) == 0, xp + chunk, rec + (chunk >> 4));
  }
}

struct TileArgs {
  const uint8_t* xp;   // [M, G*128] bf16, chunks reordered
  const uint8_t* rec;  // [M, G] records of 16 bytes
  const uint8_t* qw;   // [N, G, 128] int8 or [N, G, 64] packed int4
  const float* sw;     // [scale_rows, G]
  void* out;           // [M, N] bf16 (one split)
  float* partial;      // [splits][M][N] fp32 (more)
  int M, N, G, out_group;
  int m_tiles, n_tiles, splits, groups_per_split;
  // kEpiGateUpSilu: the prepared activation of the next GEMM (its xp and rec, next_G groups a row)
  uint8_t* next_xp;
  uint8_t* next_rec;
  int next_G;
  // GROUPED: the weight is a stack of experts' weights and the rows are sorted by expert. tiles[i] = (expert, first
  // sorted row, rows, -) of the i-th row tile, *n_row_tiles of them; sorted row r reads row row_source[r] of xp (null:
  // row r); sorted row r of the result goes to row r of `out` or of the next GEMM's prepared activation.
  const int4* tiles;
  const int* n_row_tiles;
  const int* row_source;
  int64_t expert_codes, expert_scales;   // bytes of codes and count of scales between two experts
};

// What a workgroup does with its totals. kEpiStore: rounds them to bf16 into out (or leaves fp32 partial tiles).
// kEpiGateUpSilu: the weight is gate_proj's rows followed by up_proj's (N = 2 I); a tile is 128 gate rows and the
// 128 up rows that belong to them, and the workgroup writes act = silu(bf16 gate) * bf16 up (the rounding points of
// `act_fn(gate) * up` on bf16 tensors) for its 128 x 128 block straight into the next GEMM's prepared activation:
// the block is one group of 128 of that activation's reduction axis, so its chunks and records are complete.
enum Epilogue { kEpiStore = 0, kEpiGateUpSilu = 1 };
constexpr int kEpiRowBytes = 128 * 2 + 16;   // a row of the gate (or up) block in LDS: 16 bytes of padding per row

// LDS, per stage: the activation tile [BM rows][16 slots of 16 bytes], the raw codes of the workgroup's weight rows
// for one group ([BN][64] bytes of int4 or [BN][128] of int8, slots XOR-swizzled by row like the activation), the
// activation-sum records and the group's scales.
// slot of chunk c in weight row `row`: 16 consecutive rows read the same chunk at once and must land in
// 16 different bank quads
template <int BITS> __device__ __forceinline__ int code_slot(int row, int c) {
  return BITS == 4 ? c ^ ((row >> 2) & 3) : c ^ ((row >> 1) & 7);
}


// The four operand words of a k-step of the wave (`raw`: its k-steps' codes one after the other, one 32-bit word
// of int4 or two of int8 a step). bfloat16: word i pairs the biased codes i and i + 4. float16: word i pairs codes 2 i and
// 2 i + 1, the order of the activation as it lies in memory, so that there nothing prepares it (333 x 14336 values: a
// launch of 5.8 us; 333 x 4096 x 14336 int4 60.7 -> 55.2 us, 200 x 4096 x 4096 23.1 -> 19.9): a byte of two nibbles goes to both halves, the even code stays where it is (1024 + n) and the odd
// one sixteen times as high (1024 + 16 n), and the multiply-add that takes the bias out brings it down, all exact.
template <typename T, int BITS>
constexpr uint32_t kOperandMagic = std::is_same<T, f16_t>::value && BITS == 4 ? 0x64006400u : BiasedCodes<T, BITS>::kMagic;
// word `i` of step `step` (int8: of codes whose sign bits are flipped already)
template <typename T, int BITS>
__device__ __forceinline__ uint32_t operand_word(const uint32_t* raw, int step, int i, uint32_t magic) {
  if constexpr (kBiased<T>) return BiasedCodes<T, BITS>::word(raw, step, i, magic);
  if constexpr (BITS == 4) {
    const uint32_t both = __builtin_amdgcn_perm(0u, raw[step], 0x0c000c00u | (i << 16) | i);
    const h2 v = __builtin_bit_cast(h2, and_or(both, 0x00f0000fu, magic));
    const h2 down = {static_cast<_Float16>(1.0f), static_cast<_Float16>(0.0625f)};
    const h2 bias = {static_cast<_Float16>(-1032.0f), static_cast<_Float16>(-72.0f)};
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, down, bias));
  } else {
    // bytes 2 i and 2 i + 1 into the two halves, in the mantissa of 256.0
    const uint32_t w = raw[2 * step + i / 2];
    const uint32_t pick = i % 2 ? 0x0c030c02u : 0x0c010c00u;
    const h2 v = __builtin_bit_cast(h2, (__builtin_amdgcn_perm(0u, w, pick) << 2) | magic);
    const h2 bias = {static_cast<_Float16>(-384.0f), static_cast<_Float16>(-384.0f)};
    return __builtin_bit_cast(uint32_t, v + bias);
  }
}
template <typename T, int BITS>
__device__ __forceinline__ u32x4 operand_words(const uint32_t* raw, int step, uint32_t magic) {
  if constexpr (kBiased<T>) return BiasedCodes<T, BITS>::operand(raw, step, magic);
  uint32_t own[BITS / 4];
#pragma unroll
  for (int i = 0; i < BITS / 4; ++i) own[i] = raw[step * (BITS / 4) + i] ^ (BITS == 8 ? 0x80808080u : 0u);
  return u32x4{operand_word<T, BITS>(own, 0, 0, magic), operand_word<T, BITS>(own, 0, 1, magic),
               operand_word<T, BITS>(own, 0, 2, magic), operand_word<T, BITS>(own, 0, 3, magic)};
}

// What the loop of row blocks puts behind which of a group's multiplications (steps): conversions of codes, word by
// word (four a k-step), and folds of finished sums, register by register (register r of row tile t: 16 t + r). As even
// as the deadlines allow: the next group's codes are there from the last block's third step on and its first operand is due two
// steps later; a row tile's sums are finished after its second block and start anew with the next group's first.
struct Run {
  int first, count;
};
template <int HALVES> struct Dealt;
// Wide: steps 4 b + j of blocks b = 0..3 (row tiles against the first four k-steps) and 4..7 (against the second four).
// Row tile t is finished after step 19 + 4 t and starts anew at step 4 t.
template <> struct Dealt<2> {
  static constexpr int kEarlyWords = 6;   // of the next group, in the last two steps
  static constexpr int kMostWords = 4, kMostFolds = 4;
  static constexpr Run words(int s) {
    if (s >= 30) return {3 * (s - 30), 3};
    if (s < 3) return {6 + 3 * s, s < 2 ? 3 : 4};
    return s >= 10 && s < 18 ? Run{16 + 2 * (s - 10), 2} : Run{0, 0};
  }
  static constexpr Run folds(int s) {
    if (s >= 21 && s < 30) return {4 * (s - 21), 4};
    return s >= 3 && s < 10 ? Run{36 + 4 * (s - 3), 4} : Run{0, 0};
  }
  static constexpr int kLateFolds = 36;   // from this one on: in the next group's steps
};
// Narrow: steps 4 b + j of two row tiles, finished after steps 3 and 7. (A k-step's codes at a time: spread over five steps as
// above, 100 x 14336 x 4096 int4 is 1 to 2 % slower.)
template <> struct Dealt<1> {
  static constexpr int kEarlyWords = 8;
  static constexpr int kMostWords = 4, kMostFolds = 6;
  static constexpr Run words(int s) {
    if (s >= 6) return {4 * (s - 6), 4};
    return s < 2 ? Run{8 + 4 * s, 4} : Run{0, 0};
  }
  static constexpr Run folds(int s) {
    const int k = s % 4;
    if (s == 0 || k == 0) return {0, 0};
    return {(s > 4 ? 0 : 16) + (k == 1 ? 0 : 1 + 5 * (k - 1)), k == 1 ? 6 : 5};
  }
  static constexpr int kLateFolds = 16;
};

// Whether the tables above deal out a group of HALVES x MT blocks of HS steps: every word and fold once, in order within a
// k-step, no more of them a step than the loop has room for; a word behind the last multiplication that reads the group's before
// and ahead of its own first, with its codes there (asked for behind the last block's first step, two steps before they
// are used) and not yet overwritten; a fold behind its tile's last multiplication and ahead of the tile's first of the next group.
template <int HALVES, int MT, int HS> constexpr bool dealt_in_time() {
  using D = Dealt<HALVES>;
  constexpr int kAll = HALVES * MT * HS, kWords = 4 * HALVES * HS, kFolds = 16 * MT, kCodes = (HALVES * MT - 1) * HS;
  int word_at[kWords] = {}, fold_at[kFolds] = {};   // (step + 1; 0: none yet)
  for (int s = 0; s < kAll; ++s) {
    const Run words = D::words(s), folds = D::folds(s);
    if (words.count > D::kMostWords || folds.count > D::kMostFolds) return false;
    for (int w = words.first; w < words.first + words.count; ++w) {
      if (w >= kWords || word_at[w] != 0) return false;
      word_at[w] = s + 1;
    }
    for (int f = folds.first; f < folds.first + folds.count; ++f) {
      if (f >= kFolds || fold_at[f] != 0) return false;
      fold_at[f] = s + 1;
    }
  }
  int before = -kAll;
  for (int w = 0; w < kWords; ++w) {
    const int s = word_at[w] - 1, block = w / 4 / HS * MT, j = w / 4 % HS;
    const bool early = w < D::kEarlyWords;   // (in the steps of the group before)
    if (s < 0 || (early ? s < kCodes + 2 : s >= kCodes)) return false;
    const int when = early ? s - kAll : s, first = block * HS + j, last = (block + MT - 1) * HS + j;
    if (when >= first || when < last - kAll || (w % 4 != 0 && when < before)) return false;
    before = when;
  }
  for (int f = 0; f < kFolds; ++f) {
    const int s = fold_at[f] - 1, tile = f / 16, done = ((HALVES - 1) * MT + tile) * HS + HS - 1;
    if (s < 0 || (f >= D::kLateFolds ? s >= tile * HS : s <= done)) return false;
  }
  return true;
}

template <typename T> __device__ __forceinline__ v16f mfma(const u32x4& a, const u32x4& b, const v16f& c) {
  if constexpr (std::is_same<T, bf16_t>::value)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(v8h, a), __builtin_bit_cast(v8h, b), c, 0, 0, 0);
}
template <typename T> __device__ __forceinline__ uint16_t bits16(float v) {
  return __builtin_bit_cast(uint16_t, from_float<T>(v));
}

template <typename T, int BITS, int EPI, typename S, bool GROUPED = false>
__global__ __launch_bounds__(S::kThreads, GROUPED ? S::kWavesPerSimd : 1) void wq_gemm_a16_tile_kernel(const TileArgs a) {
  extern __shared__ __attribute__((aligned(256))) uint8_t smem[];
  static_assert(EPI == kEpiStore || (S::kBN == 256 && S::kKH == 1), "the gate|up epilogue is laid out for 128 + 128 columns");
  constexpr int kBM = S::kBM, kBN = S::kBN, kWaveM = S::kWaveM, kWaveN = S::kWaveN, kWaves = S::kWaves;
  constexpr int kThreads = S::kThreads, kTileBytes = S::kTileBytes, kMT = S::kMT, kNT = S::kNT;
  // (float16: the records are not read)
  constexpr int kRecTileBytes = S::kRecTileBytes, kRecWaves = kBiased<T> ? S::kRecWaves : 0, kScaleWaves = S::kScaleWaves;
  constexpr int kCodeTileB = S::template kCodeTileBytes<BITS>, kStageB = S::template kStageBytes<BITS>;
  constexpr int kStagesN = S::template kStages<BITS>;
  constexpr int kKH = S::kKH, kSteps = 8 / kKH;   // k-steps of a group that one wave multiplies

  // Workgroups are dealt to the 8 XCDs round-robin by their index; a run of consecutive logical tiles
  // (the m-tiles of one n-tile first: they read the same weights) is put on one XCD, so the codes come
  // out of that XCD's L2 after the first reader.
  const int n_work = GROUPED ? *a.n_row_tiles * a.n_tiles : a.m_tiles * a.n_tiles * a.splits;
  const int per_xcd = (n_work + 7) / 8;
  const int logical = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (logical >= n_work || (GROUPED && static_cast<int>(blockIdx.x / 8) >= per_xcd)) return;
  // (GROUPED: a row tile's column tiles one after the other, its rows stay in that XCD's L2, and the next row tile is
  // the same expert's while it has more rows)
  const int mt = GROUPED ? logical / a.n_tiles : logical % a.m_tiles;
  const int nt = GROUPED ? logical % a.n_tiles : (logical / a.m_tiles) % a.n_tiles;
  const int sp = GROUPED ? 0 : logical / (a.m_tiles * a.n_tiles);
  const int4 run = GROUPED ? a.tiles[mt] : int4{0, 0, 0, 0};   // (uniform: a scalar load)
  const uint8_t* qw = a.qw + (GROUPED ? run.x * a.expert_codes : 0);
  const float* sw = a.sw + (GROUPED ? run.x * a.expert_scales : 0);

  // (the wave's index as a scalar: LDS addresses of the transfers are then scalar arithmetic into M0)
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  // every wave all the rows, 32 of the columns, and half kh of every group's k-steps (kKH == 1: all of them)
  const int wm = 0, wn = wv % S::kColWaves;
  const int kh = kKH == 1 ? 0 : __builtin_amdgcn_readfirstlane(wv / S::kColWaves);
  static_assert(kKH == 1 || (kKH == kMT && kNT == 1), "the waves of a column block keep one 32 x 32 row tile each");
  const int lm = lane & 31, lh = lane >> 5;
  // (kEpiGateUpSilu: n0 is the tile's first gate row; column c of the tile is weight row weight_row(c))
  const int m0 = GROUPED ? run.y : mt * kBM, m_end = GROUPED ? run.y + run.z : a.M;
  const int n0 = EPI == kEpiGateUpSilu ? nt * (kBN / 2) : nt * kBN;
  auto weight_row = [&](int c) {
    if constexpr (EPI == kEpiGateUpSilu) return c < kBN / 2 ? n0 + c : a.N / 2 + n0 + (c - kBN / 2);
    else return min(n0 + c, a.N - 1);
  };
  const int g_begin = sp * a.groups_per_split;
  const int g_end = min(g_begin + a.groups_per_split, a.G);

  // ---- global -> LDS: what this lane fetches for each of its wave's transfer instructions -------------
  // One instruction moves 64 x 16 bytes into 1 KB of consecutive LDS; which global chunk a lane fetches
  // for its place there carries the swizzle. The activation and its records are the kernel's own
  // buffers, padded to whole tiles of rows, so their rows need no clamping.
  // (float16: an activation may be the caller's, whose last tile of rows repeats the last row.)
  // activation: instruction i of a wave = rows wv*16 + 4 i .. + 3, lane = (row, slot); slot p of row r
  // holds chunk p ^ (r & 15), and r & 15 = 4 i + lane / 16
  constexpr int kXInstr = kBM / 4 / kWaves;  // 4
  const uint32_t x_row_bytes = static_cast<uint32_t>(a.G) * kRowBytes;
  // row `row` of the tile in the prepared activation (GROUPED: rows past the run's end repeat its last one)
  auto source_row = [&](int row) {
    if constexpr (!GROUPED) return static_cast<uint32_t>(kBiased<T> ? m0 + row : min(m0 + row, m_end - 1));
    const int r = min(m0 + row, m_end - 1);
    return static_cast<uint32_t>(a.row_source != nullptr ? a.row_source[r] : r);
  };
  uint32_t x_off[kXInstr];
#pragma unroll
  for (int i = 0; i < kXInstr; ++i) {
    const int row = wv * (kBM / kWaves) + i * 4 + (lane >> 4);
    x_off[i] = source_row(row) * x_row_bytes + (((lane & 15) ^ (row & 15)) << 4);
  }
  // codes: instructions of 16 (int4) or 8 (int8) weight rows each; kCodeInstr per wave (wide: 2 / 4), and where
  // that does not come out even, one more from each of the first kLeftCodes waves
  constexpr int kCodeInstr = kCodeTileB / 1024 / kWaves, kLeftCodes = kCodeTileB / 1024 % kWaves;
  constexpr int kRowsPerInstr = 1024 / kCodeRowBytes<BITS>;
  constexpr int kSlots = kCodeRowBytes<BITS> / 16;
  const uint32_t w_row_bytes = static_cast<uint32_t>(a.G) * kCodeRowBytes<BITS>;
  uint32_t w_off[kCodeInstr + 1];
#pragma unroll
  for (int i = 0; i < kCodeInstr + 1; ++i) {
    const int instr = i < kCodeInstr ? wv * kCodeInstr + i : kWaves * kCodeInstr + wv % (kLeftCodes ? kLeftCodes : 1);
    const int row = instr * kRowsPerInstr + lane / kSlots;
    const int chunk = code_slot<BITS>(row, lane % kSlots);  // the swizzle is its own inverse
    w_off[i] = static_cast<uint32_t>(weight_row(row)) * w_row_bytes + chunk * 16;
  }
  // One further instruction from the waves after those: the records (kRecWaves waves, 64 rows each), then the
  // scales (kScaleWaves waves, 64 columns each).
  constexpr int kExtraWaves = kLeftCodes + kRecWaves + kScaleWaves;
  static_assert(kExtraWaves <= kWaves, "at most one transfer instruction per wave beyond the even share");
  const int rec_wave = (wv + kWaves - kLeftCodes) % kWaves % (kRecWaves ? kRecWaves : 1);
  const int scale_wave = (wv + kWaves - kLeftCodes - kRecWaves) % kWaves % (kScaleWaves ? kScaleWaves : 1);
  const uint32_t r_off = source_row(rec_wave * 64 + lane) * a.G * 16;
  uint32_t s_off;
  {
    const int n = weight_row(scale_wave * 64 + lane);
    s_off = static_cast<uint32_t>(a.out_group > 0 ? n / a.out_group : n) * a.G * 4;
  }

  // Transfer instruction i of a wave for group g into stage `buf`: the activation's, the codes', and the one beyond
  // the even share.
  const BufferBase x_base = buffer_base(a.xp), w_base = buffer_base(qw), r_base = buffer_base(a.rec), s_base = buffer_base(sw);
  auto transfer = [&](int i, int g, int buf) {
    uint8_t* stage = smem + buf * kStageB;
    uint8_t* codes = stage + kTileBytes;
    if (i < kXInstr) {
      buffer_to_lds<16>(x_base, stage + (wv * (kBM / kWaves) + i * 4) * kRowBytes, x_off[i], g * kRowBytes);
    } else if (i < kXInstr + kCodeInstr) {
      const int c = i - kXInstr;
      buffer_to_lds<16>(w_base, codes + (wv * kCodeInstr + c) * 1024, w_off[c], g * kCodeRowBytes<BITS>);
    } else if (wv < kLeftCodes) {
      buffer_to_lds<16>(w_base, codes + (kWaves * kCodeInstr + wv) * 1024, w_off[kCodeInstr], g * kCodeRowBytes<BITS>);
    } else if (wv < kLeftCodes + kRecWaves) {
      buffer_to_lds<16>(r_base, codes + kCodeTileB + rec_wave * 1024, r_off, g * 16);
    } else if (wv < kExtraWaves) {
      buffer_to_lds<4>(s_base, codes + kCodeTileB + kRecTileBytes + scale_wave * 256, s_off, g * 4);   // 64 columns' scales
    }
  };
  // CHUNK: a group's scales are a cache line a column for four bytes each, as many lines looked up as the codes' and the
  // activation's together; four groups' lie side by side. An instruction brings 16 columns' (lane = column, group), two a
  // wave a chunk, asked for at the first two meetings of a chunk and due at its last. The waits do not count them: they let
  // that many fewer of the others stay in flight. The 32-row tiles have LDS for one chunk and hold a column's four scales in
  // registers, in every wave's by the time the next chunk is asked for; the 64-row tiles have no registers for them (held,
  // bfloat16 x int4 spilled seven to eight, and each reload in its group loop waited for transfers just asked for) and read a
  // group's from one of two chunks. Group by group / four at a time, us a call, weights rotated: 64 experts of 2048 x 1024
  // int4, 300 tokens 107 / 101, 40 71 / 67; eight of 2048 x 4096, 40 tokens 61.5 / 57.0; 64 rows a tile (and held): 64 experts,
  // 600 tokens 144 / 139 (154), eight, 200 tokens 81.2 / 76.1 (90.1). (An expert's weight row has a scale row of its own:
  // out_group is not looked at.)
  uint8_t* const chunks = smem + kStagesN * kStageB;
  auto chunk_of = [&](int g) { return chunks + (S::kChunks == 2 ? (g >> 2 & 1) * (kBN * 16) : 0); };
  // (the first instruction's columns lie 16 a wave in the tile's first half, the second's one half on: a scalar distance, so
  // that one lane offset serves both. Columns of the second half past the weight's end, of which nothing is stored, take the
  // first half's.)
  uint32_t c_off = 0, c_half = 0;
  if constexpr (S::kChunk) {
    const uint32_t s_row_bytes = static_cast<uint32_t>(a.G) * 4;
    c_off = static_cast<uint32_t>(n0 + wv * 16 + (lane >> 2)) * s_row_bytes;
    c_half = static_cast<uint32_t>(EPI == kEpiGateUpSilu ? a.N / 2 : (n0 + kBN / 2 < a.N ? kBN / 2 : 0)) * s_row_bytes;
  }
  auto request_scales = [&](int first_group, int part) {
    const int g = min(lane & 3, g_end - 1 - first_group);
    buffer_to_lds<4>(s_base, chunk_of(first_group) + (part * kWaves + wv) * 256, c_off + g * 4, first_group * 4 + part * c_half);
  };
  static_assert(!S::kChunk || kBN == 32 * kWaves, "two instructions a wave bring a chunk");
  static_assert(!S::kChunk || kStagesN <= 3, "a chunk's last meeting waits for what was asked for two meetings before");
  constexpr int kTransfers = kXInstr + kCodeInstr + 1;
  auto request = [&](int g, int buf) {
#pragma unroll
    for (int i = 0; i < kTransfers; ++i) transfer(i, g, buf);
  };
  // (part p of `parts` of them)
  auto request_part = [&](int g, int buf, int p, int parts) {
#pragma unroll
    for (int i = 0; i < kTransfers; ++i)
      if (i * parts / kTransfers == p) transfer(i, g, buf);
  };
  // transfer instructions per wave and group (a compile-time count per branch: the waits below name how many
  // of the youngest may still be in flight)
  constexpr int kDmaPerWave = kXInstr + kCodeInstr + 1;   // the first kExtraWaves waves; the others: one fewer

  // ---- LDS -> operands ----------------------------------------------------------------------------------
  // activation operand of k-step j, row tile mi: row mi*32 + lm, chunk (8 lh + j) ^ (lm & 15)
  // (the wave's own k-steps are kh * kSteps + j, j < kSteps: its step j is at a_base ^ (j << 4))
  const uint32_t a_base = (wm * kWaveM + lm) * kRowBytes + (((8 * lh + kh * kSteps) ^ (lm & 15)) << 4);
  // this lane's codes of a group: weight row wn*32 + lm, k in [64 lh, 64 lh + 64), of which the wave's k-steps are
  // kRawBytes bytes: the 16-byte chunks (lh kKH + kh) kRawLoads + q, at c_base ^ (q << 4), or (8 bytes) one half
  // of a chunk
  constexpr int kRawBytes = kSteps * (BITS == 4 ? 4 : 8);
  constexpr int kRawLoads = kRawBytes / 16, kRawWords = kRawBytes / 4;
  static_assert(kRawBytes == 8 || kRawBytes % 16 == 0, "a wave's codes of a group: 16-byte chunks, or half of one");
  uint32_t c_base[kNT];
#pragma unroll
  for (int ni = 0; ni < kNT; ++ni) {
    const int row = wn * kWaveN + ni * 32 + lm;
    const int first = (lh * kKH + kh) * kRawBytes;   // byte of the lane's row
    c_base[ni] = kTileBytes + row * kCodeRowBytes<BITS> + code_slot<BITS>(row, first >> 4) * 16 + (first & 15);
  }
  auto read16 = [&](const uint8_t* stage, uint32_t offset) { return *reinterpret_cast<const u32x4*>(stage + offset); };

  float total[kMT][kNT][16];
#pragma unroll
  for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
    for (int ni = 0; ni < kNT; ++ni)
#pragma unroll
      for (int r = 0; r < 16; ++r) total[mi][ni][r] = 0.0f;
  uint32_t sixteen = kOperandMagic<T, BITS>;  // 16.0 (float16: 1024.0, int8 256.0) twice; kept in a vector register (see and_or)
  asm volatile("" : "+v"(sixteen));
  const uint32_t nb = bf16_bits_rne(-BiasedCodes<T, BITS>::kBias);  // exact (read where kBiased<T> only)
  const uint32_t nb2 = (lh || kh) ? 0u : (nb | (nb << 16));   // (the correction step belongs to the group's first k-steps)
  const u32x4 bias_operand = {nb2, nb2, 0u, 0u};

  // ---- prologue: the first groups on their way, the first one's operands in registers ---------------------
  // (a stage fewer where the loop can ask for it in the first group's blocks: the first group comes sooner)
  constexpr int kFirstRequests = S::kRowBlocks && kStagesN >= 3 ? kStagesN - 1 : kStagesN;
  if constexpr (S::kChunk) {
    request_scales(g_begin, 0);
    request_scales(g_begin, 1);
  }
#pragma unroll
  for (int st = 0; st < kFirstRequests; ++st) {
    if (g_begin + st < g_end) request(g_begin + st, st);
  }
  // (the first group's transfers only, where all these batches exist: the loop waits for each later one in turn)
  if (g_end - g_begin >= kFirstRequests) {
    if (wv < kExtraWaves) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kFirstRequests - 1) * kDmaPerWave) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kFirstRequests - 1) * (kDmaPerWave - 1)) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
  __builtin_amdgcn_s_barrier();

  if constexpr (S::kRowBlocks) {
    // Blocks of one 32-row tile x half a group (narrow: x the wave's k-steps): what a lane holds is the activation
    // operands of the block being multiplied and of the next, the group's converted codes, and the sums of every tile.
    // Everything that is no multiplication is dealt out over the multiplications, a piece behind each, in this order
    // (sched_barrier: left alone the compiler gathers it): the next block's operand reads, words of codes converted ahead of
    // their use, finished sums folded into the totals (Dealt), and the transfers of the group kStages ahead.
    constexpr int kHalves = kSteps == 8 ? 2 : 1, kHS = kSteps / kHalves;   // k-steps of a block
    constexpr int kBlocks = kHalves * kMT, kLast = kBlocks - 1;
    using Deal = Dealt<kHalves>;
    static_assert(dealt_in_time<kHalves, kMT, kHS>(), "the conversions and folds of this shape");
    constexpr int kParts = kBlocks == 2 || kStagesN < 3 ? 2 : 4;   // a group's transfers in so many pieces, one a block
    u32x4 fa[2][kHS], rec_op = {0u, 0u, 0u, 0u};
    uint32_t fb[kSteps * 4];   // (words of the converted codes, four a step)
    uint32_t raw[kRawWords];
    float scale_now, scale_before = 0.0f;
    v16f acc[kMT];
#pragma unroll
    for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mi][r] = 0.0f;
    auto read_codes = [&](const uint8_t* stage) {
      if constexpr (kRawBytes == 8) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(stage + c_base[0]);
        raw[0] = v.x, raw[1] = v.y;
      } else {
#pragma unroll
        for (int q = 0; q < kRawLoads; ++q) {
          const u32x4 v = read16(stage, c_base[0] ^ (q << 4));
          raw[4 * q] = v.x, raw[4 * q + 1] = v.y, raw[4 * q + 2] = v.z, raw[4 * q + 3] = v.w;
        }
      }
    };
    auto read_scale = [&](const uint8_t* stage) {
      return *reinterpret_cast<const float*>(stage + kTileBytes + kCodeTileB + kRecTileBytes + (wn * kWaveN + lm) * 4);
    };
    auto read_rec = [&](const uint8_t* stage, int mi) {
      if constexpr (kBiased<T>) rec_op = read16(stage, kTileBytes + kCodeTileB + (mi * 32 + lm) * 16);
    };
    auto read_act = [&](const uint8_t* stage, int mi, int j) { return read16(stage, mi * 32 * kRowBytes + (a_base ^ (j << 4))); };
    auto convert = [&](int w) {   // (the words of a k-step in order)
      if (BITS == 8 && w % 4 == 0) raw[w / 2] ^= 0x80808080u, raw[w / 2 + 1] ^= 0x80808080u;
      fb[w] = operand_word<T, BITS>(raw, w / 4, w % 4, sixteen);
    };
    auto operand = [&](int step) { return u32x4{fb[4 * step], fb[4 * step + 1], fb[4 * step + 2], fb[4 * step + 3]}; };

    if (kFirstRequests < kStagesN && g_begin + kFirstRequests < g_end)
      request_part(g_begin + kFirstRequests, kFirstRequests, 0, kParts);
    read_codes(smem);
    read_rec(smem, 0);
    scale_now = read_scale(smem);
#pragma unroll
    for (int j = 0; j < kHS; ++j) fa[0][j] = read_act(smem, 0, j);
#pragma unroll
    for (int w = 0; w < 4 * kSteps; ++w) {
      if (w < Deal::kEarlyWords) convert(w);
      else fb[w] = 0u;
    }

    int st = 0, st_fill = kFirstRequests % kStagesN;  // the stage of group g; the one that transfers go to
    for (int g = g_begin; g < g_end; ++g) {
      const uint8_t* stage = smem + st * kStageB;
      const int st_next = st + 1 == kStagesN ? 0 : st + 1;
      const uint8_t* stage_next = smem + st_next * kStageB;
      float scale_next = 0.0f;
#pragma unroll
      for (int b = 0; b < kBlocks; ++b) {
        const int h = b / kMT, mi = b % kMT;
        if (b == kLast) {
          // The workgroup meets in front of the group's last block, whose operands are in registers: behind the barrier
          // this stage is free, and the next one is complete (each wave has waited for its own transfers of the next
          // group; those of later groups may stay in flight).
          if (kStagesN >= 3 && g + kStagesN - 1 < g_end) {  // (the batches of groups g + 2 .. exist and are younger)
            if (wv < kExtraWaves) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStagesN - 2) * kDmaPerWave) : "memory");
            else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStagesN - 2) * (kDmaPerWave - 1)) : "memory");
          } else {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          }
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          st_fill = st;
          __builtin_amdgcn_sched_barrier(0);
        }
        {
          // transfers into the freed stage
          const int part = b == kLast ? 0 : b + 1, g_fill = b == kLast ? g + kStagesN : g + kStagesN - 1;
          if (part < kParts && g_fill < g_end && (b == kLast || kFirstRequests < kStagesN || g > g_begin))
            request_part(g_fill, st_fill, part, kParts);
          __builtin_amdgcn_sched_barrier(0);
        }
        if (h == 0) {
          // The tile's sums start at -B * xsum[m] (one k-step: the three bf16 pieces of the activation sum against the
          // constant -B; the upper half of the wave, k' 8..15, multiplies zeros).
          const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
          acc[mi] = kBiased<T> && kh == 0 ? mfma<T>(rec_op, bias_operand, zero) : zero;
        }
#pragma unroll
        for (int j = 0; j < kHS; ++j) {
          acc[mi] = mfma<T>(fa[b & 1][j], operand(h * kHS + j), acc[mi]);
          if (b == kLast && j == 0) {
            read_codes(stage_next);   // (past the last group: whatever the stage holds, and unused)
            scale_next = read_scale(stage_next);
          }
          const int next_h = (b + 1) / kMT, next_mi = (b + 1) % kMT;
          fa[(b + 1) & 1][j] = b == kLast ? read_act(stage_next, 0, j) : read_act(stage, next_mi, next_h * kHS + j);
          if (j == 0 && b == kLast) read_rec(stage_next, 0);
          if (j == 0 && b != kLast && next_h == 0) read_rec(stage, next_mi);
          const Run words = Deal::words(b * kHS + j), folds = Deal::folds(b * kHS + j);
#pragma unroll
          for (int k = 0; k < Deal::kMostWords; ++k) {
            const int w = words.first + k;
            if (k < words.count) convert(w);
          }
#pragma unroll
          for (int k = 0; k < Deal::kMostFolds; ++k) {
            const int f = folds.first + k, tile = f / 16, r = f % 16;
            if (k < folds.count) {
              total[tile][0][r] = fmaf(f >= Deal::kLateFolds ? scale_before : scale_now, acc[tile][r], total[tile][0][r]);
              asm volatile("" : "+v"(total[tile][0][r]));   // (here, and not where the totals are next read)
            }
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      scale_before = scale_now;
      scale_now = scale_next;
      st = st_next;
    }
#pragma unroll
    for (int f = Deal::kLateFolds; f < 16 * kMT; ++f)
      total[f / 16][0][f % 16] = fmaf(scale_before, acc[f / 16][f % 16], total[f / 16][0][f % 16]);
  } else {
  // What a lane holds of the group it is about to multiply: the records (operand of the correction
  // step), its raw codes, its columns' scales and the activation operands of k-step 0.
  u32x4 rec[kMT], fa[2][kMT];
  uint32_t raw[kNT][kRawWords];
  float scale = 0.0f;
  static_assert(S::kChunk && kNT == 1, "this loop is the grouped tiles'");
  u32x4 scales = {0u, 0u, 0u, 0u};   // of this lane's column: the groups still to come of the chunk
  auto fetch_group_operands = [&](int st, int g) {
    const uint8_t* stage = smem + st * kStageB;
    if constexpr (kBiased<T>) {
#pragma unroll
      for (int mi = 0; mi < kMT; ++mi)
        rec[mi] = read16(stage, kTileBytes + kCodeTileB + (wm * kWaveM + mi * 32 + lm) * 16);
    }
#pragma unroll
    for (int ni = 0; ni < kNT; ++ni) {
      if constexpr (kRawBytes == 8) {
        const u32x2 v = *reinterpret_cast<const u32x2*>(stage + c_base[ni]);
        raw[ni][0] = v.x, raw[ni][1] = v.y;
      } else {
#pragma unroll
        for (int q = 0; q < kRawLoads; ++q) {
          const u32x4 v = read16(stage, c_base[ni] ^ (q << 4));
          raw[ni][4 * q] = v.x, raw[ni][4 * q + 1] = v.y, raw[ni][4 * q + 2] = v.z, raw[ni][4 * q + 3] = v.w;
        }
      }
    }
    if constexpr (S::kChunks == 1) {
      if ((g & 3) == 0) scales = read16(chunks, (wn * kWaveN + lm) * 16);
      scale = __builtin_bit_cast(float, scales.x);
      scales = u32x4{scales.y, scales.z, scales.w, 0u};
    }
#pragma unroll
    for (int mi = 0; mi < kMT; ++mi) fa[0][mi] = read16(stage, mi * 32 * kRowBytes + a_base);
  };
  fetch_group_operands(0, g_begin);

  // (the low tiles of the grouped GEMM, two workgroups a CU: 128 registers a lane do not hold the blocks above)
  // Two waves share a SIMD: while one converts codes or adds its group sums into the totals, the other
  // keeps the matrix core busy. Within a wave the next k-step's activation operands are requested before
  // the current step's multiplications. The workgroup meets once per group, before the last k-step: by
  // then every read of the group's LDS stage has been issued and has returned (the last step's operands are
  // in registers), so behind the barrier that stage takes the transfers of the group kStages ahead; and each
  // wave has waited, in front of the barrier, for its own transfers of the next group (requested kStages - 1
  // groups ago), so behind the barrier the next group's stage is complete: the last k-step runs while the
  // next group's operands come out of it, and no wave starts a group waiting for memory or LDS.
  int st = 0;  // the stage of group g
  for (int g = g_begin; g < g_end; ++g) {
    const uint8_t* stage = smem + st * kStageB;
    const int st_next = st + 1 == kStagesN ? 0 : st + 1;
    float scale_now = scale;

    // The group's sums start at -B * xsum[m] (one k-step: the three bf16 pieces of the activation sum
    // against the constant -B; the upper half of the wave, k' 8..15, multiplies zeros), then take the
    // eight k-steps of x * (code + B).
    v16f acc[kMT][kNT];
    {
      const v16f zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
      for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
        for (int ni = 0; ni < kNT; ++ni) acc[mi][ni] = kBiased<T> && kh == 0 ? mfma<T>(rec[mi], bias_operand, zero) : zero;
    }
#pragma unroll
    for (int j = 0; j < kSteps; ++j) {
      u32x4 fb[kNT];
#pragma unroll
      for (int ni = 0; ni < kNT; ++ni) fb[ni] = operand_words<T, BITS>(raw[ni], j, sixteen);
      if (j < kSteps - 1) {
#pragma unroll
        for (int mi = 0; mi < kMT; ++mi) fa[(j + 1) & 1][mi] = read16(stage, mi * 32 * kRowBytes + (a_base ^ ((j + 1) << 4)));
        if (S::kChunks == 2 && j == kSteps - 2)
          scale_now = *reinterpret_cast<const float*>(chunk_of(g) + (wn * kWaveN + lm) * 16 + (g & 3) * 4);
      } else {
        // own transfers of the next group have landed (the youngest kStages - 2 batches may stay in flight)
        if (kStagesN >= 3 && g + kStagesN - 1 < g_end) {  // (the batches of groups g + 2 .. exist and are younger)
          if (wv < kExtraWaves) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStagesN - 2) * kDmaPerWave) : "memory");
          else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((kStagesN - 2) * (kDmaPerWave - 1)) : "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        if (g + kStagesN < g_end) request(g + kStagesN, st);
        if ((g & 3) < 2 && (g | 3) + 1 < g_end) request_scales((g | 3) + 1, g & 3);
        if (g + 1 < g_end) fetch_group_operands(st_next, g + 1);  // (fa[0]: the last step multiplies out of fa[1])
      }
#pragma unroll
      for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
        for (int ni = 0; ni < kNT; ++ni) acc[mi][ni] = mfma<T>(fa[j & 1][mi], fb[ni], acc[mi][ni]);
    }
#pragma unroll
    for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
      for (int ni = 0; ni < kNT; ++ni)
#pragma unroll
        for (int r = 0; r < 16; ++r) total[mi][ni][r] = fmaf(scale_now, acc[mi][ni][r], total[mi][ni][r]);
    st = st_next;
  }
  }

  // ---- store: register r of a 32 x 32 tile is row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32
  if constexpr (EPI == kEpiGateUpSilu) {
    // Waves 0..3 hold the block's gate columns, 4..7 its up columns: both go to LDS as bf16 (the loop's last barrier came
    // after every wave's last operand read of a group that is multiplied; what the loop of row blocks reads behind it, of the
    // group past the last, is not used), then a lane takes a 16-byte chunk of a row at a time, 16 lanes a row, as act_prep_kernel does with a tensor in memory.
    __builtin_amdgcn_s_barrier();
    uint8_t* block = smem + (wn >> 2) * (kBM * kEpiRowBytes);
    const int col = (wn & 3) * 32 + lm;
#pragma unroll
    for (int mi = 0; mi < kMT; ++mi)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = mi * 32 + 8 * (r >> 2) + 4 * lh + (r & 3);
        *reinterpret_cast<uint16_t*>(block + row * kEpiRowBytes + col * 2) = bits16<T>(total[mi][0][r]);
      }
    __syncthreads();
    u32x4* __restrict__ next_xp = reinterpret_cast<u32x4*>(a.next_xp);
    u32x4* __restrict__ next_rec = reinterpret_cast<u32x4*>(a.next_rec);
#pragma unroll
    for (int pass = 0; pass < kBM * 16 / kThreads; ++pass) {
      const int q = pass * kThreads + tid, row = q >> 4, chunk = q & 15;
      float g[8], u[8];
      Pack<T>::unpack(read16(smem, row * kEpiRowBytes + chunk * 16), g);
      Pack<T>::unpack(read16(smem, kBM * kEpiRowBytes + row * kEpiRowBytes + chunk * 16), u);
#pragma unroll
      for (int e = 0; e < 8; ++e) g[e] = round_through<T>(g[e] / (1.0f + expf(-g[e]))) * u[e];
      if (GROUPED && m0 + row >= m_end) continue;   // (a row of 16 lanes as one)
      const int64_t at = static_cast<int64_t>(m0 + row) * a.next_G + nt;   // (row, group) of the next activation
      emit_prepared<T>(Pack<T>::pack(g), true, chunk == 0, next_xp + at * 16 + chunk, next_rec + at);
    }
    return;
  }
  // Rows that are whole 16-byte packets go out through LDS, a packet a lane and whole rows of the tile at a time
  // (two bytes a lane as they lie in the registers: 0.7 us more a tile; without any store a launch takes 4.5 us less).
  const bool whole = GROUPED || a.splits == 1;   // (not a slice of the reduction axis)
  static_assert(kBM * (kBN * 2 + 16) + (kKH > 1 ? kWaves * (kKH - 1) * 4096 : 0) <= S::template kLdsBytes<BITS>,
                "a tile of the result in the stages");
  const bool packets = whole && a.N % 8 == 0;
  constexpr int kPitch = kBN * 2 + 16;   // 16 bytes of padding: a wave's two halves in different banks
  uint8_t* const block = smem + (kKH > 1 ? kWaves * (kKH - 1) * 4096 : 0);
  // one 32 x 32 tile of totals, whose first row and column are rows / columns `row0` / `col0` of the workgroup's tile
  auto store_tile = [&](const float (&v)[16], int row0, int col0) {
    const int n = n0 + col0 + lm;
    if (packets) {
      uint8_t* to = block + (row0 + 4 * lh) * kPitch + (col0 + lm) * 2;
#pragma unroll
      for (int r = 0; r < 16; ++r) *reinterpret_cast<uint16_t*>(to + (8 * (r >> 2) + (r & 3)) * kPitch) = bits16<T>(v[r]);
    } else if (whole) {
      T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + row0 + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (m < m_end && n < a.N) out[static_cast<int64_t>(m) * a.N + n] = from_float<T>(v[r]);
      }
    } else {
      float* __restrict__ part = a.partial + static_cast<int64_t>(sp) * a.M * a.N;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int m = m0 + row0 + 8 * (r >> 2) + 4 * lh + (r & 3);
        if (m < m_end && n < a.N) part[static_cast<int64_t>(m) * a.N + n] = v[r];
      }
    }
  };
  auto store_block = [&]() {
    constexpr int kRowPackets = kBN / 8;
    T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
    for (int i = 0; i < kBM * kRowPackets / kThreads; ++i) {
      const int q = i * kThreads + tid, row = q / kRowPackets, c = q % kRowPackets, m = m0 + row, n = n0 + c * 8;
      if (m < m_end && n < a.N) store16(out + static_cast<int64_t>(m) * a.N + n, read16(block, row * kPitch + c * 16));
    }
  };
  if constexpr (kKH > 1) {
    // The kKH waves of a column block hold the totals of their parts of every group. Wave kh keeps row tile kh and
    // hands the others over through LDS (4 KB a tile, [register][lane]; the stages are free: the loop's last barrier came
    // after every wave's last transfer and its last operand read of a group that is multiplied. A slower wave may still read
    // behind it, of the group past the last, while this one writes: those values are not used), then adds the parts of its
    // tile in the order of the waves, its own in its place.
    float* exchange = reinterpret_cast<float*>(smem);
    auto slot = [&](int from, int tile) { return ((from * S::kColWaves + wn) * (kKH - 1) + (tile - (tile > from))) * 1024; };
    float own[16];
#pragma unroll
    for (int t = 0; t < kKH; ++t) {
      if (t == kh) {
#pragma unroll
        for (int r = 0; r < 16; ++r) own[r] = total[t][0][r];
      } else {
#pragma unroll
        for (int r = 0; r < 16; ++r) exchange[slot(kh, t) + r * 64 + lane] = total[t][0][r];
      }
    }
    __syncthreads();
    float sum[16];
#pragma unroll
    for (int from = 0; from < kKH; ++from) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float part = from == kh ? own[r] : exchange[slot(from, kh) + r * 64 + lane];
        sum[r] = from == 0 ? part : sum[r] + part;
      }
    }
    store_tile(sum, kh * 32, wn * kWaveN);
  } else {
    if (packets) __builtin_amdgcn_s_barrier();   // (no wave reads operands of a group that is multiplied any more)
#pragma unroll
    for (int ni = 0; ni < kNT; ++ni)
#pragma unroll
      for (int mi = 0; mi < kMT; ++mi)
        store_tile(total[mi][ni], wm * kWaveM + mi * 32, wn * kWaveN + ni * 32);
  }
  if (packets) {
    __syncthreads();
    store_block();
  }
}

}  // namespace
