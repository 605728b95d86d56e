// A Mixture-of-Experts block over a prompt (or a batch of sequences), gfx950: every token through the experts it is
// routed to, four launches whatever the number of experts, nothing read back to the host.
//
// KernelQuantExperts.forward walks the experts one at a time for more than a few tokens
// (llmquant/quantizers/kernel.py:216-289): per expert a nonzero / where on the routing mask (which the host waits
// for), a gather of its rows, two projections, an index_add. For 300 tokens through 64 experts of 2048 x 1024 that is
// 1180 launches and 7.7 ms around 0.2 GB of int4 codes.
// Here:
//   plan + prepare  one launch: a workgroup counts the rows of every expert and lists the row tiles (runs of up to BM
//                   rows of one expert); the other workgroups put the tokens' rows in the tiled GEMM's prepared form
//   gate|up         wq_gemm_a16_tile_kernel, GROUPED: a tile's rows are gathered by the transfers into LDS
//                   (row -> token), its weight is its expert's; stores silu(gate) * up as the next GEMM's prepared rows
//   down            the same kernel on those rows (now contiguous per expert)
//   combine         per token, its rows times their routing weights, in the order of the experts
// with the rounding points of the per-expert form: gate and up, silu(gate), silu(gate) * up, the down projection, each
// weighted row and each partial sum are rounded to the activation dtype.
//
// Bound: the experts' codes (64 x 2048 x 1024 int4: 201 MB) for up to about 40 rows an expert, the tiled GEMM's rate
// beyond. Measured, 64 experts, 8 a token, 2048 x 1024, bf16, us a pass, per-expert loop -> here: 300 tokens int4
// 6970 -> 100; by kernel trace (with the profiler's overhead, medians of 24) at 12 / 60 / 300 / 600 tokens int4 the gate|up
// GEMM takes 33 / 36 / 59 / 97 us (at 12 tokens 51 experts have rows: 3.2 TB/s of their codes; at 600 79 to 108: the clock),
// down 18.6 / 20 / 33 / 51, the plan 4.8 / 4.9 / 5.2 / 9.2, the combination 4.7 / 4.7 / 5.6 / 8.9.
#include "wq_gemm_a16_tile.h"

namespace {

constexpr int kPlanThreads = 512;
constexpr int kMaxExperts = 1024;
constexpr int kMaxTopK = 256;

// The shapes: 256 columns (128 gate + 128 up rows of the weight make a whole group of the next reduction axis), rows by
// what an expert gets. Two workgroups a CU where their stages fit (int4), so that one's first transfers and store run
// under the other's multiplications: a tile is only 8 to 16 groups long here.
using Rows32 = Shape<32, 8, 1, 2, true>;
using Rows64 = Shape<64, 8, 1, 2, true>;
using Rows32Whole = Shape<32, 8, 1, 1, true>;
using Rows64Whole = Shape<64, 8, 1, 1, true>;

struct PlanArgs {
  const int64_t* expert_of_row;   // [n_rows] (token-major: row i is of token i / top_k)
  int n_rows, n_experts, top_k, tile_rows;
  int4* tiles;
  int* n_tiles;
  int* row_source;                // [n_rows]: sorted row -> token
  int* sorted_of_row;             // [n_rows]: row -> sorted row
};

__device__ __forceinline__ int expert_id(int64_t raw, int n_experts) {
  // an id outside the layer's experts is planned with the nearest valid one; the combination makes its token's row NaN
  return raw < 0 ? 0 : (raw >= n_experts ? n_experts - 1 : static_cast<int>(raw));
}

// Block 0: the plan. Where a row lands inside its expert's run depends on the order of the atomics; nothing downstream
// does: a row's result does not depend on its neighbours, and the combination goes by expert and slot.
// Other blocks: x -> prepared form, a lane per 16-byte chunk (act_prep_kernel's work).
template <typename T>
__global__ __launch_bounds__(kPlanThreads) void experts_plan_kernel(const PlanArgs p, const u32x4* __restrict__ x,
                                                                    u32x4* __restrict__ xp, u32x4* __restrict__ rec,
                                                                    const int64_t n_chunks) {
  const int tid = threadIdx.x;
  if (blockIdx.x > 0) {
    const int64_t i = static_cast<int64_t>(blockIdx.x - 1) * kPlanThreads + tid;
    const bool active = i < n_chunks;  // n_chunks is a multiple of 16: a row of 16 lanes is active or idle as one
    u32x4 v = {0u, 0u, 0u, 0u};
    if (active) v = x[i];
    emit_prepared<T>(v, active, (tid & 15) == 0, xp + (active ? i : 0), rec + (active ? i >> 4 : 0));
    return;
  }
  // (each id is read once, all of a thread's in flight together, and stays in a register with the row's place inside its
  // expert's run, which is what the counting atomic returns. Bound: the chain ids -> counts -> scan -> places of one
  // workgroup. Read twice and placed by further atomics, 2400 rows took 5.6 us a launch by kernel trace; this 5.0, 320 rows
  // 2.8 at best. Past kKept rows a thread the places wait in sorted_of_row.)
  constexpr int kKept = 10;
  __shared__ int s_count[kMaxExperts], s_first[kMaxExperts];
  int expert[kKept], place[kKept];
#pragma unroll
  for (int k = 0; k < kKept; ++k) {
    const int i = k * kPlanThreads + tid;
    expert[k] = i < p.n_rows ? expert_id(p.expert_of_row[i], p.n_experts) : -1;
  }
  for (int e = tid; e < p.n_experts; e += kPlanThreads) s_count[e] = 0;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < kKept; ++k) place[k] = expert[k] >= 0 ? atomicAdd(&s_count[expert[k]], 1) : 0;
  for (int i = kKept * kPlanThreads + tid; i < p.n_rows; i += kPlanThreads) {
    p.sorted_of_row[i] = atomicAdd(&s_count[expert_id(p.expert_of_row[i], p.n_experts)], 1);
  }
  __syncthreads();
  if (tid < kWave) {
    // exclusive prefix sums of rows and of row tiles: a lane takes `per` experts in a row, then a scan over the lanes
    const int per = (p.n_experts + kWave - 1) / kWave;
    int rows = 0, tiles = 0;
    for (int k = 0; k < per; ++k) {
      const int e = tid * per + k;
      if (e < p.n_experts) rows += s_count[e], tiles += (s_count[e] + p.tile_rows - 1) / p.tile_rows;
    }
    int row_end = rows, tile_end = tiles;
#pragma unroll
    for (int step = 1; step < kWave; step <<= 1) {
      const int r = __shfl_up(row_end, step), t = __shfl_up(tile_end, step);
      if (tid >= step) row_end += r, tile_end += t;
    }
    int row = row_end - rows, tile = tile_end - tiles;
    for (int k = 0; k < per; ++k) {
      const int e = tid * per + k;
      if (e < p.n_experts) {
        const int count = s_count[e];
        s_first[e] = row;
        for (int done = 0; done < count; done += p.tile_rows, ++tile) {
          p.tiles[tile] = int4{e, row + done, min(p.tile_rows, count - done), 0};
        }
        row += count;
      }
    }
    if (tid == kWave - 1) *p.n_tiles = tile_end;
  }
  __syncthreads();
  auto put = [&](int i, int at) {
    p.row_source[at] = i / p.top_k;
    p.sorted_of_row[i] = at;
  };
#pragma unroll
  for (int k = 0; k < kKept; ++k) {
    if (expert[k] >= 0) put(k * kPlanThreads + tid, s_first[expert[k]] + place[k]);
  }
  for (int i = kKept * kPlanThreads + tid; i < p.n_rows; i += kPlanThreads) {
    put(i, s_first[expert_id(p.expert_of_row[i], p.n_experts)] + p.sorted_of_row[i]);   // (its own store of above)
  }
}

// final[t] = the rows of token t, each times its routing weight, added up in the order of the experts (of the slots
// where two are the same), every product and sum rounded to T. One workgroup per token, eight columns a thread and turn.
// A token with an id outside the layer's experts: a row of NaN.
template <typename T>
__global__ __launch_bounds__(256) void experts_combine_kernel(const T* __restrict__ rows_out,
                                                              const int64_t* __restrict__ expert_of_row,
                                                              const int* __restrict__ sorted_of_row,
                                                              const T* __restrict__ weights, T* __restrict__ final_out,
                                                              const int top_k, const int n_experts, const int width) {
  __shared__ int s_expert[kMaxTopK], s_row[kMaxTopK];
  __shared__ float s_weight[kMaxTopK];
  const int t = blockIdx.x, tid = threadIdx.x;
  const int64_t first = static_cast<int64_t>(t) * top_k;
  int e = 0, row = 0;
  float weight = 0.0f;
  if (tid < top_k) {   // (kMaxTopK slots, a thread each; the three loads in flight together)
    const int64_t raw = expert_of_row[first + tid];
    row = sorted_of_row[first + tid];
    weight = llmq::to_float(weights[first + tid]);
    e = expert_id(raw, n_experts);
    if (raw != e) weight = __builtin_nanf("");
    s_expert[tid] = e;
  }
  __syncthreads();
  if (tid < top_k) {
    int rank = 0;
    for (int j = 0; j < top_k; ++j) rank += s_expert[j] < e || (s_expert[j] == e && j < tid);
    s_row[rank] = row;
    s_weight[rank] = weight;
  }
  __syncthreads();
  // eight rows' packets in flight at a time (one after the other a trip to memory each: 300 tokens of 2048 values through
  // eight experts each 6.2 us by kernel trace, this 5.5; with the plan above, a call of 40 tokens 66.7 -> 64.1 us, of 300
  // 108.8 -> 105.7, of 600 138.3 -> 134.8)
  constexpr int kAhead = 8;
  for (int c = tid * 8; c < width; c += 256 * 8) {
    float acc[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int k0 = 0; k0 < top_k; k0 += kAhead) {
      u32x4 packet[kAhead] = {};
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        if (k0 + k < top_k) packet[k] = load16(rows_out + static_cast<int64_t>(s_row[k0 + k]) * width + c);
      }
#pragma unroll
      for (int k = 0; k < kAhead; ++k) {
        if (k0 + k >= top_k) break;
        float v[8];
        Pack<T>::unpack(packet[k], v);
        const float w = s_weight[k0 + k];
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] = round_through<T>(acc[i] + round_through<T>(v[i] * w));
      }
    }
    store16(final_out + static_cast<int64_t>(t) * width + c, Pack<T>::pack(acc));
  }
}

size_t aligned(size_t bytes) { return (bytes + 255) / 256 * 256; }

struct Layout {
  size_t xp, rec, act_xp, act_rec, rows_out, tiles, n_tiles, row_source, sorted, total;
};

Layout layout_for(int T, int top_k, int E, int H, int I) {
  const size_t rows = static_cast<size_t>(T) * top_k;
  const size_t max_tiles = rows / 32 + (rows < static_cast<size_t>(E) ? rows : E) + 1;   // (of the smallest tile)
  Layout l{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += aligned(bytes);
    return here;
  };
  l.xp = take(static_cast<size_t>(T) * H * 2);
  l.rec = take(static_cast<size_t>(T) * (H / kGroup) * 16);
  l.act_xp = take(rows * I * 2);
  l.act_rec = take(rows * (I / kGroup) * 16);
  l.rows_out = take(rows * H * 2);
  l.tiles = take(max_tiles * sizeof(int4));
  l.n_tiles = take(sizeof(int));
  l.row_source = take(rows * sizeof(int));
  l.sorted = take(rows * sizeof(int));
  l.total = at;
  return l;
}

template <typename T, int BITS, int EPI, typename S>
int launch_grouped(const TileArgs& a, int max_row_tiles, hipStream_t stream) {
  auto kernel = wq_gemm_a16_tile_kernel<T, BITS, EPI, S, true>;
  constexpr int kLds = S::template kLdsBytes<BITS>;
  static bool raised = false;  // per instantiation; worst case two threads both set it
  if (!raised) {
    const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (err != hipSuccess) {
      llmq_host::set_error("raising the LDS limit failed: %s", hipGetErrorString(err));
      return static_cast<int>(err);
    }
    raised = true;
  }
  const int work = max_row_tiles * a.n_tiles;
  hipLaunchKernelGGL(kernel, dim3((work + 7) / 8 * 8), dim3(S::kThreads), kLds, stream, a);
  return llmq_host::check_launch("wq_gemm_a16_tile_kernel (grouped)");
}

template <typename T, int BITS, typename S>
int run_shape(const TileArgs& gate_up, const TileArgs& down, int max_row_tiles, hipStream_t stream) {
  if (int rc = launch_grouped<T, BITS, kEpiGateUpSilu, S>(gate_up, max_row_tiles, stream)) return rc;
  return launch_grouped<T, BITS, kEpiStore, S>(down, max_row_tiles, stream);
}

// Rows of a tile: 32 or 64. The host does not know the experts' counts; an expert's last tile is about half full, so that
// there are some rows / height + 0.45 E row tiles (no fewer than experts with rows), each with I / 128 column tiles of H / 128
// groups in the gate|up launch and H / 256 of I / 128 in the down launch. A launch's time goes by rounds of one workgroup a CU: one
// that does not fill the chip takes part of a round, one that is just begun a quarter; a round of 64-row tiles takes 1.5 (int8
// 1.46) of 32-row ones. Measured, both heights, 968 problems in graphs (bf16, routers without and with favourites; 4 to 128 experts, H
// from 0.3 I to 32 I, 4 to 200 rows an expert), us a call, 32 / 64 rows: 64 experts of 2048 x 1024 int4 at 10 rows an expert
// 65 / 74, 30: 86 / 96, 37.5: 96 / 100, 75: 143 / 130, 200: 285 / 243; int8 30: 119 / 134, 37.5: 140 / 136, 52: 169 / 145; eight of
// 2048 x 4096 int4 at 45: 67 / 79, 64: 78 / 85, 130: 118 / 106, int8 45: 94 / 103, 52: 109 / 104, 130: 187 / 136; eight of 4096 x
// 14336 int8 37.5: 489 / 395; forty of 1024 x 512 int8 30: 32 / 36, 45: 47 / 37, 75: 50 / 59; 64 of 7168 x 256 int8 45: 158 / 164,
// 64: 228 / 179. Of the 448 that the figures were fitted to, the height taken is 0.3 % (int8 0.6) behind the better one on average,
// 16 % (13) at worst (sixteen of 6144 x 1024 int4, 52: 92 / 106; 32 of 2048 x 2048 int8, 16: 117 / 104); of the 520 others 0.7
// (1.1) and 16 % (35, a round begun by a few tiles more than were reckoned with). By the gate|up launch's rounds alone 0.9 (1.4) and 15 %
// (30), 1.3 (2.4) and 16 % (40); by a line at 40 rows an expert 2.9 (2.3) and 22 % (30), 2.6 (3.6) and 40 % (47).
int tile_rows_for(int rows, int E, int H, int I, bool int4) {
  const double hit = rows < E ? rows : E, least = int4 ? 0.5 : 0.25;
  auto rounds = [&](double tiles) {
    const double all = tiles / 256.0, whole = static_cast<int64_t>(all);
    if (all <= 1.0) return least + (1.0 - least) * all;
    return all > whole ? whole + 0.25 + 0.75 * (all - whole) : whole;
  };
  auto cost = [&](int height) {
    const double by_rows = static_cast<double>(rows) / height + 0.45 * E, row_tiles = by_rows > hit ? by_rows : hit;
    return rounds(row_tiles * (I / kGroup)) * (H / kGroup) + rounds(row_tiles * ((H + 255) / 256)) * (I / kGroup);
  };
  return (int4 ? 1.5 : 1.46) * cost(64) < cost(32) ? 64 : 32;
}

template <typename T, int BITS>
int run(const void* x, const int64_t* index, const void* weights, const void* q1, const float* s1, const void* q2,
        const float* s2, void* out, uint8_t* ws, int n_tokens, int top_k, int E, int H, int I, hipStream_t stream) {
  const Layout l = layout_for(n_tokens, top_k, E, H, I);
  const int rows = n_tokens * top_k;
  const int tile_rows = tile_rows_for(rows, E, H, I, BITS == 4);
  const PlanArgs p{index, rows, E, top_k, tile_rows, reinterpret_cast<int4*>(ws + l.tiles),
                   reinterpret_cast<int*>(ws + l.n_tiles), reinterpret_cast<int*>(ws + l.row_source),
                   reinterpret_cast<int*>(ws + l.sorted)};
  const int64_t n_chunks = static_cast<int64_t>(n_tokens) * (H / 8);
  const dim3 plan_grid(1 + static_cast<unsigned>((n_chunks + kPlanThreads - 1) / kPlanThreads));
  hipLaunchKernelGGL(experts_plan_kernel<T>, plan_grid, dim3(kPlanThreads), 0, stream, p, static_cast<const u32x4*>(x),
                     reinterpret_cast<u32x4*>(ws + l.xp), reinterpret_cast<u32x4*>(ws + l.rec), n_chunks);
  if (int rc = llmq_host::check_launch("experts_plan_kernel")) return rc;

  const int g1 = H / kGroup, g2 = I / kGroup;
  TileArgs up{};
  up.xp = ws + l.xp, up.rec = ws + l.rec, up.qw = static_cast<const uint8_t*>(q1), up.sw = s1;
  up.M = rows, up.N = 2 * I, up.G = g1, up.n_tiles = I / 128, up.splits = 1, up.groups_per_split = g1;
  up.next_xp = ws + l.act_xp, up.next_rec = ws + l.act_rec, up.next_G = g2;
  up.tiles = p.tiles, up.n_row_tiles = p.n_tiles, up.row_source = p.row_source;
  up.expert_codes = static_cast<int64_t>(2) * I * H * BITS / 8, up.expert_scales = static_cast<int64_t>(2) * I * g1;
  TileArgs down{};
  down.xp = ws + l.act_xp, down.rec = ws + l.act_rec, down.qw = static_cast<const uint8_t*>(q2), down.sw = s2;
  down.out = ws + l.rows_out;
  down.M = rows, down.N = H, down.G = g2, down.n_tiles = (H + 255) / 256, down.splits = 1, down.groups_per_split = g2;
  down.tiles = p.tiles, down.n_row_tiles = p.n_tiles;
  down.expert_codes = static_cast<int64_t>(H) * I * BITS / 8, down.expert_scales = static_cast<int64_t>(H) * g2;
  const int max_row_tiles = rows / tile_rows + (rows < E ? rows : E);
  int rc;
  if constexpr (BITS == 4) {
    rc = tile_rows == 32 ? run_shape<T, BITS, Rows32>(up, down, max_row_tiles, stream)
                         : run_shape<T, BITS, Rows64>(up, down, max_row_tiles, stream);
  } else {
    rc = tile_rows == 32 ? run_shape<T, BITS, Rows32Whole>(up, down, max_row_tiles, stream)
                         : run_shape<T, BITS, Rows64Whole>(up, down, max_row_tiles, stream);
  }
  if (rc) return rc;
  hipLaunchKernelGGL(experts_combine_kernel<T>, dim3(n_tokens), dim3(256), 0, stream,
                     reinterpret_cast<const T*>(ws + l.rows_out), index, p.sorted_of_row, static_cast<const T*>(weights),
                     static_cast<T*>(out), top_k, E, H);
  return llmq_host::check_launch("experts_combine_kernel");
}

}  // namespace

extern "C" int llmq_wq_experts_supported(int n_tokens, int top_k, int n_experts, int hidden, int intermediate) {
  if (n_tokens < 1 || top_k < 1 || top_k > kMaxTopK || n_experts < 1 || n_experts > kMaxExperts) return 0;
  if (hidden < kGroup || intermediate < kGroup || hidden % kGroup || intermediate % kGroup) return 0;
  // the GEMMs' 32-bit offsets: an activation, and one expert's weight
  const uint64_t rows = static_cast<uint64_t>(n_tokens) * top_k, limit = 1ull << 32;
  const uint64_t wide = hidden > intermediate ? hidden : intermediate;
  if (rows * wide * 2 >= limit || rows > (1u << 24) || 2ull * hidden * intermediate >= limit) return 0;
  return 1;
}

extern "C" size_t llmq_wq_experts_workspace_bytes(int n_tokens, int top_k, int n_experts, int hidden, int intermediate) {
  if (!llmq_wq_experts_supported(n_tokens, top_k, n_experts, hidden, intermediate)) return 0;
  return layout_for(n_tokens, top_k, n_experts, hidden, intermediate).total;
}

extern "C" int llmq_wq_experts_tile_rows(int n_tokens, int top_k, int n_experts, int hidden, int intermediate, int wformat) {
  if (!llmq_wq_experts_supported(n_tokens, top_k, n_experts, hidden, intermediate)) return 0;
  return tile_rows_for(n_tokens * top_k, n_experts, hidden, intermediate, wformat == LLMQ_W_INT4_PACKED);
}

extern "C" int llmq_wq_experts(const void* x, const int64_t* top_k_index, const void* top_k_weights,
                               const void* gate_up, const float* gate_up_scale, const void* down,
                               const float* down_scale, void* out, void* workspace, size_t workspace_bytes,
                               int n_tokens, int top_k, int n_experts, int hidden, int intermediate, int wformat,
                               int dtype, llmq_stream_t stream) {
  if (n_tokens == 0) return 0;
  if (!llmq_wq_experts_supported(n_tokens, top_k, n_experts, hidden, intermediate))
    return llmq_host::fail_invalid("the experts' GEMM does not take tokens=%d top_k=%d experts=%d hidden=%d intermediate=%d",
                                   n_tokens, top_k, n_experts, hidden, intermediate);
  if (wformat != LLMQ_W_INT8 && wformat != LLMQ_W_INT4_PACKED)
    return llmq_host::fail_invalid("unsupported weight format %d, expected 8 or 4", wformat);
  if (dtype != LLMQ_BF16 && dtype != LLMQ_F16)
    return llmq_host::fail_invalid("the experts' GEMM takes bfloat16 or float16 activations, got dtype code %d", dtype);
  if (!x || !top_k_index || !top_k_weights || !gate_up || !gate_up_scale || !down || !down_scale || !out || !workspace)
    return llmq_host::fail_invalid("null tensor pointer");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(gate_up) | reinterpret_cast<uintptr_t>(down) |
       reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(workspace)) & 15u)
    return llmq_host::fail_invalid("activation, weight, output and workspace pointers must be 16-byte aligned");
  const size_t need = layout_for(n_tokens, top_k, n_experts, hidden, intermediate).total;
  if (workspace_bytes < need)
    return llmq_host::fail_invalid("workspace of %zu bytes is too small, need %zu", workspace_bytes, need);
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const bool int4 = wformat == LLMQ_W_INT4_PACKED;
#define LLMQ_EXPERTS(T, BITS)                                                                                      \
  run<T, BITS>(x, top_k_index, top_k_weights, gate_up, gate_up_scale, down, down_scale, out, ws, n_tokens, top_k, \
               n_experts, hidden, intermediate, s)
  if (dtype == LLMQ_BF16) return int4 ? LLMQ_EXPERTS(bf16_t, 4) : LLMQ_EXPERTS(bf16_t, 8);
  return int4 ? LLMQ_EXPERTS(f16_t, 4) : LLMQ_EXPERTS(f16_t, 8);
#undef LLMQ_EXPERTS
}
