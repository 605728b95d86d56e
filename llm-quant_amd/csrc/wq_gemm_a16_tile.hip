// The tiled weight-only GEMM: launches and plans. The kernel, its tile shapes and the prepared form of an activation are
// in wq_gemm_a16_tile.h (shared with the routed experts' GEMM, wq_gemm_experts.hip).
#include <stdlib.h>

#include "wq_gemm_a16_tile.h"

namespace {

// out[i] = bf16(partial[0][i] + partial[1][i] + ...), slices added in order; four values per lane.
template <typename T>
__global__ __launch_bounds__(256) void add_splits_kernel(const float* __restrict__ partial, T* __restrict__ out,
                                                         const int64_t count, const int splits) {
  const int64_t i4 = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
  if (i4 >= count) return;
  if (i4 + 4 <= count && (count & 3) == 0) {
    u32x4 v = load16(partial + i4);
    float s[4];
    Pack<float>::unpack(v, s);
    for (int k = 1; k < splits; ++k) {
      float t[4];
      Pack<float>::unpack(load16(partial + k * count + i4), t);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = s[e] + t[e];
    }
    *reinterpret_cast<u32x2*>(out + i4) =
        u32x2{static_cast<uint32_t>(bits16<T>(s[0])) | static_cast<uint32_t>(bits16<T>(s[1])) << 16,
              static_cast<uint32_t>(bits16<T>(s[2])) | static_cast<uint32_t>(bits16<T>(s[3])) << 16};
  } else {
    // a count that is not a multiple of four leaves the later slices off 16-byte alignment: this lane's own
    // (up to) four values one at a time
    const int64_t end = i4 + 4 < count ? i4 + 4 : count;
    for (int64_t i = i4; i < end; ++i) {
      float s = partial[i];
      for (int k = 1; k < splits; ++k) s = s + partial[k * count + i];
      out[i] = from_float<T>(s);
    }
  }
}

template <typename T, int BITS, int EPI, typename S = Wide>
int launch_tiles(const TileArgs& a, dim3 grid, hipStream_t stream) {
  auto kernel = wq_gemm_a16_tile_kernel<T, BITS, EPI, S>;
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
  hipLaunchKernelGGL(kernel, grid, dim3(S::kThreads), kLds, stream, a);
  return llmq_host::check_launch("wq_gemm_a16_tile_kernel");
}

constexpr size_t kAlign = 256;
size_t aligned(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

struct Plan {
  int m_tiles, n_tiles, splits, groups_per_split;
  size_t xp_bytes, rec_bytes, partial_bytes;
};

// LLMQ_A16_TILE=wide / narrow in the environment pins the tile shape whatever the problem (read per call; the
// tests run shapes through both).
int forced_shape() {
  const char* v = getenv("LLMQ_A16_TILE");
  if (v == nullptr) return 0;
  return v[0] == 'w' ? 1 : (v[0] == 'n' ? 2 : 0);
}

Plan plan_for(int M, int N, int G, bool narrow = false) {
  Plan p{};
  p.m_tiles = narrow ? (M + Narrow::kBM - 1) / Narrow::kBM : (M + kBM - 1) / kBM;
  p.n_tiles = narrow ? (N + Narrow::kBN - 1) / Narrow::kBN : (N + kBN - 1) / kBN;
  const int tiles = p.m_tiles * p.n_tiles;
  // fewer tiles than would occupy most CUs: cut the reduction axis, at least four groups per slice and no more
  // workgroups than CUs (a workgroup has a CU's LDS to itself: one over is a second round)
  int splits = 1;
  if (tiles < 160) {
    splits = 256 / tiles;
    if (splits > G / 4) splits = G / 4;
    if (splits < 1) splits = 1;
  }
  p.groups_per_split = (G + splits - 1) / splits;
  p.splits = (G + p.groups_per_split - 1) / p.groups_per_split;  // every slice holds at least one group
  // (rows padded to whole wide tiles, which covers whole narrow ones: the kernel reads them without clamping; what
  // the pad rows hold is never stored)
  const size_t padded_rows = static_cast<size_t>((M + kBM - 1) / kBM) * kBM;
  p.xp_bytes = aligned(padded_rows * G * kRowBytes);
  p.rec_bytes = aligned(padded_rows * G * 16);
  p.partial_bytes = p.splits > 1 ? aligned(static_cast<size_t>(p.splits) * M * N * sizeof(float)) : 0;
  return p;
}

// What a plan costs, in microseconds, from the measured shape of a launch: rounds of 256 workgroups, each a fixed
// part (first transfers from memory, the store) plus a time per group of the reduction axis (wide 8 + 1.93 / 2.1 a
// group for int4 / int8, narrow 6 + 0.75 / 1.0), and where the axis is cut the partial tiles' way through memory
// and the second launch (3 us + 8 bytes per partial value at 9 TB/s: most of it overlaps the tiles). The figures are of
// the kernel whose loop went a k-step at a time; the present one is faster and they were not fitted again: over 420
// problems (72 to 1024 rows, weights of 512 to 28672 rows of 16 to 112 groups) the cheaper plan's estimate with the
// preparation is 0.84 to 1.39 times the measured launch, 1.05 in the middle, half of them 1.00 to 1.11; the other width would
// be faster by 0.3 % on average.
double plan_cost(const Plan& p, int M, int N, bool narrow, bool int4) {
  const double fixed = narrow ? 6.0 : 8.0;
  const double per_group = narrow ? (int4 ? 0.75 : 1.0) : (int4 ? 1.93 : 2.1);
  const int workgroups = p.m_tiles * p.n_tiles * p.splits;
  const double rounds = static_cast<double>((workgroups + 255) / 256);
  double cost = rounds * (fixed + p.groups_per_split * per_group);
  if (p.splits > 1) cost += 3.0 + static_cast<double>(p.splits) * M * N * 8.0 / 9.0e6;
  return cost;
}

// Whether the 64 x 128 tile is the faster one: outputs of few 128 x 256 tiles, where the narrow tile fills the
// chip without cutting the reduction axis (512 x 3072 x 2048 int8: 24.4 us against 29.3; 128 x 14336 x 4096 int4:
// 31.7 / 36.4), and not where its tiles need a second round (1024 x 3072 x 2048: 42.6 / 33.0) or the rows are long
// enough for the wide tile's slices to pay for their partial sums (512 x 4096 x 4096: 41.2 / 37.2).
bool narrow_tile(int M, int N, int G, bool int4) {
  const int forced = forced_shape();
  if (forced) return forced == 2;
  return plan_cost(plan_for(M, N, G, true), M, N, true, int4) < plan_cost(plan_for(M, N, G, false), M, N, false, int4);
}

}  // namespace

extern "C" size_t llmq_wq_gemm_a16_tile_workspace_bytes(int M, int N, int G) {
  if (M <= 0 || N <= 0 || G <= 0) return 0;
  // (the larger of the two shapes' needs: the shape is chosen per call, and may be pinned from the environment)
  const Plan w = plan_for(M, N, G, false), n = plan_for(M, N, G, true);
  return w.xp_bytes + w.rec_bytes + (w.partial_bytes > n.partial_bytes ? w.partial_bytes : n.partial_bytes);
}

namespace {

// The checks the three entry points share; `x` is null when the activation is already prepared.
int check_common(const void* x, bool prepared, const void* qweight, const float* wscale, const void* workspace, int M,
                 int N, int G, int gs, int out_group, int wformat, int dtype) {
  if (M < 0 || N < 0 || G < 0) return llmq_host::fail_invalid("negative dimension M=%d N=%d G=%d", M, N, G);
  if (gs != kGroup) return llmq_host::fail_invalid("the tiled fused GEMM needs group_size 128, got %d", gs);
  if (dtype != LLMQ_BF16 && dtype != LLMQ_F16)
    return llmq_host::fail_invalid("the tiled fused GEMM takes bfloat16 or float16 activations, got dtype code %d", dtype);
  if (wformat != LLMQ_W_INT8 && wformat != LLMQ_W_INT4_PACKED)
    return llmq_host::fail_invalid("unsupported weight format %d, expected 8 or 4", wformat);
  if (out_group < 0) return llmq_host::fail_invalid("out_group must be >= 0, got %d", out_group);
  if (M == 0 || N == 0) return 0;
  if (G == 0) return llmq_host::fail_invalid("a weight with no groups has no reduction axis");
  if ((!prepared && !x) || !qweight || !wscale || !workspace) return llmq_host::fail_invalid("null tensor pointer");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(qweight) | reinterpret_cast<uintptr_t>(workspace)) & 15u)
    return llmq_host::fail_invalid("activation, weight, output and workspace pointers must be 16-byte aligned");
  if ((static_cast<uint64_t>(M) + kBM) * G * kRowBytes >= (1ull << 32))
    return llmq_host::fail_invalid("activation of %d x %d values is beyond the kernel's 32-bit offsets", M, G * kGroup);
  if (static_cast<uint64_t>(N) * G * kGroup >= (1ull << 32))
    return llmq_host::fail_invalid("weight of %d x %d codes is beyond the kernel's 32-bit offsets", N, G * kGroup);
  return 0;
}

int prepare(const void* x, uint8_t* xp, uint8_t* rec, int M, int G, hipStream_t s) {
  const int64_t n_chunks = static_cast<int64_t>(M) * G * 16;
  hipLaunchKernelGGL(act_prep_kernel<bf16_t>, dim3(static_cast<unsigned>((n_chunks + 255) / 256)), dim3(256), 0, s,
                     static_cast<const u32x4*>(x), reinterpret_cast<u32x4*>(xp), reinterpret_cast<u32x4*>(rec), n_chunks);
  return llmq_host::check_launch("act_prep_kernel");
}

// The kernel for a weight format, an epilogue and a tile shape, by activation dtype.
template <int EPI, typename S>
int launch_by_type(const TileArgs& a, dim3 grid, int wformat, int dtype, hipStream_t s) {
  const bool int4 = wformat == LLMQ_W_INT4_PACKED;
  if (dtype == LLMQ_BF16) return int4 ? launch_tiles<bf16_t, 4, EPI, S>(a, grid, s) : launch_tiles<bf16_t, 8, EPI, S>(a, grid, s);
  return int4 ? launch_tiles<f16_t, 4, EPI, S>(a, grid, s) : launch_tiles<f16_t, 8, EPI, S>(a, grid, s);
}

// x (or, x null, the prepared activation already in the workspace) times the weight, into out.
int run_store(const void* x, const void* qweight, const float* wscale, void* out, void* workspace,
              size_t workspace_bytes, int M, int N, int G, int gs, int out_group, int wformat, int dtype,
              hipStream_t s) {
  if (int rc = check_common(x, x == nullptr, qweight, wscale, workspace, M, N, G, gs, out_group, wformat, dtype)) return rc;
  if (M == 0 || N == 0) return 0;
  if (!out || (reinterpret_cast<uintptr_t>(out) & 15u)) return llmq_host::fail_invalid("out must be a 16-byte aligned pointer");
  const bool narrow = narrow_tile(M, N, G, wformat == LLMQ_W_INT4_PACKED);
  const Plan p = plan_for(M, N, G, narrow);
  if (workspace_bytes < p.xp_bytes + p.rec_bytes + p.partial_bytes)
    return llmq_host::fail_invalid("workspace of %zu bytes is too small, need %zu", workspace_bytes,
                                   p.xp_bytes + p.rec_bytes + p.partial_bytes);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const uint8_t* xp = ws;
  uint8_t* rec = ws + p.xp_bytes;
  float* partial = reinterpret_cast<float*>(ws + p.xp_bytes + p.rec_bytes);
  if (x != nullptr && dtype == LLMQ_F16) {
    xp = static_cast<const uint8_t*>(x);   // (read as it lies)
  } else if (x != nullptr) {
    if (int rc = prepare(x, ws, rec, M, G, s)) return rc;
  }
  TileArgs a{xp, rec, static_cast<const uint8_t*>(qweight), wscale, out, partial, M, N, G, out_group,
             p.m_tiles, p.n_tiles, p.splits, p.groups_per_split, nullptr, nullptr, 0};
  const int total = p.m_tiles * p.n_tiles * p.splits;
  const dim3 grid(static_cast<unsigned>((total + 7) / 8 * 8));
  const int rc = narrow ? launch_by_type<kEpiStore, Narrow>(a, grid, wformat, dtype, s)
                        : launch_by_type<kEpiStore, Wide>(a, grid, wformat, dtype, s);
  if (rc) return rc;
  if (p.splits > 1) {
    const int64_t count = static_cast<int64_t>(M) * N;
    const dim3 add_grid(static_cast<unsigned>((count / 4 + 256) / 256));
    if (dtype == LLMQ_BF16) {
      hipLaunchKernelGGL(add_splits_kernel<bf16_t>, add_grid, dim3(256), 0, s, partial, static_cast<bf16_t*>(out), count, p.splits);
    } else {
      hipLaunchKernelGGL(add_splits_kernel<f16_t>, add_grid, dim3(256), 0, s, partial, static_cast<f16_t*>(out), count, p.splits);
    }
    return llmq_host::check_launch("add_splits_kernel");
  }
  return 0;
}

}  // namespace

extern "C" int llmq_wq_gemm_a16_tile(const void* x, const void* qweight, const float* wscale, void* out,
                                     void* workspace, size_t workspace_bytes, int M, int N, int G, int gs,
                                     int out_group, int wformat, int dtype, llmq_stream_t stream) {
  if (M > 0 && N > 0 && !x) return llmq_host::fail_invalid("null tensor pointer");
  return run_store(x, qweight, wscale, out, workspace, workspace_bytes, M, N, G, gs, out_group, wformat, dtype,
                   static_cast<hipStream_t>(stream));
}

extern "C" int llmq_wq_gemm_a16_tile_prepared(const void* qweight, const float* wscale, void* out, void* workspace,
                                              size_t workspace_bytes, int M, int N, int G, int gs, int out_group,
                                              int wformat, int dtype, llmq_stream_t stream) {
  return run_store(nullptr, qweight, wscale, out, workspace, workspace_bytes, M, N, G, gs, out_group, wformat, dtype,
                   static_cast<hipStream_t>(stream));
}

extern "C" size_t llmq_wq_gemm_a16_tile_prepared_bytes(int M, int G) {
  if (M <= 0 || G <= 0) return 0;
  const Plan p = plan_for(M, kBN, G);   // (the prepared part of the workspace does not depend on N)
  return p.xp_bytes + p.rec_bytes;
}

namespace {

// x null: the activation is already in `workspace` in prepared form.
int run_gate_up_silu(const void* x, const void* qweight, const float* wscale, void* workspace, size_t workspace_bytes,
                     void* next_workspace, size_t next_workspace_bytes, int M, int I, int G, int gs, int out_group,
                     int wformat, int dtype, llmq_stream_t stream) {
  if (I < 0 || I > (1 << 29)) return llmq_host::fail_invalid("bad intermediate size %d", I);
  if (int rc = check_common(x, x == nullptr, qweight, wscale, workspace, M, 2 * I, G, gs, out_group, wformat, dtype)) return rc;
  if (M == 0 || I == 0) return 0;
  if (I % (kBN / 2)) return llmq_host::fail_invalid("the intermediate size must be a multiple of %d, got %d", kBN / 2, I);
  if (!next_workspace || (reinterpret_cast<uintptr_t>(next_workspace) & 15u))
    return llmq_host::fail_invalid("next_workspace must be a 16-byte aligned pointer");
  const int next_G = I / kGroup;
  Plan p = plan_for(M, 2 * I, G);
  const Plan next = plan_for(M, kBN, next_G);
  if (workspace_bytes < p.xp_bytes + p.rec_bytes)
    return llmq_host::fail_invalid("workspace of %zu bytes is too small, need %zu", workspace_bytes, p.xp_bytes + p.rec_bytes);
  if (next_workspace_bytes < next.xp_bytes + next.rec_bytes)
    return llmq_host::fail_invalid("next_workspace of %zu bytes is too small, need %zu", next_workspace_bytes,
                                   next.xp_bytes + next.rec_bytes);
  if ((static_cast<uint64_t>(M) + kBM) * next_G * kRowBytes >= (1ull << 32))
    return llmq_host::fail_invalid("activation of %d x %d values is beyond the next GEMM's 32-bit offsets", M, I);
  hipStream_t s = static_cast<hipStream_t>(stream);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  const uint8_t* xp = ws;
  uint8_t* rec = ws + p.xp_bytes;
  if (x != nullptr && dtype == LLMQ_F16) {
    xp = static_cast<const uint8_t*>(x);   // (read as it lies)
  } else if (x != nullptr) {
    if (int rc = prepare(x, ws, rec, M, G, s)) return rc;
  }
  uint8_t* nws = static_cast<uint8_t*>(next_workspace);
  // whole reduction axis per workgroup: a tile's epilogue needs its finished totals
  TileArgs a{xp, rec, static_cast<const uint8_t*>(qweight), wscale, nullptr, nullptr, M, 2 * I, G, out_group,
             p.m_tiles, I / (kBN / 2), 1, G, nws, nws + next.xp_bytes, next_G};
  const int total = a.m_tiles * a.n_tiles;
  const dim3 grid(static_cast<unsigned>((total + 7) / 8 * 8));
  return launch_by_type<kEpiGateUpSilu, Wide>(a, grid, wformat, dtype, s);
}

}  // namespace

extern "C" int llmq_wq_gemm_a16_tile_gate_up_silu(const void* x, const void* qweight, const float* wscale,
                                                  void* workspace, size_t workspace_bytes, void* next_workspace,
                                                  size_t next_workspace_bytes, int M, int I, int G, int gs,
                                                  int out_group, int wformat, int dtype, llmq_stream_t stream) {
  if (M > 0 && I > 0 && !x) return llmq_host::fail_invalid("null tensor pointer");
  return run_gate_up_silu(x, qweight, wscale, workspace, workspace_bytes, next_workspace, next_workspace_bytes, M, I,
                          G, gs, out_group, wformat, dtype, stream);
}

extern "C" int llmq_wq_gemm_a16_tile_gate_up_silu_prepared(const void* qweight, const float* wscale, void* workspace,
                                                           size_t workspace_bytes, void* next_workspace,
                                                           size_t next_workspace_bytes, int M, int I, int G, int gs,
                                                           int out_group, int wformat, int dtype,
                                                           llmq_stream_t stream) {
  return run_gate_up_silu(nullptr, qweight, wscale, workspace, workspace_bytes, next_workspace, next_workspace_bytes,
                          M, I, G, gs, out_group, wformat, dtype, stream);
}

extern "C" int llmq_add_rmsnorm_prepared(const void* x, const void* delta_or_null, const void* weight,
                                         void* sum_out_or_null, void* workspace, size_t workspace_bytes, int rows,
                                         int hidden, float eps, int dtype, llmq_stream_t stream) {
  if (rows < 0 || hidden <= 0) return llmq_host::fail_invalid("bad dimension rows=%d hidden=%d", rows, hidden);
  if (dtype != LLMQ_BF16 && dtype != LLMQ_F16)
    return llmq_host::fail_invalid("the prepared form is of bfloat16 or float16 activations, got dtype code %d", dtype);
  if (hidden % kGroup) return llmq_host::fail_invalid("hidden must be a multiple of %d, got %d", kGroup, hidden);
  if (rows == 0) return 0;
  if (!x || !weight || !workspace) return llmq_host::fail_invalid("null tensor pointer");
  if ((delta_or_null == nullptr) != (sum_out_or_null == nullptr))
    return llmq_host::fail_invalid("delta and sum_out go together");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(weight) | reinterpret_cast<uintptr_t>(workspace) |
       reinterpret_cast<uintptr_t>(delta_or_null) | reinterpret_cast<uintptr_t>(sum_out_or_null)) & 15u)
    return llmq_host::fail_invalid("tensors and the workspace must be 16-byte aligned");
  const int G = hidden / kGroup;
  if ((static_cast<uint64_t>(rows) + kBM) * G * kRowBytes >= (1ull << 32))
    return llmq_host::fail_invalid("activation of %d x %d values is beyond the tiled GEMM's 32-bit offsets", rows, hidden);
  const Plan p = plan_for(rows, kBN, G);
  if (workspace_bytes < p.xp_bytes + p.rec_bytes)
    return llmq_host::fail_invalid("workspace of %zu bytes is too small, need %zu", workspace_bytes, p.xp_bytes + p.rec_bytes);
  uint8_t* ws = static_cast<uint8_t*>(workspace);
  hipStream_t s = static_cast<hipStream_t>(stream);
  u32x4* xp = reinterpret_cast<u32x4*>(ws);
  u32x4* rec = reinterpret_cast<u32x4*>(ws + p.xp_bytes);
#define LLMQ_NORM_PREP(T, ADD)                                                                                      \
  hipLaunchKernelGGL((rmsnorm_prep_kernel<T, ADD>), dim3(rows), dim3(kNormThreads), 0, s, static_cast<const T*>(x), \
                     static_cast<const T*>(delta_or_null), static_cast<const T*>(weight),                           \
                     static_cast<T*>(sum_out_or_null), xp, rec, hidden, eps)
  if (dtype == LLMQ_BF16) {
    if (delta_or_null) LLMQ_NORM_PREP(bf16_t, true); else LLMQ_NORM_PREP(bf16_t, false);
  } else {
    if (delta_or_null) LLMQ_NORM_PREP(f16_t, true); else LLMQ_NORM_PREP(f16_t, false);
  }
#undef LLMQ_NORM_PREP
  return llmq_host::check_launch("rmsnorm_prep_kernel");
}
