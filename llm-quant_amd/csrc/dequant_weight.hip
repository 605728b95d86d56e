// Quantized weight -> dense matrix in the activation dtype, gfx950: what KernelQuantLinear
// multiplies by when more rows arrive than the GEMV takes (llmquant/quantizers/kernel.py:68-79,
// `(qweight * scale).to(dtype)`), as one pass: read the codes once, write each value once.
//
//   out[n, g * keep + k] = (dtype)(code[n, g, k] * wscale[sr(n), g])        k < keep <= group_size
//
// keep < group_size drops the zero padding of head-aligned groups (o_proj with head_dim 64 in
// groups of 128), so the dense matrix has the layer's real input width and the activation
// needs no padding either.
//
//
// A lane produces eight consecutive values per step (from 4 or 8 bytes of int4 / int8 codes) and
// stores them as one 16-byte packet (two for fp32), so a wave's store is a contiguous KiB; the write
// is four fifths of the traffic and is what has to be coalesced. Four steps are in flight per lane.
//
// What bounds it is that traffic, once the index arithmetic is out of the way: with 64-bit divisions for (row, group)
// per packet the vector ALU was the limit. The packet's group is a shift where a group is a power of two packets, the
// scale's index IS the group's where every row has scales of its own, and the rest is 32-bit (64-bit only for weights of
// more than 2^35 values). 14336 x 4096 int4 to bf16: 25.2 -> 23.4 us
// (6.3 TB/s; a large copy reaches 5.1), int8 28.5 -> 27.0, 3072 x 2048 int8 with shared scales 6.3 -> 4.7.
#include "llmq_device.h"

namespace {

using namespace llmq;

constexpr int kDqInFlight = 4;

// SHARED: out_group rows share a scale row. `shift`: log2 of a group's packets, or -1.
template <typename T, int BITS, bool SHARED, typename Index>
__global__ __launch_bounds__(256) void dequant_weight_kernel(
    const uint8_t* __restrict__ qw, const float* __restrict__ ws, T* __restrict__ out, const Index n_out_packets,
    const int G, const int gs, const int per_group, const int shift, const int out_group) {
  constexpr int V = 8;                  // values per step
  constexpr int kBytes = V * BITS / 8;  // code bytes behind them
  const Index n_threads = static_cast<Index>(gridDim.x) * 256;
  const Index group_bytes = static_cast<Index>(gs) * BITS / 8;
  // (an index past the end is never formed into an address, and p0 + 4 n_threads stays below 2^32: the host's bound)
  for (Index p0 = static_cast<Index>(blockIdx.x) * 256 + threadIdx.x; p0 < n_out_packets; p0 += kDqInFlight * n_threads) {
    uint32_t raw[kDqInFlight][kBytes / 4];
    float scale[kDqInFlight];
#pragma unroll
    for (int u = 0; u < kDqInFlight; ++u) {
      const Index p = p0 + u * n_threads;
      if (p >= n_out_packets) break;
      const Index group = shift >= 0 ? p >> shift : p / static_cast<Index>(per_group);  // n * G + g
      const Index packet = p - group * per_group;
      const uint8_t* src = qw + (static_cast<uint64_t>(group) * group_bytes + packet * kBytes);
#pragma unroll
      for (int w = 0; w < kBytes / 4; ++w) raw[u][w] = reinterpret_cast<const uint32_t*>(src)[w];
      Index at = group;
      if constexpr (SHARED) {
        const Index n = group / static_cast<Index>(G);
        at = n / static_cast<Index>(out_group) * G + (group - n * G);
      }
      scale[u] = ws[at];
    }
#pragma unroll
    for (int u = 0; u < kDqInFlight; ++u) {
      const Index p = p0 + u * n_threads;
      if (p >= n_out_packets) break;
      float f[V];
      if constexpr (BITS == 8) {
#pragma unroll
        for (int i = 0; i < V; ++i) f[i] = static_cast<float>(static_cast<int8_t>(raw[u][i / 4] >> (8 * (i % 4)))) * scale[u];
      } else {
        // nibble i of the little-endian word holds code + 8: with its top bit flipped it is the code in two's complement
        const uint32_t signs = raw[u][0] ^ 0x88888888u;
#pragma unroll
        for (int i = 0; i < V; ++i) f[i] = static_cast<float>(static_cast<int32_t>(signs << (28 - 4 * i)) >> 28) * scale[u];
      }
      T* dst = out + static_cast<uint64_t>(p) * V;
      if constexpr (Pack<T>::N == 8) {
        store16(dst, Pack<T>::pack(f));
      } else {
        store16(dst, Pack<T>::pack(f));
        store16(dst + 4, Pack<T>::pack(f + 4));
      }
    }
  }
}

// Any keep (not a multiple of the packet width): one thread per (row, group), element at a time.
template <typename T, int BITS>
__global__ __launch_bounds__(256) void dequant_weight_ragged_kernel(
    const uint8_t* __restrict__ qw, const float* __restrict__ ws, T* __restrict__ out, const int64_t n_groups,
    const int G, const int gs, const int keep, const int out_group) {
  const int64_t group = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (group >= n_groups) return;
  const int64_t n = group / G;
  const int g = static_cast<int>(group - n * G);
  const float scale = ws[(out_group > 0 ? n / out_group : n) * G + g];
  for (int k = 0; k < keep; ++k) {
    const int64_t idx = group * gs + k;
    int code;
    if constexpr (BITS == 8) {
      code = static_cast<int8_t>(qw[idx]);
    } else {
      const uint8_t byte = qw[idx >> 1];
      code = static_cast<int>((idx & 1) ? (byte >> 4) : (byte & 0xf)) - 8;
    }
    out[group * keep + k] = from_float<T>(static_cast<float>(code) * scale);
  }
}

template <typename T, int BITS>
int launch_bits(const void* qw, const float* ws, void* out, int64_t N, int G, int gs, int keep, int out_group,
                hipStream_t stream) {
  const uint8_t* q = static_cast<const uint8_t*>(qw);
  T* o = static_cast<T*>(out);
  if (keep % 8 == 0) {
    const int per_group = keep / 8;
    const int64_t n_out_packets = N * G * per_group;
    int64_t blocks = (n_out_packets + 256 * kDqInFlight - 1) / (256 * kDqInFlight);
    if (blocks > 256 * 32) blocks = 256 * 32;  // the rest is walked in stripes
    int shift = -1;
    if ((per_group & (per_group - 1)) == 0) shift = __builtin_ctz(per_group);
    const dim3 grid(static_cast<unsigned>(blocks));
    // (32-bit indices run up to n_out_packets + one stripe of four packets a thread)
    const bool narrow = n_out_packets <= 0xffffffffll - int64_t{kDqInFlight} * 256 * 256 * 32;
#define LLMQ_DEQUANT(SHARED, INDEX)                                                                                    \
  hipLaunchKernelGGL((dequant_weight_kernel<T, BITS, SHARED, INDEX>), grid, dim3(256), 0, stream, q, ws, o,             \
                     static_cast<INDEX>(n_out_packets), G, gs, per_group, shift, out_group)
    if (narrow) {
      if (out_group > 0) LLMQ_DEQUANT(true, uint32_t); else LLMQ_DEQUANT(false, uint32_t);
    } else {
      if (out_group > 0) LLMQ_DEQUANT(true, uint64_t); else LLMQ_DEQUANT(false, uint64_t);
    }
#undef LLMQ_DEQUANT
    return llmq_host::check_launch("dequant_weight_kernel");
  }
  const int64_t n_groups = N * G;
  const int64_t blocks = (n_groups + 255) / 256;
  if (blocks > 0x7fffffff) return llmq_host::fail_invalid("weight too large for one launch");
  hipLaunchKernelGGL((dequant_weight_ragged_kernel<T, BITS>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0,
                     stream, q, ws, o, n_groups, G, gs, keep, out_group);
  return llmq_host::check_launch("dequant_weight_ragged_kernel");
}

template <typename T>
int launch_typed(const void* qw, const float* ws, void* out, int64_t N, int G, int gs, int keep, int out_group,
                 int wformat, hipStream_t stream) {
  return wformat == LLMQ_W_INT8 ? launch_bits<T, 8>(qw, ws, out, N, G, gs, keep, out_group, stream)
                                : launch_bits<T, 4>(qw, ws, out, N, G, gs, keep, out_group, stream);
}

}  // namespace

extern "C" int llmq_dequant_weight(const void* qweight, const float* wscale, void* out, int N, int G, int gs,
                                   int keep_per_group, int out_group, int wformat, int dtype,
                                   llmq_stream_t stream) {
  if (N < 0 || G < 0) return llmq_host::fail_invalid("negative dimension N=%d G=%d", N, G);
  if (wformat != LLMQ_W_INT8 && wformat != LLMQ_W_INT4_PACKED)
    return llmq_host::fail_invalid("unsupported weight format %d, expected 8 or 4", wformat);
  if (gs <= 0 || gs % 8)
    return llmq_host::fail_invalid("group_size must be a positive multiple of 8, got %d", gs);
  if (keep_per_group <= 0 || keep_per_group > gs)
    return llmq_host::fail_invalid("keep_per_group must be in [1, %d], got %d", gs, keep_per_group);
  if (out_group < 0) return llmq_host::fail_invalid("out_group must be >= 0, got %d", out_group);
  if (N == 0 || G == 0) return 0;
  if (!qweight || !wscale || !out) return llmq_host::fail_invalid("null tensor pointer");
  if ((reinterpret_cast<uintptr_t>(qweight) | reinterpret_cast<uintptr_t>(out)) & 15u)
    return llmq_host::fail_invalid("weight and output pointers must be 16-byte aligned");
  if (keep_per_group % 8 == 0 && (static_cast<int64_t>(G) * keep_per_group) % 8)
    return llmq_host::fail_invalid("internal: row width not a multiple of 8");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case LLMQ_F32: return launch_typed<float>(qweight, wscale, out, N, G, gs, keep_per_group, out_group, wformat, s);
    case LLMQ_F16: return launch_typed<f16_t>(qweight, wscale, out, N, G, gs, keep_per_group, out_group, wformat, s);
    case LLMQ_BF16: return launch_typed<bf16_t>(qweight, wscale, out, N, G, gs, keep_per_group, out_group, wformat, s);
  }
  return llmq_host::fail_invalid("out must be float32, float16 or bfloat16, got dtype code %d", dtype);
}
