// Symmetric RTN group quantizer for gfx950: quantize-dequantize (fake quant) and the
// codes-emitting variant used for int8 activations.
//
// Arithmetic contract (llmquant/core/observers.py:74-98, llmquant/core/quant_ops.py:13-37,
// restated by the reference's CUDA kernel at llmquant/cuda/csrc/fake_quant.cu:50-84):
//   amax  = max |x| over the group                      (exact in any order)
//   scale = max(amax / qmax, 1e-8)                      fp32, true IEEE division
//   q     = clamp(rint(x / scale), -qmax-1, qmax)       round half to even
//   out   = cast(q * scale)                             round to nearest even
// Nothing here may be contracted, reordered or approximated: the file is built with
// -ffp-contract=off and without fast-math.
//
// Shape of the kernel. The input is read ONCE (the reference's kernel reads it twice): a
// lane owns one 16-byte packet (8 half-width or 4 fp32 elements) and keeps it in registers
// between the abs-max reduction and the quantize step. A group of `gs` elements is
// gs / packet lanes wide -- 16 lanes for the default 128-wide bf16 group, exactly one DPP
// row -- so the reduction is a short butterfly inside the wave and a wave covers a
// contiguous 1 KiB of the tensor per step, fully coalesced. Groups of any other size (or misaligned tensors) take
// quant_group_kernel, which holds a group in the registers of one wave or of four and rereads only beyond 16 Ki
// (fp32: 8 Ki) elements. Rows that are not a whole number of groups are read and written as they lie
// (quant_rows_kernel): the missing elements count as zeros, no padded copy is made.
//
// Bound: HBM (one read, one write), with a third of the vector ALU's time for the IEEE divisions beside it.
#include "llmq_device.h"

namespace {

using namespace llmq;

enum OutMode { kQdq = 0, kCodes8 = 1, kCodes4 = 2 };

template <typename T, int LPG, int MODE>
__global__ __launch_bounds__(256) void quant_lanes_kernel(
    const T* __restrict__ x, void* __restrict__ out, float* __restrict__ scale_out,
    const int64_t total, const int group_size, const float qmin, const float qmax) {
  constexpr int V = Pack<T>::N;
  const int lane = threadIdx.x & (kWave - 1);
  const int64_t wave = (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x) / kWave;
  const int64_t n_waves = static_cast<int64_t>(gridDim.x) * blockDim.x / kWave;
  const int64_t per_wave = static_cast<int64_t>(kWave) * V;

  for (int64_t base = wave * per_wave; base < total; base += n_waves * per_wave) {
    const int64_t e0 = base + static_cast<int64_t>(lane) * V;
    const bool active = e0 < total;  // whole lane groups fall on one side: LPG*V == group_size
    float f[V];
    if (active) {
      Pack<T>::unpack(load16(x + e0), f);
    } else {
#pragma unroll
      for (int i = 0; i < V; ++i) f[i] = 0.0f;
    }
    float amax = 0.0f;
#pragma unroll
    for (int i = 0; i < V; ++i) amax = fmaxf(amax, fabsf(f[i]));
    amax = group_max<LPG>(amax);
    const float scale = scale_from_amax(amax, qmax);
    if (!active) continue;
    if (scale_out != nullptr && (lane & (LPG - 1)) == 0) scale_out[e0 / group_size] = scale;

    float q[V];
#pragma unroll
    for (int i = 0; i < V; ++i) q[i] = quant_code(f[i], scale, qmin, qmax);

    if constexpr (MODE == kQdq) {
#pragma unroll
      for (int i = 0; i < V; ++i) q[i] = q[i] * scale;
      store16(static_cast<T*>(out) + e0, Pack<T>::pack(q));
    } else if constexpr (MODE == kCodes8) {
      uint32_t w[V / 4];
#pragma unroll
      for (int i = 0; i < V / 4; ++i) {
        w[i] = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          w[i] |= (static_cast<uint32_t>(static_cast<int>(q[4 * i + j])) & 0xffu) << (8 * j);
        }
      }
      int8_t* dst = static_cast<int8_t*>(out) + e0;
      if constexpr (V == 8) {
        *reinterpret_cast<u32x2*>(dst) = u32x2{w[0], w[1]};
      } else {
        *reinterpret_cast<uint32_t*>(dst) = w[0];
      }
    } else {
      // nibble packing of llmquant/packing/packing.py:20-33: +8 bias, even index low
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < V; ++i) {
        w |= (static_cast<uint32_t>(static_cast<int>(q[i]) + 8) & 0xfu) << (4 * i);
      }
      uint8_t* dst = static_cast<uint8_t*>(out) + e0 / 2;
      if constexpr (V == 8) {
        *reinterpret_cast<uint32_t*>(dst) = w;
      } else {
        *reinterpret_cast<uint16_t*>(dst) = static_cast<uint16_t>(w);
      }
    }
  }
}

// Packets of T at any address (the memory unit takes 16-byte accesses at element alignment), and the first n elements
// of one, zeros beyond.
template <typename T> __device__ __forceinline__ u32x4 load_packet(const T* p) {
  u32x4 v;
  __builtin_memcpy(&v, p, sizeof v);
  return v;
}
template <typename T, int V = Pack<T>::N> __device__ __forceinline__ void load_elements(const T* p, int n, float* f) {
  if constexpr (V == Pack<T>::N) {
    if (n >= V) {
      Pack<T>::unpack(load_packet(p), f);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < V; ++i) f[i] = i < n ? to_float(p[i]) : 0.0f;
}
template <typename T, int V = Pack<T>::N> __device__ __forceinline__ void store_elements(T* p, int n, const float* q) {
  if constexpr (V == Pack<T>::N) {
    if (n >= V) {
      const u32x4 v = Pack<T>::pack(q);
      __builtin_memcpy(p, &v, sizeof v);
      return;
    }
  }
#pragma unroll
  for (int i = 0; i < V; ++i) {
    if (i < n) p[i] = from_float<T>(q[i]);
  }
}

// Quantize-dequantize of rows whose width is not a whole number of groups. The lanes walk the padded rows (`packets`
// of them a row, a multiple of the group's LPG lanes), and touch what exists of each packet. Measured, 4096 x 5000
// bf16, groups of 128: padding, the kernel on the padded copy and trimming 39.6 us, here 15.3 (82 MB: 5.4 TB/s).
template <typename T, int LPG>
__global__ __launch_bounds__(256) void quant_rows_kernel(
    const T* __restrict__ x, T* __restrict__ out, float* __restrict__ scale_out, const uint32_t total_packets,
    const uint32_t packets, const uint32_t magic, const int shift, const int width, const float qmin, const float qmax) {
  constexpr int V = Pack<T>::N;
  const uint32_t stride = gridDim.x * 256;
  for (uint32_t i0 = blockIdx.x * 256; i0 < total_packets; i0 += stride) {
    const uint32_t i = i0 + threadIdx.x;
    const uint32_t row = shift < 0 ? i : __umulhi(i, magic) >> shift;   // i / packets (i < 2^31)
    const uint32_t packet = i - row * packets;
    const int col = static_cast<int>(packet) * V;
    const int n = i < total_packets ? width - col : 0;   // elements from here to the row's end
    // every lane loads a whole packet, at the latest the row's last one; the elements in front of its own count as zeros
    const int from = min(col, width - V);
    const int64_t at = static_cast<int64_t>(i < total_packets ? row : 0) * width + from;
    float f[V];
    Pack<T>::unpack(load_packet(x + at), f);
    const int skip = n > 0 ? col - from : V;
#pragma unroll
    for (int e = 0; e < V; ++e) f[e] = e >= skip ? f[e] : 0.0f;
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < V; ++e) amax = fmaxf(amax, fabsf(f[e]));
    amax = group_max<LPG>(amax);
    const float scale = scale_from_amax(amax, qmax);
    if (n <= 0) continue;
    if (scale_out != nullptr && (packet & (LPG - 1)) == 0) scale_out[i / LPG] = scale;
    float q[V];
#pragma unroll
    for (int e = 0; e < V; ++e) q[e] = quant_code(f[e], scale, qmin, qmax) * scale;
    if (skip == 0) {
      store_elements(out + at, V, q);
    } else {
#pragma unroll
      for (int e = 1; e < V; ++e) {
        if (e >= skip) out[at + e] = from_float<T>(q[e]);
      }
    }
  }
}

// Any group size, any alignment: WAVES waves per group (one: four groups a workgroup), every thread HELD packets of it
// in registers between the reduction and the quantize step; what goes beyond is read again. Packets are V elements: 16
// bytes at any address (a group a row, one element at a time / here, us: 4096 x 14336 bf16 73 / 37, fp32 137 / 107, int8
// codes of fp32 81 / 60; 3000 x 3000 fp32 12.1 / 11.9, its int8 codes 9.5 / 9.9; 1024 x 4096 bf16 7.0 / 5.3). Groups below
// a packet, and fp32 groups that a wave's lanes hold in four elements each, go element by element (codes of two: nibble
// pairs): one division a lane instead of a chain of eight (64 groups of 4 bf16 2.3 us, 3.0 in a packet; 100000 groups of 20
// fp32 13.3 us, 19.9 in packets).
constexpr int kBlockThreads = 256;

template <typename T, int MODE, int WAVES, int HELD, int V>
__global__ __launch_bounds__(kBlockThreads) void quant_group_kernel(
    const T* __restrict__ x, void* __restrict__ out, float* __restrict__ scale_out, const int64_t n_groups,
    const int group_size, const float qmin, const float qmax) {
  constexpr int kThreads = WAVES * kWave;   // threads of a group
  __shared__ float s_part[kBlockThreads / kWave];
  const int tid = threadIdx.x % kThreads;
  const int64_t group = WAVES * kWave == kBlockThreads ? blockIdx.x
                                                       : static_cast<int64_t>(blockIdx.x) * (kBlockThreads / kThreads) + threadIdx.x / kThreads;
  if (kThreads < kBlockThreads && group >= n_groups) return;   // (whole waves)
  const int64_t base = group * group_size;

  // A packet that would run past the group's end starts earlier: what it repeats changes no maximum, and is written
  // twice with the same values. (Groups below a packet come with a smaller V, element by element.)
  constexpr bool kPackets = V == Pack<T>::N;
  const int last = group_size - V;
  float held[HELD][V];
  float amax = 0.0f;
  if constexpr (kPackets) {
    // (four waves: threads past the group's end load nothing, clamped loads that nobody needs cost up to a seventh there;
    // one wave: they repeat the last packet, 514 elements 5.25 us a launch of 4096 groups against 5.5)
    u32x4 raw[HELD];
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      const int i = (tid + j * kThreads) * V;
      raw[j] = WAVES == 1 || i < group_size ? load_packet(x + base + min(i, last)) : u32x4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < HELD; ++j) Pack<T>::unpack(raw[j], held[j]);
  } else {
#pragma unroll
    for (int j = 0; j < HELD; ++j) {
      const int i = (tid + j * kThreads) * V;
      load_elements<T, V>(x + base + i, group_size - i, held[j]);
    }
  }
#pragma unroll
  for (int j = 0; j < HELD; ++j) {
#pragma unroll
    for (int e = 0; e < V; ++e) amax = fmaxf(amax, fabsf(held[j][e]));
  }
  // (unsigned: the last step of a group of close to 2^31 elements passes that)
  for (uint32_t i = (tid + HELD * kThreads) * V; i < static_cast<uint32_t>(group_size); i += kThreads * V) {
    float f[V];
    load_elements<T, V>(x + base + i, static_cast<int>(group_size - i), f);
#pragma unroll
    for (int e = 0; e < V; ++e) amax = fmaxf(amax, fabsf(f[e]));
  }
  amax = group_max<kWave>(amax);
  if constexpr (WAVES > 1) {
    if ((tid & (kWave - 1)) == 0) s_part[tid / kWave] = amax;
    __syncthreads();
    amax = s_part[0];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) amax = fmaxf(amax, s_part[w]);
  }
  const float scale = scale_from_amax(amax, qmax);
  if (scale_out != nullptr && tid == 0) scale_out[group] = scale;

  auto emit = [&](int i, int n, const float* f) {   // (n: elements from there to the group's end, V if more do not matter)
    float q[V];
#pragma unroll
    for (int e = 0; e < V; ++e) q[e] = quant_code(f[e], scale, qmin, qmax);
    if constexpr (MODE == kQdq) {
#pragma unroll
      for (int e = 0; e < V; ++e) q[e] = q[e] * scale;
      store_elements<T, V>(static_cast<T*>(out) + base + i, n, q);
    } else if constexpr (MODE == kCodes8) {
      int8_t* dst = static_cast<int8_t*>(out) + base + i;
      int8_t codes[V];
#pragma unroll
      for (int e = 0; e < V; ++e) codes[e] = static_cast<int8_t>(static_cast<int>(q[e]));
      if (n >= V) {
        __builtin_memcpy(dst, codes, V);
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) {
          if (e < n) dst[e] = codes[e];
        }
      }
    } else {
      // (an even group size: element pairs of one byte are of one group)
      uint8_t* dst = static_cast<uint8_t*>(out) + (base + i) / 2;
      uint8_t bytes[V / 2 > 0 ? V / 2 : 1];
#pragma unroll
      for (int e = 0; e < V; e += 2) {
        const int lo = static_cast<int>(q[e]) + 8, hi = static_cast<int>(q[e + 1]) + 8;
        bytes[e / 2] = static_cast<uint8_t>((lo & 0xf) | ((hi & 0xf) << 4));
      }
      if (n >= V) {
        __builtin_memcpy(dst, bytes, V / 2);
      } else {
#pragma unroll
        for (int e = 0; e < V; e += 2) {
          if (e < n) dst[e / 2] = bytes[e / 2];
        }
      }
    }
  };
#pragma unroll
  for (int j = 0; j < HELD; ++j) {
    const int i = (tid + j * kThreads) * V;
    if (i < group_size) emit(kPackets ? min(i, last) : i, kPackets ? V : group_size - i, held[j]);
  }
  for (uint32_t i = (tid + HELD * kThreads) * V; i < static_cast<uint32_t>(group_size); i += kThreads * V) {
    float f[V];
    load_elements<T, V>(x + base + i, static_cast<int>(group_size - i), f);
    emit(i, group_size - i, f);
  }
}

// What quant_rows_kernel walks: lanes a group, and whether there is an instance for that many.
template <typename T> bool lanes_of(int group_size, int* lpg) {
  constexpr int V = Pack<T>::N;
  *lpg = group_size / V;
  return group_size % V == 0 && *lpg >= 1 && *lpg <= kWave && (*lpg & (*lpg - 1)) == 0;
}

template <typename T>
int launch_rows(const void* x, void* out, float* scale, int64_t rows, int width, int group_size, float qmin, float qmax,
                hipStream_t stream) {
  int lpg = 0;
  if (width < Pack<T>::N) return llmq_host::fail_invalid("ragged rows need at least a packet of 16 bytes, got width %d", width);
  if (!lanes_of<T>(group_size, &lpg))
    return llmq_host::fail_invalid("ragged rows need a group of a power of two packets, got group_size %d", group_size);
  const int64_t packets = (static_cast<int64_t>(width) + group_size - 1) / group_size * lpg, total = rows * packets;
  if (total >= (1ll << 31)) return llmq_host::fail_invalid("too many elements for one launch: %lld rows of %d", (long long)rows, width);
  // i / packets as (i * magic) >> (31 + bits), 2^(bits - 1) < packets <= 2^bits, magic = ceil(2^(31 + bits) / packets) <
  // 2^32: magic * packets exceeds 2^(31 + bits) by less than packets <= 2^bits, so for i < 2^31 the quotient by less
  // than 1 / packets, which does not reach the next whole number. (packets == 1: shift -1, no division)
  int bits = 0;
  while ((1ll << bits) < packets) ++bits;
  const int shift = bits - 1;
  const uint64_t magic = bits == 0 ? 0 : ((1ull << (31 + bits)) + packets - 1) / packets;
  int64_t blocks = (total + 255) / 256;
  if (blocks > 256 * 32) blocks = 256 * 32;
#define LLMQ_ROWS(L)                                                                                                  \
  case L:                                                                                                             \
    hipLaunchKernelGGL((quant_rows_kernel<T, L>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream,           \
                       static_cast<const T*>(x), static_cast<T*>(out), scale, static_cast<uint32_t>(total),           \
                       static_cast<uint32_t>(packets), static_cast<uint32_t>(magic), shift, width, qmin, qmax);       \
    break;
  switch (lpg) {
    LLMQ_ROWS(1) LLMQ_ROWS(2) LLMQ_ROWS(4) LLMQ_ROWS(8) LLMQ_ROWS(16) LLMQ_ROWS(32) LLMQ_ROWS(64)
  }
#undef LLMQ_ROWS
  return llmq_host::check_launch("quant_rows_kernel");
}

template <typename T, int MODE>
int launch_typed(const void* x, void* out, float* scale, int64_t n_groups, int group_size,
                 float qmin, float qmax, hipStream_t stream) {
  constexpr int V = Pack<T>::N;
  const int64_t total = n_groups * group_size;
  const bool aligned = ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(out)) & 15u) == 0;
  int lpg = 0;
  if (lanes_of<T>(group_size, &lpg) && aligned) {
    const int64_t per_wave = static_cast<int64_t>(kWave) * V;
    const int64_t waves = (total + per_wave - 1) / per_wave;
    int64_t blocks = (waves + 3) / 4;
    const int64_t cap = 256 * 32;  // enough resident waves to cover HBM latency; rest strides
    if (blocks > cap) blocks = cap;
    const dim3 grid(static_cast<unsigned>(blocks)), block(256);
    const T* xp = static_cast<const T*>(x);
#define LLMQ_LANES(L)                                                                        \
  case L:                                                                                    \
    hipLaunchKernelGGL((quant_lanes_kernel<T, L, MODE>), grid, block, 0, stream, xp, out,    \
                       scale, total, group_size, qmin, qmax);                                \
    break;
    switch (lpg) {
      LLMQ_LANES(1) LLMQ_LANES(2) LLMQ_LANES(4) LLMQ_LANES(8)
      LLMQ_LANES(16) LLMQ_LANES(32) LLMQ_LANES(64)
    }
#undef LLMQ_LANES
    return llmq_host::check_launch("quant_lanes_kernel");
  }
  // one wave a group while its lanes hold it in four packets each, four waves beyond
  const bool one_wave = group_size <= kWave * V * 4;
  const int64_t blocks = one_wave ? (n_groups + 3) / 4 : n_groups;
  if (blocks > 2147483647LL) {
    return llmq_host::fail_invalid("too many groups for a 1D grid: %lld", (long long)n_groups);
  }
  const dim3 grid(static_cast<unsigned>(blocks)), block(kBlockThreads);
#define LLMQ_GROUP(WAVES, HELD, V)                                                                                   \
  hipLaunchKernelGGL((quant_group_kernel<T, MODE, WAVES, HELD, V>), grid, block, 0, stream,                          \
                     static_cast<const T*>(x), out, scale, n_groups, group_size, qmin, qmax)
  if (MODE != kCodes4 && V == 4 && group_size <= kWave * 4) LLMQ_GROUP(1, 4, 1);
  else if (group_size < V) LLMQ_GROUP(1, 1, MODE == kCodes4 ? 2 : 1);
  else if (group_size <= kWave * V) LLMQ_GROUP(1, 1, V);
  else if (one_wave) LLMQ_GROUP(1, 4, V);
  else if (group_size <= 4 * kWave * V * 2) LLMQ_GROUP(4, 2, V);   // (2048 groups of 2050 bf16: 6.3 us, 6.9 with four turns)
  else if (group_size <= 4 * kWave * V * 4) LLMQ_GROUP(4, 4, V);
  else LLMQ_GROUP(4, 8, V);
#undef LLMQ_GROUP
  return llmq_host::check_launch("quant_group_kernel");
}

template <int MODE>
int launch(const void* x, void* out, float* scale, int64_t n_groups, int group_size,
           int num_bits, int dtype, hipStream_t stream) {
  const float qmax = static_cast<float>((1 << (num_bits - 1)) - 1);
  const float qmin = -qmax - 1.0f;
  switch (dtype) {
    case LLMQ_F32:
      return launch_typed<float, MODE>(x, out, scale, n_groups, group_size, qmin, qmax, stream);
    case LLMQ_F16:
      return launch_typed<f16_t, MODE>(x, out, scale, n_groups, group_size, qmin, qmax, stream);
    case LLMQ_BF16:
      return launch_typed<bf16_t, MODE>(x, out, scale, n_groups, group_size, qmin, qmax, stream);
  }
  return llmq_host::fail_invalid("x must be float32, float16 or bfloat16, got dtype code %d", dtype);
}

int check_common(const void* x, const void* out, int64_t n_groups, int group_size, int num_bits) {
  if (n_groups < 0) return llmq_host::fail_invalid("n_groups must be >= 0, got %lld", (long long)n_groups);
  if (group_size <= 0) return llmq_host::fail_invalid("group_size must be positive, got %d", group_size);
  if (num_bits < 2 || num_bits > 8) return llmq_host::fail_invalid("num_bits must be in [2, 8], got %d", num_bits);
  if (n_groups > 0 && (x == nullptr || out == nullptr)) return llmq_host::fail_invalid("null tensor pointer");
  return 0;
}

}  // namespace

extern "C" int llmq_fake_quant_group(const void* x, void* out, float* scale_or_null,
                                     int64_t n_groups, int group_size, int num_bits, int dtype,
                                     llmq_stream_t stream) {
  if (int rc = check_common(x, out, n_groups, group_size, num_bits)) return rc;
  if (n_groups == 0) return 0;
  return launch<kQdq>(x, out, scale_or_null, n_groups, group_size, num_bits, dtype,
                      static_cast<hipStream_t>(stream));
}

extern "C" int llmq_fake_quant_rows(const void* x, void* out, float* scale_or_null, int64_t rows, int width,
                                    int group_size, int num_bits, int dtype, llmq_stream_t stream) {
  if (width < 0) return llmq_host::fail_invalid("width must be >= 0, got %d", width);
  if (int rc = check_common(x, out, rows, group_size, num_bits)) return rc;
  if (rows == 0 || width == 0) return 0;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const float qmax = static_cast<float>((1 << (num_bits - 1)) - 1), qmin = -qmax - 1.0f;
  switch (dtype) {
    case LLMQ_F32: return launch_rows<float>(x, out, scale_or_null, rows, width, group_size, qmin, qmax, s);
    case LLMQ_F16: return launch_rows<f16_t>(x, out, scale_or_null, rows, width, group_size, qmin, qmax, s);
    case LLMQ_BF16: return launch_rows<bf16_t>(x, out, scale_or_null, rows, width, group_size, qmin, qmax, s);
  }
  return llmq_host::fail_invalid("x must be float32, float16 or bfloat16, got dtype code %d", dtype);
}

extern "C" int llmq_quant_group_codes(const void* x, void* codes, float* scale, int64_t n_groups,
                                      int group_size, int num_bits, int pack4, int dtype,
                                      llmq_stream_t stream) {
  if (int rc = check_common(x, codes, n_groups, group_size, num_bits)) return rc;
  if (pack4 && num_bits > 4) return llmq_host::fail_invalid("nibble packing needs num_bits <= 4, got %d", num_bits);
  if (pack4 && group_size % 2) return llmq_host::fail_invalid("group_size %d must be even to pack into nibbles", group_size);
  if (n_groups == 0) return 0;
  if (scale == nullptr) return llmq_host::fail_invalid("scale output is required");
  hipStream_t s = static_cast<hipStream_t>(stream);
  return pack4 ? launch<kCodes4>(x, codes, scale, n_groups, group_size, num_bits, dtype, s)
               : launch<kCodes8>(x, codes, scale, n_groups, group_size, num_bits, dtype, s);
}
