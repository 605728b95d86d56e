// Weight-only quantized GEMM for a handful to a few dozen activation rows, gfx950: the codes go from
// HBM to the matrix cores without a dense copy of the weight in between.
//
// KernelQuantLinear takes more than KERNEL_MAX_ROWS rows by rebuilding the whole weight in the
// activation dtype and handing it to a dense matmul (llmquant/quantizers/kernel.py:68-79, 88-91): for
// 4-bit codes that is nine times the codes' bytes through HBM (read codes, write 16-bit values, read
// them again), whatever the row count. Here, for 16-bit activations,
//
//   out[m, n] = sum over g of  wscale[sr(n), g] * sum_k x[m, g*128 + k] * code[n, g, k]
//
// the form of RealQuantLinear's weight-only branch (llmquant/quantizers/real.py:84-91): the codes
// are small integers and exact in bf16 / fp16, so the products are exact in the fp32 accumulator of
// v_mfma_f32_16x16x32_{bf16,f16} and the scale is applied once per group. (The reference's dense
// branch rounds code*scale to the activation dtype first; its own test holds the two branches
// together only within a tolerance, tests/test_kernel_linear.py:62-78.)
//
// A workgroup owns 16, 32 or 64 weight rows; its waves split the groups of the reduction axis between them
// (wave w takes groups w, w + waves, ...) and meet in LDS at the end. Per group a wave reads
//   weights   16 rows x 64 B (4-bit) or 128 B (8-bit), 16 or 32 bytes per lane, straight from HBM
//             in operand layout: lane = (row j = lane % 16, block = lane / 16) holds k = 32 block ..
//             32 block + 31, eight of them per MFMA step
//   x         the group's 128 values of every activation row, through the wave's own LDS tile: whole rows
//             go there straight from L2 (buffer_load_dwordx4 ... lds: four rows of 256 bytes per instruction, eight
//             cache lines; as operand loads, 64 bytes per lane at a row each, the same bytes were 64 lines per
//             instruction and the address unit, not memory, set the pace), 16-byte slots XOR-swizzled by row,
//             and come out as operands: the 32 k of row (lane % 16) that the lane's codes belong to
// and issues 4 MFMAs per activation tile. The next group's transfer and codes are requested once this group's
// operands are in registers (how far they run under its multiplications: at the loop). Rows past M or N are clamped for the loads and dropped at the store, so the load
// sequence is the same for every lane.
#include <type_traits>

#include "llmq_device.h"

namespace {

using namespace llmq;

constexpr int kGroup = 128;
constexpr int kTileN = 16;
constexpr int kTileM = 16;
constexpr int kMaxWaves = 8;
constexpr int kSlabRows = 64;  // activation rows one launch takes (four tiles of 16)

typedef float v4f __attribute__((ext_vector_type(4)));
typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

struct A16Args {
  const void* x;
  const uint8_t* qw;
  const float* ws;
  void* out;
  int M, N, G, out_group;
  int64_t row_bytes;
  int wk, each, more;   // waves of a workgroup; groups of a wave, and waves that have one more
  int scales_at;   // (HELD) where the workgroup's scales lie in LDS
  uint32_t per_row;   // (HELD, G > 1) ceil(2^32 / G): e / G is the upper half of e * per_row, e a scale's place among the workgroup's
};

// HELD: the scales come first, all of a workgroup's in one sweep (its weight rows' are one run of memory, whole lines to a
// load), and wait in LDS. Read group by group, they are a cache line a weight row for four bytes each. Four row tiles, weights
// rotated through 600 MB, in graphs, group by group / held, us: 14336 x 4096 int4 M = 3 12.1 / 9.7, 16 13.6 / 11.1, 32 16.2 / 13.6,
// int8 16 17.6 / 15.7. Short rows do not give the sweep in front back: form_of. Of two row tiles 14336 x 4096 int4, M = 16 14.2 /
// 12.1, but 8192 x 2048 6.0 / 6.1; of one 4096 x 4096 6.7 / 6.8: neither is built. Nor is it for three activation tiles: with an
// earlier loop they had no registers left for it (48 rows: 19.9 / 21.9); with this one they have (18.5 / 16.4).
__host__ __device__ constexpr int scale_pitch(int G) { return G | 1; }   // (odd: sixteen rows in sixteen banks)

// operands of s_waitcnt: none of the wave's vector loads / LDS reads outstanding, the other counters as they are
constexpr int kAllLoads = 0x0f70, kAllReads = 0xc07f;

template <typename T> struct Mfma16;
template <> struct Mfma16<bf16_t> {
  using Vec = v8bf;
  using Elem = __bf16;
  static __device__ __forceinline__ v4f run(Vec a, Vec b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma16<f16_t> {
  using Vec = v8h;
  using Elem = _Float16;
  static __device__ __forceinline__ v4f run(Vec a, Vec b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Eight codes -> eight values of the operand type (exact: |code| <= 128), the signed code itself.
template <typename T, int BITS>
__device__ __forceinline__ typename Mfma16<T>::Vec codes_to_operand(const uint32_t* raw, int step) {
  using E = typename Mfma16<T>::Elem;
  typename Mfma16<T>::Vec v;
  if constexpr (BITS == 4) {
    // nibble i (even i is the low nibble of byte i/2) is code + 8: with its top bit flipped, the code in two's complement
    const uint32_t w = raw[step] ^ 0x88888888u;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = static_cast<E>(static_cast<float>(static_cast<int>(w << (28 - 4 * i)) >> 28));
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[i] = static_cast<E>(static_cast<float>(static_cast<int8_t>(raw[2 * step + i / 4] >> (8 * (i % 4)))));
    }
  }
  return v;
}

template <typename T, int BITS, int MT, int NT, bool BIASED, bool HELD>
__global__ __launch_bounds__(kMaxWaves * kWave) void wq_gemm_a16_kernel(const A16Args a) {
  using Vec = typename Mfma16<T>::Vec;
  constexpr int kRaw = BITS == 4 ? 4 : 8;  // dwords of codes per lane per group and row tile
  constexpr bool kBiased = BIASED;
  constexpr int kRows = NT * kTileN;       // weight rows of the workgroup
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* part = reinterpret_cast<float*>(smem);  // [waves][MT * 16][NT * 16]

  const int tid = threadIdx.x;
  const int lane = tid & (kWave - 1);
  const int wv = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wk = a.wk;
  const int j = lane & 15;
  const int blk = lane >> 4;
  const int G = a.G;
  const int64_t K = static_cast<int64_t>(G) * kGroup;

  const int n0 = blockIdx.x * kRows;
  // (four row tiles: offsets of 32 bits from a scalar base instead of addresses, their registers are needed; the others
  // keep addresses: 8192 x 2048 int4, M = 16: 5.85 us, 5.98 from offsets)
  using Place = typename std::conditional<NT == 4, uint32_t, const uint8_t*>::type;
  auto place = [](const auto* base, int64_t count) {
    if constexpr (NT == 4) return static_cast<uint32_t>(count * sizeof(*base));
    else return reinterpret_cast<const uint8_t*>(base + count);
  };
  auto address = [](const void* base, Place at, int64_t step) {
    if constexpr (NT == 4) return static_cast<const uint8_t*>(base) + step + at;
    else return at + step;
  };
  float* const held = reinterpret_cast<float*>(smem + (HELD ? a.scales_at : 0));
  const int pitch = scale_pitch(G);
  Place wrow[NT], srow[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = min(n0 + nt * kTileN + j, a.N - 1);
    wrow[nt] = place(a.qw, static_cast<int64_t>(n) * a.row_bytes + blk * (BITS == 4 ? 16 : 32));
    srow[nt] = place(a.ws, static_cast<int64_t>(a.out_group > 0 ? n / a.out_group : n) * G);
  }
  // ---- x of one group: [16 MT rows][16 slots of 16 bytes], slot p of row r holds chunk p ^ (r & 15) ------------
  // transfer i of the wave covers rows 4 i .. 4 i + 3; lane = (row 4 i + lane / 16, slot lane % 16)
  constexpr int kXInstr = MT * 4;
  constexpr int kXTileBytes = MT * kTileM * kGroup * 2;
  unsigned char* xtile = smem + wv * kXTileBytes;
  uint32_t xsrc[kXInstr];   // (bytes; launch_typed: a slab's rows span less than 4 GiB)
#pragma unroll
  for (int i = 0; i < kXInstr; ++i) {
    const int row = 4 * i + (lane >> 4), chunk = (lane & 15) ^ (row & 15);
    xsrc[i] = static_cast<uint32_t>(min(row, a.M - 1) * K * 2 + chunk * 16);
  }
  auto request_rows = [&](int g) {
    const BufferBase base = buffer_base(static_cast<const uint8_t*>(a.x) + static_cast<int64_t>(g) * (kGroup * 2));
#pragma unroll
    for (int i = 0; i < kXInstr; ++i) {
      // (four rows past the activation's end are not fetched: what the tile holds there feeds only result rows
      // that are dropped at the store)
      if (4 * i < a.M) buffer_to_lds<16>(base, xtile + 1024 * i, xsrc[i], 0);
    }
  };
  // operand of step s, tile mt: row 16 mt + j, chunk 4 blk + s
  uint32_t x_at[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) x_at[mt] = static_cast<uint32_t>((mt * kTileM + j) * (kGroup * 2));

  struct Weights {
    uint32_t raw[NT][kRaw];
    float scale[HELD ? 1 : NT];
  };
  struct Rows {
    u32x4 xa[MT][4];
  };
  auto load_weights = [&](int g, Weights& W) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      const uint8_t* p = address(a.qw, wrow[nt], static_cast<int64_t>(g) * (kGroup * BITS / 8));
#pragma unroll
      for (int q = 0; q < kRaw / 4; ++q) {
        const u32x4 r = load16(p + 16 * q);
        W.raw[nt][4 * q] = r.x; W.raw[nt][4 * q + 1] = r.y; W.raw[nt][4 * q + 2] = r.z; W.raw[nt][4 * q + 3] = r.w;
      }
      if constexpr (!HELD) W.scale[nt] = *reinterpret_cast<const float*>(address(a.ws, srow[nt], static_cast<int64_t>(g) * 4));
    }
  };
  auto read_rows = [&](Rows& X) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(xtile + x_at[mt] + (((4 * blk + s) ^ j) << 4));
        X.xa[mt][s] = kBiased ? interleave_halves(v) : v;
      }
    }
  };

  v4f acc[NT][MT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};

  // BIASED (int4): the codes become operands without a conversion per element (BiasedCodes: a nibble placed in the
  // mantissa of 16.0 is the value 16 + n: 0.9 vector instructions a code; the signed code takes 2.5). The matrix core then
  // sums x (code + bias); bias * sum_k x comes out per group through four more MFMAs per activation tile against a vector
  // of ones, and the activation's halves are interleaved, both shared by the workgroup's row tiles. It pays where they
  // are: four row tiles, or two with up to two activation tiles. Measured, signed / biased us: 14336 x 4096 int4, four
  // tiles, M = 16: 14.1 / 12.4, 32: 15.9 / 14.7, 48: 18.1 / 17.8 (before the scales were held); two, 16: 13.8 / 13.0, 48: 21.2 / 22.1; one,
  // 4096 x 14336, 16: 12.4 / 12.8. int8 codes gain nothing: a v_cvt either way.
  using Codes = BiasedCodes<T, BITS>;
  uint32_t magic = Codes::kMagic;
  asm volatile("" : "+v"(magic));   // (in a vector register: see and_or)
  const uint32_t one = __builtin_bit_cast(uint16_t, from_float<T>(1.0f));
  const u32x4 ones = {one | (one << 16), one | (one << 16), one | (one << 16), one | (one << 16)};
  auto multiply = [&](int g, const Weights& W, const Rows& X) {
    v4f xsum[MT];   // sum_k x of the group: rows 4 blk + r of tile mt, the same in every column
    if constexpr (kBiased) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        xsum[mt] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          xsum[mt] = Mfma16<T>::run(__builtin_bit_cast(Vec, X.xa[mt][s]), __builtin_bit_cast(Vec, ones), xsum[mt]);
        }
      }
    }
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      Vec b[4];
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        if constexpr (kBiased) b[s] = __builtin_bit_cast(Vec, Codes::operand(W.raw[nt], s, magic));
        else b[s] = codes_to_operand<T, BITS>(W.raw[nt], s);
      }
      const float scale = HELD ? held[(nt * kTileN + j) * pitch + g] : W.scale[HELD ? 0 : nt];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        v4f d = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 4; ++s) d = Mfma16<T>::run(__builtin_bit_cast(Vec, X.xa[mt][s]), b[s], d);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float sum = kBiased ? fmaf(-Codes::kBias, xsum[mt][r], d[r]) : d[r];
          acc[nt][mt][r] = fmaf(sum, scale, acc[nt][mt][r]);
        }
      }
    }
  };

  // (the scales are asked for in front of everything else, kAhead of a thread's values at once: thread by thread they
  // are the rows' scales laid end to end)
  constexpr int kAhead = 8;
  const int n_scales = kRows * G;
  float ahead[kAhead] = {};
  auto row_of = [&](int e) { return static_cast<int>(__umulhi(static_cast<uint32_t>(e), a.per_row)); };   // (e / G)
  auto scale_of = [&](int e) {
    const int row = row_of(e), n = min(n0 + row, a.N - 1);
    return a.ws + static_cast<int64_t>(a.out_group > 0 ? n / a.out_group : n) * G + (e - row * G);
  };
  auto hold = [&](int e, float scale) { held[e + (pitch - G) * row_of(e)] = scale; };
  if constexpr (HELD) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      if (i * blockDim.x < n_scales) ahead[i] = *scale_of(min(i * blockDim.x + tid, n_scales - 1));
    }
  }

  // The wave's groups wv, wv + wk, ...: this group's rows and codes have arrived (nothing else of the wave is in
  // flight), the rows go from the tile to registers, and with the tile free again the next group's transfer
  // and codes are requested; they run under this group's multiplications. That takes a wait the compiler counts (a builtin:
  // one written as assembly it does not see, and it waits for everything once more behind the next group's requests) and
  // transfers that are not FLAT (buffer_to_lds). And nothing slow lies in front of the first request: the host sends the waves'
  // shares along (a division here, and the workgroup's size out of the dispatch packet, are 0.1 to 0.4 us). In graphs, weights
  // rotated, bf16, us, with the waits and FLAT transfers / with a division in front / now: 14336 x 4096 int4, M = 4 / 16 / 32 11.8 /
  // 10.2 / 9.7, 12.7 / 11.4 / 11.0, 15.6 / 14.3 / 13.7; int8 16.0 / 14.7 / 14.4, 16.9 / 15.8 / 15.4, 19.3 / 18.1 / 17.8; 128256 x
  // 2048 int4 M = 24 64.8 / 57.6 / 55.8, int8 78.4 / 73.1 / 71.9; 8192 x 2048 int4 M = 16 6.2 / 6.1 / 6.0, int8 7.1 / 7.3 / 7.0; 4096 x
  // 4096 int4 M = 12 6.2 / 6.2 / 6.2, 32 8.7 / 8.5 / 8.5; the other way: 4096 x 4096 of 16 rows, int4 6.5 / 6.6 / 6.6, int8 7.4 / 7.5
  // / 7.5. What bounds it now: a wave's chain of groups, and the fixed part of a launch (3.5 us). Two groups on their way (two
  // tiles a wave, exact counts) are no faster: 14336 x 4096 int4 M = 16 11.3, 4096 x 14336 17.2 against 15.6, 128256 x 2048 int8 M =
  // 16 84.8 against 62.3.
  Weights W0, W1;
  request_rows(wv);   // (wv < wk <= G)
  load_weights(wv, W0);
  if constexpr (HELD) {
#pragma unroll
    for (int i = 0; i < kAhead; ++i) {
      const int e = i * blockDim.x + tid;
      if (e < n_scales) hold(e, ahead[i]);
    }
    for (int e = kAhead * blockDim.x + tid; e < n_scales; e += blockDim.x) hold(e, *scale_of(e));
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  auto step = [&](int g, bool last, const Weights& now, Weights& next) {
    Rows X;
    __builtin_amdgcn_s_waitcnt(kAllLoads);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    read_rows(X);
    __builtin_amdgcn_s_waitcnt(kAllReads);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (!last) {
      request_rows(g + wk);
      load_weights(g + wk, next);
    }
    multiply(g, now, X);
  };
  // (Two groups a round: the register sets swap by name. By counts, the loop of four row tiles is 0 to 3 % slower, 14336 x 4096 int4
  // M = 17 12.8 us; by groups, short launches of one tile are: 512 x 2048 int8 M = 4 3 %, 1024 x 4096 int4 2.)
  if constexpr (NT == 4) {
    int g = wv;
    do {
      step(g, g + wk >= G, W0, W1);
      if (g + wk < G) step(g + wk, g + 2 * wk >= G, W1, W0);
      g += 2 * wk;
    } while (g < G);
  } else {
    const int count = a.each + (wv < a.more);
    for (int i = 0; i < count; i += 2) {
      step(wv + i * wk, i + 1 >= count, W0, W1);
      if (i + 1 < count) step(wv + (i + 1) * wk, i + 2 >= count, W1, W0);
    }
  }
  __syncthreads();   // every wave is done with its tile: the partial sums take the same memory

  // ---- waves meet: part[wave][m][n], summed in wave order ---------------------------------------
#pragma unroll
  for (int nt = 0; nt < NT; ++nt)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        part[(wv * MT * kTileM + mt * kTileM + 4 * blk + r) * kRows + nt * kTileN + j] = acc[nt][mt][r];
      }
  __syncthreads();
  T* __restrict__ out = static_cast<T*>(a.out);
  const int live = min(wk, G);
  for (int e = tid; e < MT * kTileM * kRows; e += blockDim.x) {
    const int m = e / kRows, jj = e % kRows;
    float total = 0.0f;
    for (int w = 0; w < live; ++w) total += part[(w * MT * kTileM + m) * kRows + jj];
    if (m < a.M && n0 + jj < a.N) out[static_cast<int64_t>(m) * a.N + n0 + jj] = from_float<T>(total);
  }
}

constexpr int kMostScales = 64 * 1024;   // (a workgroup of four row tiles has the CU to itself: 255 groups a row)
constexpr int64_t held_bytes(int row_tiles, int G) { return int64_t{row_tiles * kTileN} * scale_pitch(G) * 4; }

template <typename T, int BITS, int MT, int NT, bool BIASED, bool HELD = false>
int launch_tile(A16Args a, int wk, hipStream_t stream) {
  a.wk = wk, a.each = a.G / wk, a.more = a.G % wk;
  const int grid = (a.N + NT * kTileN - 1) / (NT * kTileN);
  // the waves' activation tiles, then (the same memory) their partial sums
  const int part = wk * MT * kTileM * NT * kTileN * static_cast<int>(sizeof(float));
  const int tiles = wk * MT * kTileM * kGroup * 2;
  int lds = part > tiles ? part : tiles;
  if constexpr (HELD) {   // (form_of: they fit)
    a.scales_at = lds, lds += static_cast<int>(held_bytes(NT, a.G));
    a.per_row = static_cast<uint32_t>(((uint64_t{1} << 32) + a.G - 1) / a.G);
  }
  auto kernel = wq_gemm_a16_kernel<T, BITS, MT, NT, BIASED, HELD>;
  if (lds > 64 * 1024) {
    static bool raised = false;  // per instantiation; worst case two threads both set it
    if (!raised) {
      const hipError_t err = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      if (err != hipSuccess) {
        llmq_host::set_error("raising the LDS limit failed: %s", hipGetErrorString(err));
        return static_cast<int>(err);
      }
      raised = true;
    }
  }
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(wk * kWave), lds, stream, a);
  return llmq_host::check_launch("wq_gemm_a16_kernel");
}

// Which form a slab of activation rows takes: row tiles of a workgroup, and whether its scales are held.
struct Form {
  int row_tiles;
  bool held;
};
// Row tiles of a workgroup share the activation rows a wave loads: those come from L2 once per workgroup, and 16
// weight rows a workgroup make that traffic four times the codes' at M = 16. Two tiles as long as a workgroup per CU
// and more is left (in graphs, weights rotated through 600 MB, bf16, us, one / two tiles: 14336 x 4096 int4 M = 16 17.8 / 14.2, 32
// 24.2 / 18.2, 48 33.9 / 23.5; 4096 x 4096, M = 64: 12.1 / 14.4).
// Four tiles (one workgroup a CU) by how full their last round of 256 workgroups is. The lines are those of an earlier loop;
// measured with the present one, as above, two tiles / four / four with the scales held (fp16 within 3 %):
//  17 rows and more, K = 4096: 192 workgroups int4 M = 17 / 32 / 48: 15.1 / 14.5 / 12.1, 17.9 / 15.9 / 13.4, 23.0 / 18.1 / 16.1, int8
//  32: 23.8 / 19.9 / 17.5; 256: 15.0 / 14.6 / 12.3, 17.8 / 16.1 / 13.6, 23.2 / 18.4 / 16.3, int8 25.9 / 20.9 / 19.4; two for 260 to
//  384, a second round at most half full: 288 20.2 / 26.0 / 21.3, 24.7 / 28.9 / 23.9, 32.9 / 33.0 / 28.9, int8 17 28.8 / 33.3 / 29.5;
//  384 21.5 / 26.6 / 21.9, 25.6 / 29.5 / 24.6, int8 17 32.2 / 34.3 / 31.4; 416 25.6 / 26.9 / 22.2, 31.8 / 29.8 / 24.9, int8 32 45.2 /
//  38.1 / 34.0; 528 int4 32 38.6 / 42.2 / 34.9, int8 56.0 / 54.8 / 47.6. Below 192: 8192 x 2048 M = 32 7.4 / 9.5 (four).
//  Up to 16 rows there is less to share: one round only (288, M = 3 / 16: 15.2 / 19.9 / 14.4, 19.2 / 23.0 / 17.6; 448: 20.2 / 20.5 /
//  15.1, 24.9 / 23.7 / 18.6), rows of 32 groups (256 workgroups, K = 2048: 7.5 / 8.1 / 7.3, 8.6 / 8.5 / 7.8; K = 4096 11.3 / 12.0 /
//  9.7, 14.0 / 13.4 / 11.0; K = 8192, 16: 26.8 / 25.2 / 19.6), and for int8 codes up to eight rows, the fuller the round the longer
//  the rows that it takes (two / held; 192: 32 groups M = 3 / 8 15.9 / 13.3, 16.5 / 13.7; 224: 17.0 / 14.6, 17.0 / 14.5; 240: 32
//  groups 17.1 / 15.4, 17.1 / 15.4, 48 groups 22.2 / 19.2, 24.5 / 19.7; 256: 32 groups M = 3 17.0 / 16.8, 64 groups M = 3 / 5 30.1 /
//  29.9, 30.6 / 30.0, 96 groups 44.9 / 43.7, 46.3 / 43.6, 255 groups M = 3 143 / 134).
//  With the scales held four tiles are ahead of where the lines lie, by most at 288 and 448 workgroups of up to 16 rows and at
//  33 to 48 rows; two are at 2004 workgroups of K = 2048 int4, M = 17 (50.7 / 52.4).
// Four tiles against 64 rows, and int8 codes against 48, are more registers than a wave has (spills: 39, int8 50 and 3).
constexpr Form form_of(int bits, int rows, int N, int G) {
  const int quads = (N + 4 * kTileN - 1) / (4 * kTileN), mt = (rows + kTileM - 1) / kTileM;
  const bool int4 = bits == 4;
  const int64_t K = static_cast<int64_t>(G) * kGroup, limit = int64_t{1} << 32;   // the four-tile form's offsets from its scalar bases
  const bool offsets32 = N * (K * bits / 8) < limit && static_cast<int64_t>(N) * G * 4 < limit && kSlabRows * K * 2 < limit;
  const bool few_codes = int4 || rows > 8 || quads <= 224 || G >= (quads < 256 ? 40 : rows > 4 ? 96 : 192);
  const bool few_rows = mt == 1 && quads <= 256 && G >= 32 && few_codes;
  const bool more_rows = (mt == 2 || (mt == 3 && int4)) && (quads <= 256 || quads > 384);
  if (quads >= 192 && offsets32 && (few_rows || more_rows)) {
    // The scales of rows that are long enough to pay for the sweep are held, and of somewhat shorter ones where several rounds of
    // workgroups overlap it and the waves have equal shares: with an earlier loop the sweep cost shorter ones up to 16 %. With the
    // present one, group by group / held, us, in graphs, M = 17 / 32, int4, 256 workgroups: K = 512 7.1 / 7.0, 7.4 / 7.4; 2048 9.3 /
    // 8.5, 10.2 / 9.4; 2560 10.9 / 9.5, 11.5 / 11.0; 3584 13.5 / 11.6, 14.5 / 13.1; 4096 14.6 / 12.3, 16.1 / 13.6; 2004 workgroups, K =
    // 2048 59.8 / 52.4, 65.5 / 58.7; int8, 256 workgroups, K = 512 7.9 / 7.8, 8.2 / 8.2; 2048 11.7 / 10.5, 11.9 / 11.4; 2560 13.4 / 12.9,
    // 14.4 / 14.0 (fp16 15.2 / 13.4, 14.7 / 14.6); 4096 19.3 / 18.5, 20.9 / 19.4; 2004, K = 2048 76.5 / 68.8, 82.2 / 75.2.
    const bool long_rows = int4 ? mt == 1 || G >= 20 : G >= (quads > 240 && quads <= 256 ? 40 : 32);
    const bool pays = long_rows || (G >= 16 && G % kMaxWaves == 0 && quads >= (int4 ? 385 : 1024));
    return {4, mt <= 2 && pays && held_bytes(4, G) <= kMostScales};
  }
  return {N >= 2 * kTileN * 256 ? 2 : 1, false};
}

template <typename T, int BITS>
int launch_typed(const void* x, const void* qw, const float* ws, void* out, int M, int N, int G, int out_group,
                 hipStream_t stream) {
  const int64_t K = static_cast<int64_t>(G) * kGroup;
  int wk = G < kMaxWaves ? G : kMaxWaves;
  // rows of few groups: two groups per wave at least
  if (G >= 4 && wk * 2 > G) wk = G / 2;
  // (Sixteen waves for few row tiles of long rows, down_proj, measured no faster than eight, with an earlier loop.)
  // (a slab's offsets have 32 bits)
  const int64_t fit = (int64_t{1} << 32) / (K * 2);
  const int slab = fit >= kSlabRows ? kSlabRows : (fit > 0 ? static_cast<int>(fit) : 1);
  for (int m0 = 0; m0 < M; m0 += slab) {
    A16Args a{};
    a.x = static_cast<const T*>(x) + static_cast<int64_t>(m0) * K;
    a.qw = static_cast<const uint8_t*>(qw);
    a.ws = ws;
    a.out = static_cast<T*>(out) + static_cast<int64_t>(m0) * N;
    a.M = M - m0 < slab ? M - m0 : slab;
    a.N = N; a.G = G; a.out_group = out_group;
    a.row_bytes = K * BITS / 8;
    const int mt = (a.M + kTileM - 1) / kTileM;
    const Form form = form_of(BITS, a.M, N, G);
    int rc = 0;
    if (form.row_tiles == 4) {
      constexpr bool kBi = BITS == 4;
      if (mt == 1) {
        rc = form.held ? launch_tile<T, BITS, 1, 4, kBi, true>(a, wk, stream) : launch_tile<T, BITS, 1, 4, kBi>(a, wk, stream);
      } else if (mt == 2) {
        rc = form.held ? launch_tile<T, BITS, 2, 4, kBi, true>(a, wk, stream) : launch_tile<T, BITS, 2, 4, kBi>(a, wk, stream);
      } else if constexpr (BITS == 4) {
        rc = launch_tile<T, BITS, 3, 4, kBi>(a, wk, stream);
      }
    } else if (form.row_tiles == 2) {
      switch (mt) {
        case 1: rc = launch_tile<T, BITS, 1, 2, BITS == 4>(a, wk, stream); break;
        case 2: rc = launch_tile<T, BITS, 2, 2, BITS == 4>(a, wk, stream); break;
        case 3: rc = launch_tile<T, BITS, 3, 2, false>(a, wk, stream); break;
        default: rc = launch_tile<T, BITS, 4, 2, false>(a, wk, stream); break;
      }
    } else {
      switch (mt) {
        case 1: rc = launch_tile<T, BITS, 1, 1, false>(a, wk, stream); break;
        case 2: rc = launch_tile<T, BITS, 2, 1, false>(a, wk, stream); break;
        case 3: rc = launch_tile<T, BITS, 3, 1, false>(a, wk, stream); break;
        default: rc = launch_tile<T, BITS, 4, 1, false>(a, wk, stream); break;
      }
    }
    if (rc) return rc;
  }
  return 0;
}

}  // namespace

extern "C" int llmq_wq_gemm_a16(const void* x, const void* qweight, const float* wscale, void* out, int M, int N,
                                int G, int gs, int out_group, int wformat, int dtype, llmq_stream_t stream) {
  if (M < 0 || N < 0 || G < 0) return llmq_host::fail_invalid("negative dimension M=%d N=%d G=%d", M, N, G);
  if (gs != kGroup) return llmq_host::fail_invalid("the fused GEMM needs group_size 128, got %d", gs);
  if (out_group < 0) return llmq_host::fail_invalid("out_group must be >= 0, got %d", out_group);
  if (wformat != LLMQ_W_INT8 && wformat != LLMQ_W_INT4_PACKED)
    return llmq_host::fail_invalid("unsupported weight format %d, expected 8 or 4", wformat);
  if (dtype != LLMQ_F16 && dtype != LLMQ_BF16)
    return llmq_host::fail_invalid("the fused GEMM takes float16 or bfloat16 activations, got dtype code %d", dtype);
  if (M == 0 || N == 0) return 0;
  if (G == 0) return llmq_host::fail_invalid("a weight with no groups has no reduction axis");
  if (!x || !qweight || !wscale || !out) return llmq_host::fail_invalid("null tensor pointer");
  if ((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(qweight)) & 15u)
    return llmq_host::fail_invalid("x and qweight must be 16-byte aligned");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (dtype == LLMQ_BF16) {
    return wformat == LLMQ_W_INT8 ? launch_typed<bf16_t, 8>(x, qweight, wscale, out, M, N, G, out_group, s)
                                  : launch_typed<bf16_t, 4>(x, qweight, wscale, out, M, N, G, out_group, s);
  }
  return wformat == LLMQ_W_INT8 ? launch_typed<f16_t, 8>(x, qweight, wscale, out, M, N, G, out_group, s)
                                : launch_typed<f16_t, 4>(x, qweight, wscale, out, M, N, G, out_group, s);
}
