// W4A16 support kernels: packet builder, dequantisers, activation group sums, split-K reduction.
//
// Each follows the math of its reference counterpart in arc_w4a16.cu (cited per kernel) with a
// gfx950-shaped decomposition: 16-byte global accesses, one thread per 8 codes (one uint32 of
// nibbles), and no per-element 1-byte loads.
#include "w4a16_aux.h"

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

#include "w4a16_device.h"

namespace fk {
namespace {

constexpr int kAuxThreads = 256;

// Code words of one 128-row tile over 256 values of K in LDS, word row by word row as in a reference
// packet; the pitch keeps rows 16-byte aligned and spreads the word rows over the banks.
constexpr int kTurnK = 256;
constexpr int kTurnWords = kTurnK / 8;
constexpr int kTurnPitch = kTileCols + 4;
constexpr int kMaxTurns = 4;  // turns of 256 values a packing workgroup takes at most

// half_rn(fma(alpha, q, beta)) for the 8 codes of one uint32 word (k = 8w .. 8w+7). For the
// quantisation recipes used here alpha*q + beta is exact in fp32, so the single fp16 rounding
// makes the result bit-exact whatever the evaluation order (dequant_w4a16_kernel,
// arc_w4a16.cu:160-181, computes the same value).
__device__ __forceinline__ uint4 dequant_word(uint32_t word, float a, float b) {
  uint32_t h[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float q = static_cast<float>((word >> (4 * j)) & 0xfu);
    h[j] = float_to_half_bits(fmaf(a, q, b));
  }
  return make_uint4(h[0] | (h[1] << 16), h[2] | (h[3] << 16), h[4] | (h[5] << 16), h[6] | (h[7] << 16));
}

// dequant_w4a16_kernel (arc_w4a16.cu:160-181): q_u8[N, K/2] + alpha/beta[N, NG] -> W[N, K] fp16.
template <int G>
__global__ void __launch_bounds__(kAuxThreads)
dequant_kernel(const uint32_t* __restrict__ q, const uint16_t* __restrict__ alpha,
               const uint16_t* __restrict__ beta, uint4* __restrict__ out, size_t total_words,
               int words_per_row, int num_groups) {
  const size_t idx = static_cast<size_t>(blockIdx.x) * kAuxThreads + threadIdx.x;
  if (idx >= total_words) {
    return;
  }
  const size_t row = idx / words_per_row;
  const int w = static_cast<int>(idx % words_per_row);
  const int g = (w * 8) / G;
  const float a = half_bits_to_float(alpha[row * num_groups + g]);
  const float b = half_bits_to_float(beta[row * num_groups + g]);
  out[idx] = dequant_word(q[idx], a, b);
}

// dequant_arc_packets_kernel (arc_w4a16.cu:183-220): packets -> W[N, K] fp16. A workgroup takes a
// tile over 256 values of K: 512-byte word rows in, through LDS, 512 bytes of each row of W out
// (a row's words are 512 bytes apart in the packets: reading them in W's order fetched every line
// many times over). HBM-bound: 8192 x 8192 G128 69.2 -> 29.5 us with cold packets (5.8 TB/s; a large copy
// runs at 5.2), 28672 x 4096 118 -> 55. (A few workgroups take longer, below a call's 8 us on the host: 1920
// x 1152 4.0 -> 6.2.)
template <int G>
__global__ void __launch_bounds__(kAuxThreads)
dequant_packets_kernel(const uint8_t* __restrict__ packets, uint4* __restrict__ out, int k,
                       int num_groups) {
  constexpr int QB = kTileCols * G / 2;
  constexpr int WR = G / 8;
  constexpr int kGroups = kTurnK / G;
  __shared__ __attribute__((aligned(16))) uint32_t words[kTurnWords][kTurnPitch];
  __shared__ uint16_t scales[kGroups][2 * kTileCols];
  const int tid = static_cast<int>(threadIdx.x);
  const int tile = static_cast<int>(blockIdx.y);
  const int g0 = static_cast<int>(blockIdx.x) * kGroups;
  const int groups = min(kGroups, num_groups - g0);
  const size_t stride = static_cast<size_t>(packet_stride_bytes(G));
  const uint8_t* src = packets + (static_cast<size_t>(tile) * num_groups + g0) * stride;
#pragma unroll
  for (int it = 0; it < kTurnWords * kTileCols / 4 / kAuxThreads; ++it) {
    const int u = it * kAuxThreads + tid;
    const int wr = u / (kTileCols / 4);
    const int c = u % (kTileCols / 4) * 4;
    if (wr < groups * WR) {
      *reinterpret_cast<uint4*>(&words[wr][c]) =
          stream_load16(src + (wr / WR) * stride + (wr % WR * kTileCols + c) * 4);
    }
  }
  for (int i = tid; i < groups * kTileCols; i += kAuxThreads) {  // two scales a thread
    const int g = i / kTileCols;
    reinterpret_cast<uint32_t*>(scales[g])[i % kTileCols] =
        reinterpret_cast<const uint32_t*>(src + g * stride + QB)[i % kTileCols];
  }
  __syncthreads();
  const int words_per_row = k / 8;
#pragma unroll 4
  for (int it = 0; it < kTurnWords * kTileCols / kAuxThreads; ++it) {
    const int u = it * kAuxThreads + tid;
    const int c = u / kTurnWords;
    const int wr = u % kTurnWords;
    if (wr < groups * WR) {
      const uint16_t* ab = scales[wr / WR];
      out[(static_cast<size_t>(tile) * kTileCols + c) * words_per_row + g0 * WR + wr] = dequant_word(
          words[wr][c], half_bits_to_float(ab[c]), half_bits_to_float(ab[kTileCols + c]));
    }
  }
}

// compute_arc_group_sums_kernel (arc_w4a16.cu:124-158): sums[b, g] = sum of x[b, g*G .. +G) in
// fp32. One wave per (row, group): each lane adds two values, then a shuffle tree.
template <int G>
__global__ void __launch_bounds__(64)
group_sums_kernel(const uint32_t* __restrict__ x, float* __restrict__ sums, int k,
                  int num_groups) {
  const int b = static_cast<int>(blockIdx.x);
  const int g = static_cast<int>(blockIdx.y);
  const int lane = static_cast<int>(threadIdx.x);
  float v = 0.0f;
  if (lane < G / 2) {
    const uint32_t pair = x[(static_cast<size_t>(b) * k + static_cast<size_t>(g) * G) / 2 + lane];
    v = half_bits_to_float(static_cast<uint16_t>(pair)) + half_bits_to_float(static_cast<uint16_t>(pair >> 16));
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    v += __shfl_xor(v, off);
  }
  if (lane == 0) {
    sums[static_cast<size_t>(b) * num_groups + g] = v;
  }
}

// reduce_arc_w4a16_split_k_partials_kernel (arc_w4a16.cu:388-402): out[i] = half_rn(sum over
// slices of partials[s, i]), slices added in order 0..S-1.
__global__ void __launch_bounds__(kAuxThreads)
reduce_partials_kernel(const float* __restrict__ partials, uint16_t* __restrict__ out,
                       size_t total, int split_k_slices) {
  const size_t idx = static_cast<size_t>(blockIdx.x) * kAuxThreads + threadIdx.x;
  if (idx >= total) {
    return;
  }
  float v = 0.0f;
  for (int s = 0; s < split_k_slices; ++s) {
    v += partials[static_cast<size_t>(s) * total + idx];
  }
  out[idx] = float_to_half_bits(v);
}

unsigned int blocks_for(size_t n, int threads) {
  return static_cast<unsigned int>((n + threads - 1) / threads);
}


// Where column c (0..127) of tile `tile`, group g lives in the native slabs (PacketFormat in
// w4a16_device.h): its slab and its column 16*i + n inside the slab.
struct NativeSlot {
  uint8_t* slab;
  int i;
  int n;
};

template <int G, PacketFormat F>
__device__ __forceinline__ NativeSlot native_slot(uint8_t* packets, int tile, int g, int c,
                                                  int num_groups) {
  const size_t slab = (static_cast<size_t>(tile) * kSlicesPerTile + c / kSliceCols) * num_groups + g;
  const int cs = c % kSliceCols;
  return {packets + slab * static_cast<size_t>(format_packet_stride(G, F)), cs / 16, cs % 16};
}

// Code word w (codes k = 8w .. 8w+7 of the group) of the slot's column.
template <int G>
__device__ __forceinline__ uint32_t* slab_word(NativeSlot s, int w) {
  constexpr int U = native_unit_words(G);
  return reinterpret_cast<uint32_t*>(s.slab + native_word_offset(G, s.i, w / U, s.n, w % U));
}

template <int G, PacketFormat F>
__device__ __forceinline__ uint16_t* slab_alpha(NativeSlot s) {
  return reinterpret_cast<uint16_t*>(s.slab + native_record_offset(G) + native_record_bytes(F) * s.n) +
         s.i;
}

// kNativeAsym: the word after the column pair's alphas (-zp[n] and -zp[n + 16] as fp16).
template <int G>
__device__ __forceinline__ uint32_t* slab_zp_word(NativeSlot s) {
  return reinterpret_cast<uint32_t*>(s.slab + native_record_offset(G) +
                                     native_record_bytes(PacketFormat::kNativeAsym) * s.n + 4);
}

// Writes -zp of this thread's column (half s.i of the column pair's word).
template <int G>
__device__ __forceinline__ void store_neg_zp(NativeSlot s, uint32_t zp) {
  reinterpret_cast<uint16_t*>(slab_zp_word<G>(s))[s.i] = neg_zp_half_bits(zp & 0xFu);
}

// Packets of any format from q_u8 [N, K/2], alpha [N, NG] and the offsets: beta fp16 (kArc,
// pack_arc_packets_kernel, arc_w4a16.cu:87-122: word w of column c at byte (w*128 + c)*4, then
// alpha[128], then beta[128]) or zero points uint8 [N, NG], values 0..15 (kNativeAsym). A workgroup
// takes a tile, 256 values of K at a time: 128 bytes of each of the tile's rows in, through LDS,
// whole word rows (kArc) or 1 KB runs of slabs out; scales through LDS too, those of up to four
// turns at once. (One thread per column and group read 64 bytes of each row, with the line's other
// half read by another workgroup much later, and every scale with a line of its own.) HBM-bound. With
// cold tensors: to reference packets 57344 x 8192 G128 144.5 -> 105 us (4.8 TB/s), 8192 x 8192 22.9 -> 17.8,
// 28672 x 4096 30.3 -> 30.1, G64 41.8 -> 35.9; to native slabs 127.5 -> 103.5, 20.9 -> 15.9, 28.3 -> 27.6 and
// 34.5 -> 30.7. (Weights of a few MB take longer, below a call's 8 us on the host: 1024 x 4096 2.8 -> 3.4.)
template <int G, PacketFormat F>
__global__ void __launch_bounds__(kAuxThreads)
pack_kernel(const uint8_t* __restrict__ q, const uint16_t* __restrict__ alpha,
            const void* __restrict__ offsets, uint8_t* __restrict__ packets, int k, int num_groups,
            int turns_per_group) {
  constexpr int WR = G / 8;
  constexpr int kGroups = kTurnK / G;
  constexpr size_t kStride = format_packet_stride(G, F);
  constexpr bool kOffsets = F != PacketFormat::kNativeSym;
  constexpr int kScalePitch = kTileCols + 2;  // 4-byte aligned, groups on different banks
  __shared__ __attribute__((aligned(16))) uint32_t words[kTurnWords][kTurnPitch];
  __shared__ __attribute__((aligned(4))) uint16_t scales[kOffsets ? 2 : 1][kMaxTurns * kGroups][kScalePitch];
  const int tid = static_cast<int>(threadIdx.x);
  const int tile = static_cast<int>(blockIdx.y);
  const size_t row0 = static_cast<size_t>(tile) * kTileCols;
  const int turns = (num_groups + kGroups - 1) / kGroups;
  const int turn0 = static_cast<int>(blockIdx.x) * turns_per_group;
  const int turn1 = min(turns, turn0 + turns_per_group);
  // Group g of the tile: its packet (kArc), or its slab of slice s.
  auto packet = [&](int s, int g) {
    const size_t unit = F == PacketFormat::kArc ? static_cast<size_t>(tile)
                                                : static_cast<size_t>(tile) * kSlicesPerTile + s;
    return packets + (unit * num_groups + g) * kStride;
  };
  // The workgroup's scales first, consecutive lanes on consecutive groups of a row.
  const int first = turn0 * kGroups;
  const int width = turns_per_group * kGroups;  // a power of two
  const int shift = __builtin_ctz(width);
  const int have = min(num_groups - first, width);
  for (int i = tid; i < kTileCols << shift; i += kAuxThreads) {
    const int c = i >> shift;
    const int g = i & (width - 1);
    if (g < have) {
      const size_t at = (row0 + c) * num_groups + first + g;
      scales[0][g][c] = alpha[at];
      if constexpr (F == PacketFormat::kArc) {
        scales[1][g][c] = static_cast<const uint16_t*>(offsets)[at];
      } else if constexpr (kOffsets) {
        scales[1][g][c] = neg_zp_half_bits(static_cast<const uint8_t*>(offsets)[at] & 0xFu);
      }
    }
  }
  for (int turn = turn0; turn < turn1; ++turn) {
    const int g0 = turn * kGroups;
    const int groups = min(kGroups, num_groups - g0);
    if (turn != turn0) {
      __syncthreads();
    }
    const uint8_t* src = q + row0 * (k / 2) + static_cast<size_t>(g0) * (G / 2);
#pragma unroll
    for (int it = 0; it < kTurnWords * kTileCols / 4 / kAuxThreads; ++it) {
      const int u = it * kAuxThreads + tid;
      const int v = u % (kTurnWords / 4);
      const int r = u / (kTurnWords / 4);
      if (4 * v < groups * WR) {
        const uint4 d = stream_load16(src + static_cast<size_t>(r) * (k / 2) + v * 16);
        words[4 * v + 0][r] = d.x;
        words[4 * v + 1][r] = d.y;
        words[4 * v + 2][r] = d.z;
        words[4 * v + 3][r] = d.w;
      }
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < kTurnWords * kTileCols / 4 / kAuxThreads; ++it) {
      const int u = it * kAuxThreads + tid;
      constexpr int kUnits = WR * kTileCols / 4;  // 16-byte units of a group
      const int g = u / kUnits;
      const int e = u % kUnits;
      if (g < groups) {
        if constexpr (F == PacketFormat::kArc) {
          const uint4 d = *reinterpret_cast<const uint4*>(&words[g * WR + e / 32][e % 32 * 4]);
          *reinterpret_cast<uint4*>(packet(0, g0 + g) + e * 16) = d;
        } else {
          // unit l of half i (G = 128), or both halves' two words (G = 64), of slice s
          constexpr int kPerSlice = kUnits / kSlicesPerTile;
          const int s = e / kPerSlice;
          const int l = e % 64;
          const int n = s * kSliceCols + l % 16;
          const int w0 = g * WR + l / 16 * native_unit_words(G);
          uint4 d;
          if constexpr (G == 128) {
            const int c = n + 16 * (e % kPerSlice / 64);
            d = make_uint4(words[w0][c], words[w0 + 1][c], words[w0 + 2][c], words[w0 + 3][c]);
          } else {
            d = make_uint4(words[w0][n], words[w0 + 1][n], words[w0][n + 16], words[w0 + 1][n + 16]);
          }
          *reinterpret_cast<uint4*>(packet(s, g0 + g) + e % kPerSlice * 16) = d;
        }
      }
    }
    // scales, 4 bytes a store: two columns' alphas or betas (kArc), a record or half of one
    for (int i = tid; i < groups * kTileCols; i += kAuxThreads) {
      const int g = i / kTileCols;
      const int e = i % kTileCols;
      const int gs = g0 - first + g;
      if constexpr (F == PacketFormat::kArc) {
        const int c = 2 * e % kTileCols;
        reinterpret_cast<uint32_t*>(packet(0, g0 + g) + kTileCols * G / 2)[e] =
            *reinterpret_cast<const uint32_t*>(&scales[2 * e / kTileCols][gs][c]);
      } else {
        constexpr int kWords = native_record_bytes(F) / 4;
        const int s = e / (16 * kWords);
        const int n = e / kWords % 16;
        if (s < kSlicesPerTile) {
          const uint16_t* row = scales[kOffsets ? e % kWords : 0][gs] + s * kSliceCols + n;
          reinterpret_cast<uint32_t*>(packet(s, g0 + g) + native_record_offset(G))[e % (16 * kWords)] =
              row[0] | (static_cast<uint32_t>(row[16]) << 16);
        }
      }
    }
  }
}

// Reference packets -> native slabs. The zero point of a (column, group) is the integer zp in
// 0..15 with half_rn(-alpha * zp) == beta (bit for bit); kNativeSym requires zp = 8.
// (column, group)s with no such zp raise *bad, and the caller rejects the conversion.
template <int G, PacketFormat F>
__global__ void __launch_bounds__(kTileCols)
arc_to_native_kernel(const uint8_t* __restrict__ arc, uint8_t* __restrict__ native, int num_groups,
                     uint32_t* __restrict__ bad) {
  constexpr int QB = kTileCols * G / 2;
  const int tile = static_cast<int>(blockIdx.x);
  const int g = static_cast<int>(blockIdx.y);
  const int c = static_cast<int>(threadIdx.x);
  const size_t unit = static_cast<size_t>(tile) * num_groups + g;
  const uint8_t* src = arc + unit * static_cast<size_t>(packet_stride_bytes(G));
  const NativeSlot s = native_slot<G, F>(native, tile, g, c, num_groups);
  const uint32_t* sw = reinterpret_cast<const uint32_t*>(src);
#pragma unroll
  for (int w = 0; w < G / 8; ++w) {
    *slab_word<G>(s, w) = sw[w * kTileCols + c];
  }
  const uint16_t a_bits = reinterpret_cast<const uint16_t*>(src + QB)[c];
  const uint16_t b_bits = reinterpret_cast<const uint16_t*>(src + QB)[kTileCols + c];
  *slab_alpha<G, F>(s) = a_bits;
  int zp = -1;
  if constexpr (F == PacketFormat::kNativeSym) {
    zp = neg_alpha_zp_bits(a_bits, 8) == b_bits ? 8 : -1;
  } else {
    for (int z = 0; z < 16; ++z) {
      if (zp < 0 && neg_alpha_zp_bits(a_bits, static_cast<uint32_t>(z)) == b_bits) {
        zp = z;
      }
    }
  }
  // *bad is host memory: one store a wave, and none for packets that convert
  if (__any(zp < 0) && (c & 63) == 0) {
    __hip_atomic_store(bad, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
  zp = max(zp, 0);
  if constexpr (F == PacketFormat::kNativeAsym) {
    store_neg_zp<G>(s, static_cast<uint32_t>(zp));
  }
}

// Native slabs -> reference packets: the same codes and alpha, beta = half_rn(-alpha * zp).
template <int G, PacketFormat F>
__global__ void __launch_bounds__(kTileCols)
native_to_arc_kernel(const uint8_t* __restrict__ native, uint8_t* __restrict__ arc, int num_groups) {
  constexpr int QB = kTileCols * G / 2;
  const int tile = static_cast<int>(blockIdx.x);
  const int g = static_cast<int>(blockIdx.y);
  const int c = static_cast<int>(threadIdx.x);
  const size_t unit = static_cast<size_t>(tile) * num_groups + g;
  // The slab is only read here; native_slot takes a non-const pointer for the writers.
  const NativeSlot s = native_slot<G, F>(const_cast<uint8_t*>(native), tile, g, c, num_groups);
  uint8_t* dst = arc + unit * static_cast<size_t>(packet_stride_bytes(G));
  uint32_t* dw = reinterpret_cast<uint32_t*>(dst);
#pragma unroll
  for (int w = 0; w < G / 8; ++w) {
    dw[w * kTileCols + c] = *slab_word<G>(s, w);
  }
  const uint16_t a_bits = *slab_alpha<G, F>(s);
  uint32_t zp = 8;
  if constexpr (F == PacketFormat::kNativeAsym) {
    const uint16_t neg = reinterpret_cast<const uint16_t*>(slab_zp_word<G>(s))[s.i];
    zp = static_cast<uint32_t>(static_cast<float>(__builtin_bit_cast(_Float16, neg)) * -1.0f);
  }
  reinterpret_cast<uint16_t*>(dst + QB)[c] = a_bits;
  reinterpret_cast<uint16_t*>(dst + QB)[kTileCols + c] = neg_alpha_zp_bits(a_bits, zp);
}

}  // namespace

namespace {

// Turns (256 values of K) per workgroup: up to 4, so that a row's scales are read by few
// workgroups, while at least 4 workgroups per CU remain.
template <int G, PacketFormat F>
hipError_t launch_pack(const void* q, const void* alpha, const void* offsets, void* packets, int n,
                       int k, hipStream_t stream) {
  const int tiles = n / kTileCols;
  const int turns = (k + kTurnK - 1) / kTurnK;
  int per = kMaxTurns;
  while (per > 1 && static_cast<long long>(tiles) * ((turns + per - 1) / per) < 1024) {
    per /= 2;
  }
  const dim3 grid(static_cast<unsigned int>((turns + per - 1) / per), static_cast<unsigned int>(tiles));
  hipLaunchKernelGGL((pack_kernel<G, F>), grid, dim3(kAuxThreads), 0, stream,
                     static_cast<const uint8_t*>(q), static_cast<const uint16_t*>(alpha), offsets,
                     static_cast<uint8_t*>(packets), k, k / G, per);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_pack_packets(const void* q, const void* alpha, const void* beta, void* packets,
                               int n, int k, int group_size, hipStream_t stream) {
  return group_size == 64
             ? launch_pack<64, PacketFormat::kArc>(q, alpha, beta, packets, n, k, stream)
             : launch_pack<128, PacketFormat::kArc>(q, alpha, beta, packets, n, k, stream);
}

hipError_t launch_dequant(const void* q, const void* alpha, const void* beta, void* out, int n,
                          int k, int group_size, hipStream_t stream) {
  const int words_per_row = k / 8;
  const size_t total = static_cast<size_t>(n) * words_per_row;
  const int num_groups = k / group_size;
  auto* qp = static_cast<const uint32_t*>(q);
  auto* ap = static_cast<const uint16_t*>(alpha);
  auto* bp = static_cast<const uint16_t*>(beta);
  auto* op = static_cast<uint4*>(out);
  if (group_size == 64) {
    hipLaunchKernelGGL(dequant_kernel<64>, dim3(blocks_for(total, kAuxThreads)), dim3(kAuxThreads), 0, stream,
                       qp, ap, bp, op, total, words_per_row, num_groups);
  } else {
    hipLaunchKernelGGL(dequant_kernel<128>, dim3(blocks_for(total, kAuxThreads)), dim3(kAuxThreads), 0, stream,
                       qp, ap, bp, op, total, words_per_row, num_groups);
  }
  return hipGetLastError();
}

hipError_t launch_dequant_packets(const void* packets, void* out, int n, int k, int group_size,
                                  hipStream_t stream) {
  const int num_groups = k / group_size;
  const dim3 grid(static_cast<unsigned int>((k + kTurnK - 1) / kTurnK),
                  static_cast<unsigned int>(n / kTileCols));
  auto* pp = static_cast<const uint8_t*>(packets);
  auto* op = static_cast<uint4*>(out);
  if (group_size == 64) {
    hipLaunchKernelGGL(dequant_packets_kernel<64>, grid, dim3(kAuxThreads), 0, stream, pp, op, k, num_groups);
  } else {
    hipLaunchKernelGGL(dequant_packets_kernel<128>, grid, dim3(kAuxThreads), 0, stream, pp, op, k, num_groups);
  }
  return hipGetLastError();
}

hipError_t launch_group_sums(const void* x, void* sums, int batch, int k, int group_size,
                             hipStream_t stream) {
  const int num_groups = k / group_size;
  const dim3 grid(static_cast<unsigned int>(batch), static_cast<unsigned int>(num_groups));
  auto* xp = static_cast<const uint32_t*>(x);
  auto* sp = static_cast<float*>(sums);
  if (group_size == 64) {
    hipLaunchKernelGGL(group_sums_kernel<64>, grid, dim3(64), 0, stream, xp, sp, k, num_groups);
  } else {
    hipLaunchKernelGGL(group_sums_kernel<128>, grid, dim3(64), 0, stream, xp, sp, k, num_groups);
  }
  return hipGetLastError();
}

hipError_t launch_reduce_partials(const void* partials, void* out, int batch, int n,
                                  int split_k_slices, hipStream_t stream) {
  const size_t total = static_cast<size_t>(batch) * n;
  hipLaunchKernelGGL(reduce_partials_kernel, dim3(blocks_for(total, kAuxThreads)), dim3(kAuxThreads), 0, stream,
                     static_cast<const float*>(partials), static_cast<uint16_t*>(out), total, split_k_slices);
  return hipGetLastError();
}


hipError_t launch_pack_native(const void* q, const void* alpha, const void* zero_points,
                              void* packets, int n, int k, int group_size, PacketFormat format,
                              hipStream_t stream) {
  const bool g64 = group_size == 64;
  if (format == PacketFormat::kNativeSym) {
    return g64 ? launch_pack<64, PacketFormat::kNativeSym>(q, alpha, zero_points, packets, n, k, stream)
               : launch_pack<128, PacketFormat::kNativeSym>(q, alpha, zero_points, packets, n, k, stream);
  }
  if (format == PacketFormat::kNativeAsym) {
    return g64 ? launch_pack<64, PacketFormat::kNativeAsym>(q, alpha, zero_points, packets, n, k, stream)
               : launch_pack<128, PacketFormat::kNativeAsym>(q, alpha, zero_points, packets, n, k, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_arc_to_native(const void* arc, void* native, int n, int k, int group_size,
                                PacketFormat format, void* bad_flag, hipStream_t stream) {
  const int ng = k / group_size;
  const dim3 grid(static_cast<unsigned int>(n / kTileCols), static_cast<unsigned int>(ng));
  auto* src = static_cast<const uint8_t*>(arc);
  auto* dst = static_cast<uint8_t*>(native);
  auto* bad = static_cast<uint32_t*>(bad_flag);
  const bool g64 = group_size == 64;
  if (format == PacketFormat::kNativeSym) {
    if (g64) hipLaunchKernelGGL((arc_to_native_kernel<64, PacketFormat::kNativeSym>), grid, dim3(kTileCols), 0, stream, src, dst, ng, bad);
    else hipLaunchKernelGGL((arc_to_native_kernel<128, PacketFormat::kNativeSym>), grid, dim3(kTileCols), 0, stream, src, dst, ng, bad);
  } else if (format == PacketFormat::kNativeAsym) {
    if (g64) hipLaunchKernelGGL((arc_to_native_kernel<64, PacketFormat::kNativeAsym>), grid, dim3(kTileCols), 0, stream, src, dst, ng, bad);
    else hipLaunchKernelGGL((arc_to_native_kernel<128, PacketFormat::kNativeAsym>), grid, dim3(kTileCols), 0, stream, src, dst, ng, bad);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_native_to_arc(const void* native, void* arc, int n, int k, int group_size,
                                PacketFormat format, hipStream_t stream) {
  const int ng = k / group_size;
  const dim3 grid(static_cast<unsigned int>(n / kTileCols), static_cast<unsigned int>(ng));
  auto* src = static_cast<const uint8_t*>(native);
  auto* dst = static_cast<uint8_t*>(arc);
  const bool g64 = group_size == 64;
  if (format == PacketFormat::kNativeSym) {
    if (g64) hipLaunchKernelGGL((native_to_arc_kernel<64, PacketFormat::kNativeSym>), grid, dim3(kTileCols), 0, stream, src, dst, ng);
    else hipLaunchKernelGGL((native_to_arc_kernel<128, PacketFormat::kNativeSym>), grid, dim3(kTileCols), 0, stream, src, dst, ng);
  } else if (format == PacketFormat::kNativeAsym) {
    if (g64) hipLaunchKernelGGL((native_to_arc_kernel<64, PacketFormat::kNativeAsym>), grid, dim3(kTileCols), 0, stream, src, dst, ng);
    else hipLaunchKernelGGL((native_to_arc_kernel<128, PacketFormat::kNativeAsym>), grid, dim3(kTileCols), 0, stream, src, dst, ng);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace fk
