// W4A16 GEMM over row tiles on the gfx950 matrix cores: 8-16 activation rows that the stream kernel
// does not take, 17 and more (batched serving, chunks of a prompt), over reference packets or native slabs.
//
// Above 32 rows, and under a fused neighbour, a first launch (w4a16_gemm_tile_prepare_kernel) writes the
// activations in the order the tiles read them: re-paired (x0,x4)(x1,x5)(x2,x6)(x3,x7) like the code
// words unpack, [32-row block][group][16-byte unit][row], so staging is a straight copy and every
// LDS access is 512 consecutive bytes per half wave; beside them the (row, group) sums. It applies
// the RMSNorm where one is fused, so that costs no pass of its own. Up to 32 plain rows the tiles
// stage the activations themselves: the launch costs 4-5 us there and the pairing little (32 rows,
// bf16 native: 28672 x 4096 23.6 -> 22.1 us, 4096 x 14336 18.9 -> 16.0, 10240 x 8192 21.1 -> 18.1,
// 4096 x 4096 12.9 -> 11.0).
//
// The GEMM's workgroup (8 waves) owns BM rows x BN columns. Each wave owns whole 32-column slices
// of the tile, reads their code words straight into registers (each word is unpacked once per
// wave and multiplied against all of the wave's rows; nothing but activations goes through LDS)
// and runs v_mfma_f32_32x32x16 on them: lane l holds column l % 32 and, by halves, 8 consecutive k.
//
//  * Codes unpack to 64 + q (fp16: the nibble lands on mantissa bits 4-7 of 0x5400) or 128 + q
//    (bf16: bits 0-3 of 0x4300), exact in the activation dtype, so bf16 activations are multiplied
//    as they are. Three shifts and four and-or per 8 codes.
//  * Per group, D = sum (bias + q) x in fp32 and y += alpha * D. What is left, per (row, group,
//    column), is (beta - bias * alpha) * S with S the group's activation sum: a product over the
//    groups, which the matrix cores take too, two groups per v_mfma_f32_32x32x16_bf16, both
//    factors split into three bf16 parts (24 bits; the eight largest of the nine products).
//  * Work split: a workgroup takes one tile, or one of its K splits where the tiles alone would
//    leave CUs idle (tile_shape); the last split to arrive adds the partial tiles in split order
//    (deterministic).
//  * The loop is bound by the SIMDs' issue: per wave and 128 k of a 64 x 64 block 34 MFMAs (32
//    cycles each) against about 200 VALU instructions (4 cycles each: 112 unpack, 64 scale), which
//    overlap only in part. Timestamps: 2.0 us per 128 x 256 x 128 chunk of the largest tile (1057
//    TFLOP/s over the loop at 8192 x 8192, 512 rows).
//
// Measured on MI355X against the 16-row tiles of w4a16_gemm_mfma.hip, which read and unpack the
// weights once per 16 rows: 10240 x 8192, 512 rows, bf16 native 256 -> 108 us; 4096 x 14336, 64
// rows 31.5 -> 23.5; 22016 x 4096, 33 rows, fp16 reference packets 34.8 -> 25.1. Of the last two
// about 5 us are the first launch; the 64-row one's seven K splits then meet in the fix-up, the 33-row
// one's 172 workgroups, one tile each, leave 84 CUs idle.
#include "w4a16_gemm_tile.h"

#include <cstdint>

namespace fk {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kBlockRows = 32;  // rows of an MFMA block

struct PrepareParams {
  const uint16_t* x;
  const uint16_t* gamma;
  uint4* xs;
  uint4* sums;
  uint32_t* counters;
  int n_counters;
  int M, K, NG;
  int quarters;  // native formats: windows take the slabs' quarter units
  float eps;
};

// A prepare workgroup takes 8 rows (a wave each) and 512 values of them.
constexpr int kPrepRows = 8;
constexpr int kPrepThreads = 64 * kPrepRows;
constexpr int kPrepUnits = 64;  // 16-byte units per row

__device__ __forceinline__ uint32_t bf16_bits_of(float f) { return float_to_bf16_bits(f); }

// The three bf16 parts of f: f = p0 + p1 + p2 to 24 bits.
__device__ __forceinline__ void bf16_parts(float f, uint32_t (&p)[3]) {
  p[0] = bf16_bits_of(f);
  f -= __builtin_bit_cast(float, p[0] << 16);
  p[1] = bf16_bits_of(f);
  f -= __builtin_bit_cast(float, p[1] << 16);
  p[2] = bf16_bits_of(f);
}

// round(gamma * round(x * inv_rms)) of a pair, in the activation dtype.
template <Act A>
__device__ __forceinline__ uint32_t prep_norm_pair(uint32_t xw, uint32_t gw, float inv) {
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const float x = act_bits_to_float<A>(static_cast<uint16_t>(xw >> (16 * i)));
    const float g = act_bits_to_float<A>(static_cast<uint16_t>(gw >> (16 * i)));
    const float xn = act_bits_to_float<A>(float_to_act_bits<A>(x * inv));
    r |= static_cast<uint32_t>(float_to_act_bits<A>(g * xn)) << (16 * i);
  }
  return r;
}

// Place of 8-value unit w of a group in the prepared activations: window v, half h at 2 v + h.
template <int G>
__device__ __forceinline__ int window_slot(int w, bool quarters) {
  constexpr int U = native_unit_words(G);
  return quarters ? 2 * (w / (2 * U) * U + w % U) + w / U % 2 : w;
}

// Rows are read along K (a wave a row) and written 128 bytes (8 rows) at a time, through LDS.
// kNorm: every workgroup first forms 1 / rms of its rows (fp32, the whole row, from L2).
template <int G, Act A, bool kNorm>
__global__ void __launch_bounds__(kPrepThreads) w4a16_gemm_tile_prepare_kernel(PrepareParams p) {
  constexpr int WR = G / 8;
  __shared__ u32x4_t turn[kPrepUnits * kPrepRows];
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63;
  const int r = tid >> 6;
  const int row0 = static_cast<int>(blockIdx.x) * kPrepRows;
  const bool live = row0 + r < p.M;
  const int units = p.K / 8;
  const int unit0 = static_cast<int>(blockIdx.y) * kPrepUnits;
  const u32x4_t* xr =
      reinterpret_cast<const u32x4_t*>(p.x + static_cast<size_t>(live ? row0 + r : 0) * p.K);
  if (blockIdx.x == 0 && blockIdx.y == 0) {
    for (int i = tid; i < p.n_counters; i += kPrepThreads) {
      p.counters[i] = 0;
    }
  }
  const int c = unit0 + lane;
  const bool in_k = c < units;
  u32x4_t v = xr[in_k ? c : 0];
  if constexpr (kNorm) {
    const u32x4_t gm = reinterpret_cast<const u32x4_t*>(p.gamma)[in_k ? c : 0];
    float ss = 0.0f;
    constexpr int kBatch = 8;
    for (int u0 = lane; u0 < units; u0 += 64 * kBatch) {
      u32x4_t w[kBatch];
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        w[i] = xr[min(u0 + 64 * i, units - 1)];
      }
#pragma unroll
      for (int i = 0; i < kBatch; ++i) {
        if (u0 + 64 * i < units) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const float lo = act_bits_to_float<A>(static_cast<uint16_t>(w[i][q]));
            const float hi = act_bits_to_float<A>(static_cast<uint16_t>(w[i][q] >> 16));
            ss = fmaf(lo, lo, ss);
            ss = fmaf(hi, hi, ss);
          }
        }
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      ss += __shfl_xor(ss, off);
    }
    const float inv = 1.0f / sqrtf(ss / static_cast<float>(p.K) + p.eps);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      v[q] = prep_norm_pair<A>(v[q], gm[q], inv);
    }
  }
  if (!live || !in_k) {
    v = u32x4_t{0u, 0u, 0u, 0u};
  }
  float s = 0.0f;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    s += act_bits_to_float<A>(static_cast<uint16_t>(v[q])) +
         act_bits_to_float<A>(static_cast<uint16_t>(v[q] >> 16));
  }
  // a group's WR units are WR consecutive lanes
  s = group_sum<WR>(s);
  const size_t block = static_cast<size_t>(row0 / kBlockRows) * p.NG;
  const int lrow0 = row0 % kBlockRows;
  if (in_k && c % WR == 0) {
    uint32_t q[3];
    bf16_parts(s, q);
    p.sums[(block + c / WR) * kBlockRows + lrow0 + r] =
        make_uint4(q[0] | (q[0] << 16), q[0] | (q[1] << 16), q[1] | (q[1] << 16), q[2] | (q[2] << 16));
  }
  const uint4 xp = pair_activations(make_uint4(v.x, v.y, v.z, v.w));
  // the slot of a row is swizzled by the unit, so 8 consecutive lanes use all LDS banks both ways
  turn[lane * kPrepRows + (r ^ (lane & 7))] = u32x4_t{xp.x, xp.y, xp.z, xp.w};
  __syncthreads();
  const int ou = tid / kPrepRows;
  const int orow = tid % kPrepRows;
  const int oc = unit0 + ou;
  if (oc < units) {
    const u32x4_t o = turn[ou * kPrepRows + (orow ^ (ou & 7))];
    const int slot = window_slot<G>(oc % WR, p.quarters != 0);
    *reinterpret_cast<u32x4_t*>(p.xs + (block + oc / WR) * (WR * kBlockRows) + slot * kBlockRows +
                                lrow0 + orow) = o;
  }
}

struct TileParams {
  const uint16_t* x;  // kDirect: the activations [M, K]
  const u32x4_t* xs;
  const u32x4_t* sums;
  const uint8_t* packets;
  uint16_t* out;
  float* partials;
  uint32_t* counters;
  int M, N, K, NG, mtiles, tile_units, per, splits;
  int grid, xcd_remap;
  int vector_out;  // out rows are 16-byte aligned
};

// RS x CS blocks of 32 x 32 per wave; WR x WC waves over the tile's rows and columns, WP wave
// groups over K. A chunk is 128 k of each wave group (one LDS buffer), a unit two chunks.
template <int G_, int RS_, int CS_, int WR_, int WC_, int WP_>
struct Tile {
  static constexpr int G = G_, RS = RS_, CS = CS_, WR = WR_, WC = WC_, WP = WP_;
  static_assert(WR * WC * WP == kTileWaves, "eight waves");
  static constexpr int kWindows = G / 16;         // MFMAs per group and block
  static constexpr int kWaveGroups = 128 / G;     // groups of a wave per chunk
  static constexpr int kChunkGroups = kWaveGroups * WP;
  static constexpr int kUnitGroups = 2 * kChunkGroups;
  static constexpr int kBlocks = RS * WR;         // 32-row blocks of the tile
  static constexpr int kBM = kBlocks * kBlockRows;
  static constexpr int kBN = CS * WC * kSliceCols;
  static constexpr int kSlices = CS * WC;
  static constexpr int kGroupUnits = G / 8 * kBlockRows;  // 16-byte units per (group, block)
  static constexpr int kXUnits = kChunkGroups * kBlocks * kGroupUnits;
  static constexpr int kSUnits = kChunkGroups * kBlocks * kBlockRows;
  static constexpr int kBufUnits = kXUnits + kSUnits;
  static constexpr int kXPer = kXUnits / kTileThreads;
  static constexpr int kOutPitch = kBN + 8;       // 16-bit elements per staged output row
  static constexpr size_t kLdsBytes = 2 * static_cast<size_t>(kBufUnits) * 16 + 16;
  static constexpr int kAcc = RS * CS * 16;       // accumulators per lane
  static constexpr int kSlotFloats = kBM * kBN;   // a partial tile
  static_assert(kXUnits % kTileThreads == 0 && kSUnits <= kTileThreads, "whole staging passes");
  static_assert(static_cast<size_t>(kBM) * kOutPitch * 2 <= 2 * static_cast<size_t>(kBufUnits) * 16,
                "the output tile fits the buffers");
};

// One group of one slice for a lane: its column's code words of every window, alpha and beta.
template <int G>
struct SliceRegs {
  uint32_t w[G / 16];
  uint32_t alpha;
  uint32_t beta;  // kArc: beta, kNativeAsym: -zp, as fp16 bits
};

// Byte offsets of a lane in a group's slab (native) or packet (kArc, of 32-column quarter 0):
// words of its window 0, and its alpha. Column lane % 32, half h = lane / 32. Native window v
// holds word U (2 (v / U) + h) + v % U of the group (U = G / 32: the layout's quarter units), kArc
// word 2 v + h; w4a16_gemm_tile_prepare_kernel orders the activations alike.
template <int G, PacketFormat F>
__device__ __forceinline__ uint32_t lane_words(int lane) {
  const int c = lane % 32;
  const int h = lane / 32;
  if (F == PacketFormat::kArc) {
    return (h * kTileCols + c) * 4;
  }
  return (16 * h + c % 16) * 16 + c / 16 * (G == 128 ? 1024 : 8);
}
template <int G, PacketFormat F>
__device__ __forceinline__ uint32_t lane_scale(int lane) {
  const int c = lane % 32;
  return F == PacketFormat::kArc
             ? kTileCols * G / 2 + c * 2
             : native_record_offset(G) + native_record_bytes(F) * (c % 16) + 2 * (c / 16);
}

// Plain loads: row tiles share the weights through the caches, and a 128-byte line that two slabs
// share is kept for the second. (Non-temporal ones were 3-5 % slower in the 32-row tile, 5-8 % at G64
// over native slabs, and 4 % in the 64-row tile with one row tile to 10 % with 9-12; 370 rows, 4864 x
// 3328 G128: 31.5 -> 27.1 us.)
template <int G, PacketFormat F>
__device__ __forceinline__ void load_slice(SliceRegs<G>& r, const uint8_t* group, uint32_t words,
                                           uint32_t scale) {
  const auto u16 = [](const uint8_t* p) -> uint32_t { return *reinterpret_cast<const uint16_t*>(p); };
  if constexpr (F == PacketFormat::kArc) {
#pragma unroll
    for (int v = 0; v < G / 16; ++v) {
      r.w[v] = *reinterpret_cast<const uint32_t*>(group + words + v * 2 * kTileCols * 4);
    }
    r.beta = u16(group + scale + kTileCols * 2);
  } else if constexpr (G == 128) {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x4_t v = *reinterpret_cast<const u32x4_t*>(group + words + s * 512);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        r.w[4 * s + j] = v[j];
      }
    }
  } else {
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const u32x2_t v = *reinterpret_cast<const u32x2_t*>(group + words + s * 512);
      r.w[2 * s] = v[0];
      r.w[2 * s + 1] = v[1];
    }
  }
  r.alpha = u16(group + scale);
  if constexpr (F == PacketFormat::kNativeAsym) {
    r.beta = u16(group + scale + 4);
  }
}

// Code word -> 64 + q (fp16) or 128 + q (bf16), in the order (k0,k4)(k1,k5)(k2,k6)(k3,k7).
template <Act A>
__device__ __forceinline__ u32x4_t unpack_codes(uint32_t w, uint32_t mask) {
  u32x4_t v;
  if constexpr (A == Act::kF16) {
    v.x = ((w << 4) & mask) | 0x54005400u;
    v.y = (w & mask) | 0x54005400u;
    v.z = ((w >> 4) & mask) | 0x54005400u;
    v.w = ((w >> 8) & mask) | 0x54005400u;
  } else {
    v.x = (w & mask) | 0x43004300u;
    v.y = ((w >> 4) & mask) | 0x43004300u;
    v.z = ((w >> 8) & mask) | 0x43004300u;
    v.w = ((w >> 12) & mask) | 0x43004300u;
  }
  return v;
}
template <Act A>
constexpr float kUnpackBias = A == Act::kF16 ? 64.0f : 128.0f;
template <Act A>
constexpr uint32_t kUnpackMask = A == Act::kF16 ? 0x00f000f0u : 0x000f000fu;

template <Act A>
__device__ __forceinline__ float16_t mfma(u32x4_t a, u32x4_t b, float16_t c) {
  if constexpr (A == Act::kF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(half8_t, a),
                                                  __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                   __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
  }
}

template <Act A>
__device__ __forceinline__ uint32_t silu_mul_pair(uint32_t gw, uint32_t uw) {
  uint32_t o = 0;
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const float g = act_bits_to_float<A>(static_cast<uint16_t>(gw >> (16 * s)));
    const float u = act_bits_to_float<A>(static_cast<uint16_t>(uw >> (16 * s)));
    const float act = act_bits_to_float<A>(float_to_act_bits<A>(g / (1.0f + expf(-g))));
    o |= static_cast<uint32_t>(float_to_act_bits<A>(act * u)) << (16 * s);
  }
  return o;
}

// The activations of unit w of group g of a row, paired (values i and i + 4).
template <int G, PacketFormat F, bool kDirect>
__device__ __forceinline__ u32x4_t paired_unit(const TileParams& p, int row, int g, int w) {
  constexpr int WR = G / 8;
  if constexpr (kDirect) {
    const u32x4_t v =
        reinterpret_cast<const u32x4_t*>(p.x + static_cast<size_t>(row) * p.K)[g * WR + w];
    const uint4 q = pair_activations(make_uint4(v.x, v.y, v.z, v.w));
    return u32x4_t{q.x, q.y, q.z, q.w};
  } else {
    const u32x4_t* xr =
        p.xs + static_cast<size_t>(row / kBlockRows) * p.NG * (WR * kBlockRows) + row % kBlockRows;
    return xr[(g * WR + window_slot<G>(w, is_native(F))) * kBlockRows];
  }
}

__device__ __forceinline__ bool has_non_finite_bf16(uint32_t pair) {
  return (pair & 0x7f80u) == 0x7f80u || (pair & 0x7f800000u) == 0x7f800000u;
}

// Whether a row of bf16 activations holds neither infinities nor NaN (asked by a whole wave).
template <int G, PacketFormat F, bool kDirect>
__device__ bool finite_row(const TileParams& p, int row, int lane) {
  constexpr int WR = G / 8;
  bool bad = false;
#pragma unroll 4
  for (int u = lane; u < p.NG * WR; u += 64) {
    const u32x4_t x = paired_unit<G, F, kDirect>(p, row, u / WR, u % WR);
    bad |= has_non_finite_bf16(x[0]) || has_non_finite_bf16(x[1]) || has_non_finite_bf16(x[2]) ||
           has_non_finite_bf16(x[3]);
  }
  return !__any(bad);
}

// One output in plain fp32 arithmetic on activations 2^-64 times smaller, by a whole wave: for bf16
// outputs that came out infinite or NaN from finite activations. The tile's accumulators hold sums of
// (128 + q) x, which overflow from |x| of about 2^113; the result itself may still be finite. (By one
// lane an output, and for rows that hold a NaN too, one such row of 64, 28672 x 4096, made a call of 28
// us take 1556; now 32.)
template <int G, PacketFormat F, bool kDirect>
__device__ uint16_t plain_bf16_output(const TileParams& p, int row, int col, int lane) {
  constexpr int WR = G / 8;
  constexpr int U = native_unit_words(G);
  constexpr int kStride = format_packet_stride(G, F);
  const uint8_t* base =
      p.packets + static_cast<size_t>(is_native(F) ? col / kSliceCols : col / kTileCols) * p.NG * kStride;
  const int c = is_native(F) ? col % kSliceCols : col % kTileCols;
  float y = 0.0f;
#pragma unroll 2
  for (int u = lane; u < p.NG * WR; u += 64) {
    const int g = u / WR;
    const int w = u % WR;
    const uint8_t* group = base + static_cast<size_t>(g) * kStride;
    const u32x4_t x = paired_unit<G, F, kDirect>(p, row, g, w);
    const int at = is_native(F) ? native_word_offset(G, c / 16, w / U, c % 16, w % U)
                                : (w * kTileCols + c) * 4;
    const uint32_t word = *reinterpret_cast<const uint32_t*>(group + at);
    float dot = 0.0f;
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float lo = bf16_bits_to_float(static_cast<uint16_t>(x[i])) * 0x1p-64f;
      const float hi = bf16_bits_to_float(static_cast<uint16_t>(x[i] >> 16)) * 0x1p-64f;
      dot = fmaf(static_cast<float>((word >> (4 * i)) & 15u), lo, dot);
      dot = fmaf(static_cast<float>((word >> (4 * i + 16)) & 15u), hi, dot);
      sum += lo + hi;
    }
    uint16_t a_bits = 0;
    float beta = 0.0f;
    if constexpr (is_native(F)) {
      const uint8_t* record = group + native_record_offset(G) + native_record_bytes(F) * (c % 16) + 2 * (c / 16);
      a_bits = *reinterpret_cast<const uint16_t*>(record);
      if constexpr (F == PacketFormat::kNativeAsym) {
        const uint16_t neg = *reinterpret_cast<const uint16_t*>(record + 4);
        beta = static_cast<float>(__builtin_bit_cast(_Float16, a_bits) * __builtin_bit_cast(_Float16, neg));
      } else {
        beta = -8.0f * half_bits_to_float(a_bits);
      }
    } else {
      const uint16_t* scales = reinterpret_cast<const uint16_t*>(group + kTileCols * G / 2);
      a_bits = scales[c];
      beta = half_bits_to_float(scales[kTileCols + c]);
    }
    y = fmaf(half_bits_to_float(a_bits), dot, y);
    y = fmaf(beta, sum, y);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    y += __shfl_xor(y, off);
  }
  return float_to_bf16_bits(y * 0x1p64f);
}

// kDirect: the workgroup stages the activations itself, from x, instead of copying prepared ones: a
// wave reads a row's 512 values of the chunk, pairs them and adds up the groups' sums, a row per
// window between the MFMAs. LDS rows are swizzled by the unit's place (consecutive lanes store
// consecutive units of one row, 512 bytes apart).
template <class T, Act A, PacketFormat F, bool kSilu, bool kDirect>
__global__ void __launch_bounds__(kTileThreads, 2) w4a16_gemm_tile_kernel(TileParams p) {
  constexpr int G = T::G;
  constexpr int RS = T::RS;
  constexpr int CS = T::CS;
  constexpr int KG = T::kWaveGroups;
  constexpr int kStride = format_packet_stride(G, F);
  extern __shared__ u32x4_t lds[];
  int* last_flag = reinterpret_cast<int*>(lds + 2 * T::kBufUnits);
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63;
  const int half = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wp = wave / (T::WR * T::WC);
  const int wrc = wave % (T::WR * T::WC);
  const int wr = wrc / T::WC;
  const int wc = wrc % T::WC;
  const uint32_t mask = vgpr_constant(kUnpackMask<A>);
  int b = static_cast<int>(blockIdx.x);
  b = p.xcd_remap != 0 ? (b & 7) * p.xcd_remap + (b >> 3) : b;
  // Workgroup order: row tiles fastest (they read the same weights at once), then the K splits of
  // a column tile (they meet in the fix-up).
  const int mt = b % p.mtiles;
  const int split = b / p.mtiles % p.splits;
  const int ct = b / p.mtiles / p.splits;
  const int u_begin = split * p.per;
  const int u_end = min(p.tile_units, u_begin + p.per);
  const int n_slices = p.N / kSliceCols;
  const uint32_t words = lane_words<G, F>(lane);

  // Group 0 of the tile's first row block and of the wave's slices (kSilu: the tile's first half
  // is gate columns, its second the same up columns; past the last slice, the last).
  const int block0 = mt * T::kBlocks;
  const u32x4_t* const x_tile = p.xs + static_cast<size_t>(block0) * p.NG * T::kGroupUnits;
  const u32x4_t* const s_tile = p.sums + static_cast<size_t>(block0) * p.NG * kBlockRows;
  const uint8_t* slice0[CS];
  uint32_t scale[CS];
#pragma unroll
  for (int j = 0; j < CS; ++j) {
    const int ls = wc * CS + j;
    int slice;
    if constexpr (kSilu) {
      constexpr int kHalf = T::kSlices / 2;
      slice = ls < kHalf ? ct * kHalf + ls : n_slices / 2 + ct * kHalf + (ls - kHalf);
    } else {
      slice = min(ct * T::kSlices + ls, n_slices - 1);
    }
    scale[j] = lane_scale<G, F>(lane);
    if constexpr (F == PacketFormat::kArc) {
      // a quarter of a packet: its words are 4 bytes a column, its scales 2
      const int quarter = slice % kSlicesPerTile;
      slice0[j] = p.packets + static_cast<size_t>(slice / kSlicesPerTile) * p.NG * kStride +
                  quarter * (kSliceCols * 4);
      scale[j] -= quarter * (kSliceCols * 2);
    } else {
      slice0[j] = p.packets + static_cast<size_t>(slice) * p.NG * kStride;
    }
  }
  SliceRegs<G> wreg[2][KG][CS];
  u32x4_t xreg[T::kXPer];
  u32x4_t sreg;
  // (past the last group, in a short last unit: that group again)
  auto load_weights = [&](int g0, SliceRegs<G> (&w)[KG][CS]) {
#pragma unroll
    for (int kk = 0; kk < KG; ++kk) {
      const int g = min(g0 + wp * KG + kk, p.NG - 1);
#pragma unroll
      for (int j = 0; j < CS; ++j) {
        load_slice<G, F>(w[kk][j], slice0[j] + static_cast<size_t>(g) * kStride, words, scale[j]);
      }
    }
  };
  auto stage_load = [&](int g0) {
    constexpr int kPerPass = kTileThreads / T::kGroupUnits;  // (group, block)s per pass: 1 or 2
    const int sub = wave / (T::kGroupUnits / 64);
    const uint32_t idx = static_cast<uint32_t>(tid % T::kGroupUnits);
#pragma unroll
    for (int it = 0; it < T::kXPer; ++it) {
      const int q = it * kPerPass + sub;
      const int g = min(g0 + q / T::kBlocks, p.NG - 1);
      const u32x4_t* base = x_tile + (static_cast<size_t>(q % T::kBlocks) * p.NG + g) * T::kGroupUnits;
      xreg[it] = base[idx];
    }
    const uint32_t v = static_cast<uint32_t>(tid % T::kSUnits);
    const uint32_t q = v / kBlockRows;
    const uint32_t g = static_cast<uint32_t>(min(g0 + static_cast<int>(q / T::kBlocks), p.NG - 1));
    sreg = s_tile[((q % T::kBlocks) * p.NG + g) * kBlockRows + v % kBlockRows];
  };
  auto stage_store = [&](u32x4_t* buf) {
#pragma unroll
    for (int it = 0; it < T::kXPer; ++it) {
      buf[it * kTileThreads + tid] = xreg[it];
    }
    // by every thread, more than once where there are fewer units: no branch in the loop
    buf[T::kXUnits + tid % T::kSUnits] = sreg;
  };
  // kDirect: lane l takes unit l of the chunk's 64 units of a row (a chunk of four wave groups is
  // 512 values), the wave rows wave, wave + 8, ... of the tile; rows and units past the end repeat
  // the last one.
  constexpr int WR = G / 8;
  static_assert(!kDirect || (T::WP == 4 && T::kXPer == T::kBM / kTileWaves), "a row per wave and pass");
  const int d_slot = window_slot<G>(lane % WR, is_native(F));
  const uint32_t d_store = static_cast<uint32_t>(
      (lane / WR * T::kBlocks * WR + d_slot) * kBlockRows + (wave ^ (d_slot & 7)));
  float d_sum = 0.0f;  // of the row of pass lane % kXPer
  auto direct_load = [&](int g0, int it) {
    const int row = min(mt * T::kBM + it * kTileWaves + wave, p.M - 1);
    const uint32_t unit = static_cast<uint32_t>(min(g0 * WR + lane, p.NG * WR - 1));
    xreg[it] = reinterpret_cast<const u32x4_t*>(p.x + static_cast<size_t>(row) * p.K)[unit];
  };
  auto direct_store = [&](u32x4_t* buf, int it) {
    const u32x4_t v = xreg[it];
    const uint4 xp = pair_activations(make_uint4(v.x, v.y, v.z, v.w));
    float s = 0.0f;
    if constexpr (A == Act::kF16) {
      constexpr uint32_t kOnes = 0x3c003c00u;
      s = dot2<A>(xp.w, kOnes, dot2<A>(xp.z, kOnes, dot2<A>(xp.y, kOnes, dot2<A>(xp.x, kOnes, s))));
    } else {
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        s += bf16_bits_to_float(static_cast<uint16_t>(v[q])) +
             __builtin_bit_cast(float, v[q] & 0xffff0000u);
      }
    }
    s = group_sum<WR>(s);
    d_sum = lane % T::kXPer == it ? s : d_sum;
    const int row8 = it * kTileWaves;  // of the pass; the wave's row is row8 + wave
    buf[d_store + (row8 / kBlockRows * WR * kBlockRows + row8 % kBlockRows)] =
        u32x4_t{xp.x, xp.y, xp.z, xp.w};
  };
  // The sums of the wave's rows, one (row, group) a lane: lane % kXPer is the pass (lanes that
  // share one write the same values).
  auto direct_sums = [&](u32x4_t* buf) {
    const int it = lane % T::kXPer;
    uint32_t q[3];
    bf16_parts(d_sum, q);
    const int row = it * kTileWaves + wave;
    buf[T::kXUnits + (lane / WR * T::kBlocks + row / kBlockRows) * kBlockRows + row % kBlockRows] =
        u32x4_t{q[0] | (q[0] << 16), q[0] | (q[1] << 16), q[1] | (q[1] << 16), q[2] | (q[2] << 16)};
  };
  auto stage_load_all = [&](int g0) {
    if constexpr (kDirect) {
#pragma unroll
      for (int it = 0; it < T::kXPer; ++it) {
        direct_load(g0, it);
      }
    } else {
      stage_load(g0);
    }
  };
  auto stage_store_all = [&](u32x4_t* buf) {
    if constexpr (kDirect) {
#pragma unroll
      for (int it = 0; it < T::kXPer; ++it) {
        direct_store(buf, it);
      }
      direct_sums(buf);
    } else {
      stage_store(buf);
    }
  };

  float16_t y[RS][CS] = {};
  stage_load_all(u_begin * T::kUnitGroups);
  load_weights(u_begin * T::kUnitGroups, wreg[0]);
  stage_store_all(lds);
  stage_load_all(u_begin * T::kUnitGroups + T::kChunkGroups);
  load_weights(u_begin * T::kUnitGroups + T::kChunkGroups, wreg[1]);
  __syncthreads();
  const u32x4_t* x_lane = lds + wp * KG * (T::kBlocks * T::kGroupUnits) +
                          wr * RS * T::kGroupUnits + (kDirect ? 0 : lane);
  // kDirect: a window's place in LDS is 64 units, half h's 32 rows second, the row swizzled by the
  // place, which repeats every four windows.
  uint32_t x_swizzled[4];
  if constexpr (kDirect) {
#pragma unroll
    for (int z = 0; z < 4; ++z) {
      x_swizzled[z] = half * kBlockRows + ((lane & 31) ^ (2 * z + half));
    }
  }
  const u32x4_t* s_lane = lds + T::kXUnits + (wp * KG * T::kBlocks + wr * RS) * kBlockRows + (lane & 31);
  for (int u = u_begin; u < u_end; ++u) {
    // Past the last unit the loads read group 0, in bounds and used by nobody.
    const int g_next = u + 1 < u_end ? (u + 1) * T::kUnitGroups : 0;
    float b_eff[CS];  // half 0: a pair's even group, half 1: its odd one
    u32x4_t sums[RS];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      // The next chunk's activations, loaded a chunk ago, into the other buffer; then the loads of
      // the chunk after it. All loads are unconditional: a branch around them would make the
      // compiler wait for every load in flight where the paths join.
      u32x4_t* other = lds + (h ^ 1) * T::kBufUnits;
      if constexpr (!kDirect) {
        stage_store(other);
        stage_load(g_next + h * T::kChunkGroups);
      }
      const u32x4_t* xg = x_lane + h * T::kBufUnits;
      const u32x4_t* sg = s_lane + h * T::kBufUnits;
      const int g_wave = u * T::kUnitGroups + h * T::kChunkGroups + wp * KG;
      // The activations of window w (over the chunk's groups) are read kAhead windows early.
      constexpr int kAll = KG * T::kWindows;
      constexpr int kAhead = RS * CS >= 4 ? 1 : 2;
      u32x4_t a[kAhead + 1][RS];
      auto read_window = [&](int w) {
        const int off = (w / T::kWindows) * (T::kBlocks * T::kGroupUnits) + w % T::kWindows * 64;
#pragma unroll
        for (int i = 0; i < RS; ++i) {
          if constexpr (kDirect) {
            a[w % (kAhead + 1)][i] = (xg + x_swizzled[w % 4])[off + i * T::kGroupUnits];
          } else {
            a[w % (kAhead + 1)][i] = xg[off + i * T::kGroupUnits];
          }
        }
      };
#pragma unroll
      for (int w = 0; w < kAhead; ++w) {
        read_window(w);
      }
      float16_t d[RS][CS];
#pragma unroll
      for (int w = 0; w < kAll; ++w) {
        const int kk = w / T::kWindows;
        const int v = w % T::kWindows;
        const bool odd = (h * KG + kk) % 2 == 1;
        if (w + kAhead < kAll) {
          read_window(w + kAhead);
        }
        if (v == 0) {
          const float16_t zero = {};
#pragma unroll
          for (int i = 0; i < RS; ++i) {
#pragma unroll
            for (int j = 0; j < CS; ++j) {
              d[i][j] = zero;
            }
          }
        }
        if (v == T::kWindows - 1) {
#pragma unroll
          for (int i = 0; i < RS; ++i) {
            const u32x4_t got = sg[(kk * T::kBlocks + i) * kBlockRows];
            sums[i] = !odd || half ? got : sums[i];
          }
        }
#pragma unroll
        for (int j = 0; j < CS; ++j) {
          const u32x4_t q = unpack_codes<A>(wreg[h][kk][j].w[v], mask);
#pragma unroll
          for (int i = 0; i < RS; ++i) {
            d[i][j] = mfma<A>(a[w % (kAhead + 1)][i], q, d[i][j]);
          }
        }
        if constexpr (kDirect) {
          if (w < T::kXPer) {
            direct_store(other, w);
            direct_load(g_next + h * T::kChunkGroups, w);
          }
          if (w == T::kXPer - 1) {
            direct_sums(other);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (v != T::kWindows - 1) {
          continue;
        }
        // the group's end
        const bool live = g_wave + kk < p.NG;  // a short last unit re-reads its last group
#pragma unroll
        for (int j = 0; j < CS; ++j) {
          const SliceRegs<G>& wr_ = wreg[h][kk][j];
          const uint16_t a_bits = static_cast<uint16_t>(wr_.alpha);
          const float alpha = live ? half_bits_to_float(a_bits) : 0.0f;
          float beta;
          if constexpr (F == PacketFormat::kNativeSym) {
            beta = -8.0f * alpha;
          } else if constexpr (F == PacketFormat::kNativeAsym) {
            const _Float16 prod = __builtin_bit_cast(_Float16, a_bits) *
                                  __builtin_bit_cast(_Float16, static_cast<uint16_t>(wr_.beta));
            beta = live ? static_cast<float>(prod) : 0.0f;
          } else {
            beta = live ? half_bits_to_float(static_cast<uint16_t>(wr_.beta)) : 0.0f;
          }
          const float eff = fmaf(-kUnpackBias<A>, alpha, beta);
          b_eff[j] = !odd || half ? eff : b_eff[j];
#pragma unroll
          for (int i = 0; i < RS; ++i) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              y[i][j][r] = fmaf(alpha, d[i][j][r], y[i][j][r]);
            }
            // here, and not sunk to the next group: both groups' d would then be live at once
            asm volatile("" : "+v"(y[i][j]));
          }
        }
        if (odd) {
#pragma unroll
          for (int j = 0; j < CS; ++j) {
            uint32_t q[3];
            bf16_parts(b_eff[j], q);
            const u32x4_t bq = {q[0] | (q[1] << 16), q[2] | (q[0] << 16), q[1] | (q[2] << 16),
                                q[0] | (q[1] << 16)};
#pragma unroll
            for (int i = 0; i < RS; ++i) {
              y[i][j] = mfma<Act::kBF16>(sums[i], bq, y[i][j]);
            }
          }
        }
      }
      load_weights(g_next + h * T::kChunkGroups, wreg[h]);
      __builtin_amdgcn_sched_barrier(0);
      __syncthreads();
    }
  }

  // Every lane's share of the tile's sums: the wave groups' accumulators are added through LDS, wave
  // group wp taking accumulators kPer * wp .. of its block column.
  constexpr int kPer = T::kAcc / T::WP;
  constexpr int kWaves1 = T::WR * T::WC;
  float v[kPer];
  if constexpr (T::WP > 1) {
    float* all = reinterpret_cast<float*>(lds) + lane;
    static_assert(static_cast<size_t>(kTileWaves) * T::kAcc * 256 <= 2 * static_cast<size_t>(T::kBufUnits) * 16,
                  "all accumulators fit the buffers");
#pragma unroll
    for (int e = 0; e < T::kAcc; ++e) {
      all[(wave * T::kAcc + e) * 64] = y[e / (16 * CS)][e / 16 % CS][e % 16];
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      v[i] = all[(wrc * T::kAcc + wp * kPer + i) * 64];
#pragma unroll
      for (int q = 1; q < T::WP; ++q) {
        v[i] += all[((q * kWaves1 + wrc) * T::kAcc + wp * kPer + i) * 64];
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < T::kAcc; ++e) {
      v[e] = y[e / (16 * CS)][e / 16 % CS][e % 16];
    }
  }
  if (p.splits > 1) {
    // Partial tile: agent-scope stores, complete before the counter is bumped; the last of the
    // tile's workgroups to arrive reads all of them back and adds them in split order.
    const int tile = ct * p.mtiles + mt;
    float* slots = p.partials + static_cast<size_t>(tile) * p.splits * T::kSlotFloats +
                   (wrc * T::kAcc + wp * kPer) * 64 + lane;
    float* mine = slots + static_cast<size_t>(split) * T::kSlotFloats;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      __hip_atomic_store(mine + i * 64, v[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
    __syncthreads();
    if (tid == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(&p.counters[tile], 1u, __ATOMIC_RELAXED,
                                                   __HIP_MEMORY_SCOPE_AGENT);
      *last_flag = prev == static_cast<uint32_t>(p.splits - 1) ? 1 : 0;
    }
    __syncthreads();
    if (*last_flag == 0) {
      return;
    }
    if (tid == 0) {
      __hip_atomic_store(&p.counters[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    constexpr int kBatch = kPer <= 16 ? 4 : 1;  // splits whose partials are in flight at once
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      v[i] = 0.0f;
    }
    for (int s0 = 0; s0 < p.splits; s0 += kBatch) {
      float got[kBatch][kPer];
#pragma unroll
      for (int q = 0; q < kBatch; ++q) {
        const float* theirs = slots + static_cast<size_t>(min(s0 + q, p.splits - 1)) * T::kSlotFloats;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
          got[q][i] = __hip_atomic_load(theirs + i * 64, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
#pragma unroll
      for (int q = 0; q < kBatch; ++q) {
        if (s0 + q < p.splits) {
#pragma unroll
          for (int i = 0; i < kPer; ++i) {
            v[i] += got[q][i];
          }
        }
      }
    }
  }
  __syncthreads();
  uint16_t* tile16 = reinterpret_cast<uint16_t*>(lds);
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int e = wp * kPer + i;
    const int r = e % 16;
    const int row = (wr * RS + e / (16 * CS)) * kBlockRows + 8 * (r / 4) + 4 * half + r % 4;
    const int col = (wc * CS + e / 16 % CS) * kSliceCols + (lane & 31);
    tile16[row * T::kOutPitch + col] = float_to_act_bits<A>(v[i]);
  }
  __syncthreads();
  const int row0 = mt * T::kBM;
  const int out_n = kSilu ? p.N / 2 : p.N;
  constexpr int kCols = kSilu ? T::kBN / 2 : T::kBN;
  const int col0 = ct * kCols;
  int asked_row = -1;  // the last row that finite_row was asked about, and its answer
  bool asked_finite = false;
  static_assert(T::kBM * (kCols / 8) % 64 == 0, "whole waves");
  for (int e = tid; e < T::kBM * (kCols / 8); e += kTileThreads) {
    const int row = e / (kCols / 8);
    const int c = e % (kCols / 8) * 8;
    const bool live = row0 + row < p.M && col0 + c < out_n;
    auto outputs = [&](int tile_col, int col) {
      u32x4_t o = *reinterpret_cast<const u32x4_t*>(tile16 + row * T::kOutPitch + tile_col);
      if constexpr (A == Act::kBF16) {
        const bool bad = live && (has_non_finite_bf16(o[0]) || has_non_finite_bf16(o[1]) ||
                                  has_non_finite_bf16(o[2]) || has_non_finite_bf16(o[3]));
        // by the whole wave, one lane's outputs after another's
        for (uint64_t todo = __ballot(bad); todo != 0; todo &= todo - 1) {
          const int of = __builtin_ctzll(todo);
          const int of_row = __builtin_amdgcn_readlane(row, of);
          const int of_col = __builtin_amdgcn_readlane(col, of);
          uint16_t* at = tile16 + of_row * T::kOutPitch + __builtin_amdgcn_readlane(tile_col, of);
          if (of_row != asked_row) {
            asked_row = of_row;
            asked_finite = finite_row<G, F, kDirect>(p, row0 + of_row, lane);
          }
          if (!asked_finite) {
            continue;
          }
#pragma unroll 1
          for (int q = 0; q < 8; ++q) {
            if ((at[q] & 0x7f80u) == 0x7f80u) {
              at[q] = plain_bf16_output<G, F, kDirect>(p, row0 + of_row, of_col + q, lane);
            }
          }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (bad) {
          o = *reinterpret_cast<const u32x4_t*>(tile16 + row * T::kOutPitch + tile_col);
        }
      }
      return o;
    };
    u32x4_t o = outputs(c, col0 + c);
    if constexpr (kSilu) {
      const u32x4_t up = outputs(kCols + c, p.N / 2 + col0 + c);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        o[q] = silu_mul_pair<A>(o[q], up[q]);
      }
    }
    if (!live) {
      continue;
    }
    uint16_t* dst = p.out + static_cast<size_t>(row0 + row) * out_n + col0 + c;
    if (p.vector_out) {
      *reinterpret_cast<u32x4_t*>(dst) = o;
    } else {
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        dst[q] = static_cast<uint16_t>(o[q / 2] >> (16 * (q % 2)));
      }
    }
  }
}

// Tile configurations by their rows.
template <int G>
using Tile32 = Tile<G, 1, 2, 1, 2, 4>;   // 32 x 128
template <int G>
using Tile64 = Tile<G, 2, 2, 1, 2, 4>;   // 64 x 128
template <int G>
using Tile128 = Tile<G, 2, 2, 2, 4, 1>;  // 128 x 256

template <class T, Act A, PacketFormat F, bool kSilu, bool kDirect = false>
hipError_t launch_tile(const TileParams& p, hipStream_t stream) {
  hipLaunchKernelGGL((w4a16_gemm_tile_kernel<T, A, F, kSilu, kDirect>), dim3(p.grid), dim3(kTileThreads),
                     T::kLdsBytes, stream, p);
  return hipGetLastError();
}

template <int G, Act A, PacketFormat F>
hipError_t launch_typed(const TileLaunch& l, const TileShape& s, hipStream_t stream) {
  char* ws = static_cast<char*>(l.workspace);
  TileParams p;
  p.x = static_cast<const uint16_t*>(l.x);
  p.xs = reinterpret_cast<const u32x4_t*>(ws + s.xs);
  p.sums = reinterpret_cast<const u32x4_t*>(ws + s.sums);
  p.packets = static_cast<const uint8_t*>(l.packets);
  p.out = static_cast<uint16_t*>(l.out);
  p.partials = reinterpret_cast<float*>(ws + s.partials);
  p.counters = reinterpret_cast<uint32_t*>(ws);
  p.M = l.M;
  p.N = l.N;
  p.K = l.K;
  p.NG = l.K / G;
  p.mtiles = s.mtiles;
  p.tile_units = s.units;
  p.per = s.per;
  p.splits = s.splits;
  p.grid = s.grid;
  p.xcd_remap = s.grid % 8 == 0 ? s.grid / 8 : 0;
  p.vector_out = reinterpret_cast<uintptr_t>(l.out) % 16 == 0;
  if (s.direct) {
    return s.bm == 32 ? launch_tile<Tile32<G>, A, F, false, true>(p, stream)
                      : hipErrorInvalidValue;
  }
  PrepareParams q;
  q.x = p.x;
  q.gamma = static_cast<const uint16_t*>(l.norm_weight);
  q.xs = reinterpret_cast<uint4*>(ws + s.xs);
  q.sums = reinterpret_cast<uint4*>(ws + s.sums);
  q.counters = p.counters;
  q.n_counters = s.splits > 1 ? s.mtiles * s.col_tiles : 0;
  q.M = l.M;
  q.K = l.K;
  q.NG = p.NG;
  q.eps = l.eps;
  q.quarters = is_native(F);
  const dim3 pgrid(static_cast<unsigned int>(s.mtiles * s.bm / kPrepRows),
                   static_cast<unsigned int>((l.K / 8 + kPrepUnits - 1) / kPrepUnits));
  if (l.norm_weight != nullptr) {
    hipLaunchKernelGGL((w4a16_gemm_tile_prepare_kernel<G, A, true>), pgrid, dim3(kPrepThreads), 0, stream, q);
  } else {
    hipLaunchKernelGGL((w4a16_gemm_tile_prepare_kernel<G, A, false>), pgrid, dim3(kPrepThreads), 0, stream, q);
  }
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) {
    return e;
  }
  constexpr bool kCanSilu = is_native(F);
  if (l.silu) {
    if constexpr (kCanSilu) {
      switch (s.bm) {
        case 32: return launch_tile<Tile32<G>, A, F, true>(p, stream);
        case 64: return launch_tile<Tile64<G>, A, F, true>(p, stream);
        case 128: return launch_tile<Tile128<G>, A, F, true>(p, stream);
        default: break;
      }
    }
    return hipErrorInvalidValue;
  }
  switch (s.bm) {
    case 32: return launch_tile<Tile32<G>, A, F, false>(p, stream);
    case 64: return launch_tile<Tile64<G>, A, F, false>(p, stream);
    case 128: return launch_tile<Tile128<G>, A, F, false>(p, stream);
    default: return hipErrorInvalidValue;
  }
}

template <PacketFormat F>
hipError_t launch_format(const TileLaunch& l, const TileShape& s, hipStream_t stream) {
  if (l.group_size == 64) {
    return l.act == Act::kF16 ? launch_typed<64, Act::kF16, F>(l, s, stream)
                              : launch_typed<64, Act::kBF16, F>(l, s, stream);
  }
  return l.act == Act::kF16 ? launch_typed<128, Act::kF16, F>(l, s, stream)
                            : launch_typed<128, Act::kBF16, F>(l, s, stream);
}

}  // namespace

// Tile choice and K splits by a cost model of the launch, in us, fitted to 560 measured launches (17
// to 512 rows, 512 to 16384 columns, K from 512 to 6144, bf16 native slabs, MI355X; the fit's
// standard deviation is 4-8 %). Over 645 drawn launches of both types and all formats, to 57344 columns
// and K of 28672, it is 5 %, 5 % and 0.5 % above the measured times of the 32-, 64- and 128-row tile (its
// costs are those of non-temporal weight loads, which the first two no longer use), with a standard
// deviation of 6-8 %, and beyond the fitted sizes within 2 %, 9 % and 2 %: workgroups run one per CU, in rounds of start-up and end (first
// loads; wave groups' sums, output), units and, with K split, the fix-up (partials out, counter,
// partials in); `prepare` is the launch before them.
struct TileCost {
  int bm, bn, phases;
  double unit, fixed, fix, fix_per_split, prepare;
};
constexpr TileCost kTileCosts64[] = {
    {32, 128, 4, 4.1, 4.5, 3.0, 0.1, 2.0},
    {64, 128, 4, 6.5, 6.4, 1.9, 0.8, 1.9},
    {128, 256, 1, 4.55, 6.1, 2.5, 2.8, 4.6},
};
constexpr TileCost kTileCosts128[] = {
    {32, 128, 4, 3.4, 4.1, 2.8, 0.1, 2.0},
    {64, 128, 4, 5.8, 6.0, 1.8, 0.85, 1.7},
    {128, 256, 1, 3.8, 7.25, 2.0, 3.1, 2.8},
};
constexpr int kMaxTileSplits = 16;

TileShape tile_shape(int rows, int n, int k, int group_size, bool direct, int cu_count,
                     size_t counter_bytes) {
  TileShape s;
  s.direct = direct;
  s.rows = rows;
  const int ng = k / group_size;
  for (const TileCost& c : group_size == 64 ? kTileCosts64 : kTileCosts128) {
    // the smallest tile serves rows that fit it, the largest more rows than the next one's
    if ((c.bm == 32 && rows > 32) || (c.bm == 64 && rows <= 32) || (c.bm == 128 && rows <= 64)) {
      continue;
    }
    const int mtiles = (rows + c.bm - 1) / c.bm;
    const int col_tiles = (n + c.bn - 1) / c.bn;
    const int unit_groups = c.phases * kTileWaveK / group_size;
    const int units = (ng + unit_groups - 1) / unit_groups;
    for (int splits = 1; splits <= std::min(units, kMaxTileSplits); ++splits) {
      const int per = (units + splits - 1) / splits;
      if ((units + per - 1) / per != splits) {
        continue;  // fewer splits give the same runs
      }
      const long long tiles = static_cast<long long>(mtiles) * col_tiles;
      const long long rounds = (tiles * splits + cu_count - 1) / cu_count;
      const double fix = splits > 1 ? c.fix + c.fix_per_split * splits : 0.0;
      const double cost = static_cast<double>(rounds) * (per * c.unit + c.fixed + fix) +
                          (direct ? 0.0 : c.prepare);
      if (s.bm == 0 || cost < s.us) {
        s.us = cost;
        s.bm = c.bm;
        s.bn = c.bn;
        s.mtiles = mtiles;
        s.col_tiles = col_tiles;
        s.unit_groups = unit_groups;
        s.units = units;
        s.per = per;
        s.splits = splits;
      }
    }
  }
  s.grid = s.mtiles * s.col_tiles * s.splits;
  auto align = [](size_t v) { return (v + 255) / 256 * 256; };
  const size_t padded = static_cast<size_t>(s.mtiles) * s.bm;
  s.partials = counter_bytes;
  const size_t partials_end = align(s.partials + (s.splits > 1 ? static_cast<size_t>(s.grid) * s.bm *
                                                             s.bn * sizeof(float)
                                                       : 0));
  s.sums = partials_end;
  s.xs = align(s.sums + padded * ng * 16);
  s.end = direct ? (s.splits > 1 ? partials_end : 0) : s.xs + padded * k * 2;
  return s;
}

hipError_t launch_w4a16_gemm_tile(const TileLaunch& l, const TileShape& s, hipStream_t stream) {
  if (l.M != s.rows || (l.silu && l.N % 256 != 0) ||
      (s.direct && (l.silu || l.norm_weight != nullptr || s.mtiles != 1))) {
    return hipErrorInvalidValue;
  }
  switch (l.format) {
    case PacketFormat::kArc: return launch_format<PacketFormat::kArc>(l, s, stream);
    case PacketFormat::kNativeSym: return launch_format<PacketFormat::kNativeSym>(l, s, stream);
    case PacketFormat::kNativeAsym: return launch_format<PacketFormat::kNativeAsym>(l, s, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fk
