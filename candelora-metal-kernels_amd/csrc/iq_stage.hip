// iq_stage.hip — activation rows as the f16 rows that the MFMA matmuls multiply.
//
// One workgroup per row, one pass over it: the row is held in registers between its
// maximum and its conversion.  Rows leave `pitch` (a multiple of 8) halves apart, zeros
// past in_dim, so rows of any length and any element alignment can be copied by the
// matmuls in 16-byte pieces.
//  * f16: a copy (for rows that are not laid out so already).
//  * bf16: x * 2^e, the power of two that brings the row's largest finite magnitude into
//    [2^14, 2^15); exact for every value at or above 2^-31 of it.  row_inv = 2^e.
//  * f32: the same scaling, as two rows: the head h = rne(v) and the tail rne(v - h)
//    (v - h is exact in fp32), about 22 bits of v.  NaN and infinities stay in the head,
//    with a zero tail.
//    Of bf16 and f32 rows, with block_inv: super-blocks of 256 columns whose largest finite
//    magnitude is more than 2^18 below the row's (they would keep fewer than 22 bits of it)
//    get a power of two of their own, 2^e * 2^f.  A row that may have one (eight neighbours
//    so far below) has its row_inv negated, and block_inv[row * ceil(in_dim / 256) + b] = 2^-f
//    for its blocks (1 for most); for other rows block_inv is not written.
//  * W8A8 (any dtype): q = clamp(round_half_away(x * inv), +-127), inv = 127 / max|x| (1
//    below 1e-8), as the reference quantises (src/iq2_matmul.rs:1025-1048).  row_inv = inv.
//
// Bound: HBM for many rows (each element read once and written once), the round trip of
// one load for few.  W8A8 rows took a pass for the scales and one for q: 256 x 14336 x 4096
// (IQ2_XXS, f16) 69.2 -> 62.3 us with one.
#include <algorithm>

#include "iq2xxs_device.h"
#include "iq2xxs_kernels.h"

namespace cmk {

// Under-aligned 16-byte loads (the hardware takes them in one instruction).
struct __attribute__((packed, aligned(2))) StageU4 {
  uint32_t v[4];
};

enum StageMode { kStageCopy = 0, kStageScaled = 1, kStagePair = 2, kStageW8A8 = 3 };

// Eight elements of a row from column 8 c, zeros past in_dim.
template <int XD>
struct StageOctet {
  uint32_t raw[XD == 0 ? 8 : 4];
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int k = 0; k < (XD == 0 ? 8 : 4); ++k) raw[k] = 0;
  }
  __device__ __forceinline__ void load(const void* row, uint32_t c, uint32_t in_dim) {
    if (8 * c + 8 <= in_dim) {
      const StageU4* p = reinterpret_cast<const StageU4*>(static_cast<const uint8_t*>(row) +
                                                          (size_t)c * (XD == 0 ? 32 : 16));
#pragma unroll
      for (int i = 0; i < (XD == 0 ? 2 : 1); ++i) {
        const StageU4 u = p[i];
#pragma unroll
        for (int k = 0; k < 4; ++k) raw[4 * i + k] = u.v[k];
      }
    } else {
      clear();
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (8 * c + k < in_dim) {
          if constexpr (XD == 0)
            raw[k] = load_x_bits<0>(row, (size_t)8 * c + k);
          else
            raw[k >> 1] |= load_x_bits<XD>(row, (size_t)8 * c + k) << (16 * (k & 1));
        }
    }
  }
  __device__ __forceinline__ float get(int k) const {
    if constexpr (XD == 0) return __uint_as_float(raw[k]);
    return x_bits_to_float<XD>((k & 1) ? raw[k >> 1] >> 16 : raw[k >> 1] & 0xFFFFu);
  }
};

__device__ __forceinline__ uint32_t stage_pack(float lo, float hi) {
  return (uint32_t)__half_as_ushort(__float2half_rn(lo)) |
         (uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16;
}

constexpr uint32_t kStageThreads = 1024;  // at most
constexpr uint32_t kStageLaunchRows = 1u << 23;

// Blocks this far below the row's largest magnitude are scaled by themselves.
constexpr int kStageSpread = 18;

// kV: octets a thread holds (rows of up to 8 kV columns a thread); 0: rows of any length,
// read twice.
// (Registers for 8 waves a SIMD, two workgroups of 1024: with one, 512 f32 rows of 28672
// columns took 5 us longer.)
template <int XD, int kMode, int kV>
__global__ __launch_bounds__(kV == 8 ? 256 : kStageThreads, kV == 8 ? 4 : 8) void iq_stage_rows_kernel(
    const void* __restrict__ x, uint32_t in_dim, uint32_t pitch, float* __restrict__ row_inv,
    float* __restrict__ block_inv, uint16_t* __restrict__ q) {
  __shared__ uint32_t s_red[kStageThreads / 64], s_low[kStageThreads / 64];
  const uint32_t row = blockIdx.x, tid = threadIdx.x, threads = blockDim.x;
  const uint8_t* r = static_cast<const uint8_t*>(x) + (size_t)row * in_dim * (XD == 0 ? 4 : 2);
  const uint32_t octets = pitch / 8;
  StageOctet<XD> v[kV ? kV : 1];
  float inv = 1.0f;
  int exponent = 0;  // (inv = 2^exponent where rows are scaled)
  // the largest magnitude, as integer bits: of the finite values where rows are scaled; of
  // all but NaN (which fmaxf ignores) where they are quantised
  constexpr bool kScaled = kMode == kStageScaled || kMode == kStagePair;
  auto largest = [&](const StageOctet<XD>& o) {
    uint32_t m = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const uint32_t b = __float_as_uint(o.get(k)) & kAbsMask;
      if (kMode == kStageW8A8 ? b <= kInfBits : b < kInfBits) m = max(m, b);
    }
    return m;
  };
  // and the least of the octets' largest magnitudes that are not 0, less 1
  uint32_t mb = 0, low = ~0u;
  auto fold = [&](const StageOctet<XD>& o) {
    const uint32_t m = largest(o);
    mb = max(mb, m);
    if (kScaled) low = min(low, m - 1);
  };
  if constexpr (kV > 0) {
#pragma unroll
    for (int j = 0; j < kV; ++j) {
      if (tid + threads * j < octets)
        v[j].load(r, tid + threads * j, in_dim);
      else
        v[j].clear();
    }
  }
  if constexpr (kMode != kStageCopy) {
    if constexpr (kV > 0) {
#pragma unroll
      for (int j = 0; j < kV; ++j) fold(v[j]);
    } else {
      for (uint32_t c = tid; c < octets; c += threads) {
        v[0].load(r, c, in_dim);
        fold(v[0]);
      }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      mb = max(mb, (uint32_t)__shfl_xor((int)mb, off));
      if (kScaled) low = min(low, (uint32_t)__shfl_xor((int)low, off));
    }
    if ((tid & 63) == 0) {
      s_red[tid >> 6] = mb;
      s_low[tid >> 6] = low;
    }
    __syncthreads();
    mb = s_red[0];
    low = s_low[0];
    for (uint32_t w = 1; w < threads / 64; ++w) {
      mb = max(mb, s_red[w]);
      low = min(low, s_low[w]);
    }
    const float mx = __uint_as_float(mb);
    if constexpr (kMode == kStageW8A8) {
      inv = mx < 1e-8f ? 1.0f : 127.0f / mx;
    } else {
      exponent = mx > 0.0f ? min(14 - ilogbf(mx), 126) : 0;
      inv = ldexpf(1.0f, exponent);
    }
  }
  // What an octet's super-block has beyond the row's exponent.  Called by whole waves: 32
  // lanes hold a block, zeros past the row.
  const uint32_t far = mb >= (kStageSpread << 23) ? mb - (kStageSpread << 23) : 0;  // mx * 2^-18
  auto block_extra = [&](const StageOctet<XD>& o) {
    uint32_t bm = largest(o);
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) bm = max(bm, (uint32_t)__shfl_xor((int)bm, off));
    if (bm == 0 || bm >= far) return 0;
    return min(min(14 - ilogbf(__uint_as_float(bm)), 126) - exponent, 126);
  };
  uint16_t* const dst = q + (size_t)row * pitch * (kMode == kStagePair ? 2 : 1);
  auto put = [&](const StageOctet<XD>& o, uint32_t c, float inv) {
    uint32_t w[4], t[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float lo = o.get(2 * k), hi = o.get(2 * k + 1);
      if constexpr (kMode == kStageCopy) {
        w[k] = o.raw[k];
      } else if constexpr (kMode == kStageW8A8) {
        w[k] = stage_pack(quant_w8a8(lo, inv), quant_w8a8(hi, inv));
      } else {
        const float a = lo * inv, b = hi * inv;
        w[k] = stage_pack(a, b);
        if constexpr (kMode == kStagePair) {
          const bool fa = (__float_as_uint(a) & kAbsMask) < kInfBits;
          const bool fb = (__float_as_uint(b) & kAbsMask) < kInfBits;
          t[k] = stage_pack(fa ? a - half_bits_to_float((uint16_t)w[k]) : 0.0f,
                            fb ? b - half_bits_to_float((uint16_t)(w[k] >> 16)) : 0.0f);
        }
      }
    }
    *reinterpret_cast<uint4*>(dst + 8 * (size_t)c) = make_uint4(w[0], w[1], w[2], w[3]);
    if constexpr (kMode == kStagePair)
      *reinterpret_cast<uint4*>(dst + pitch + 8 * (size_t)c) = make_uint4(t[0], t[1], t[2], t[3]);
  };
  // Nearly every row: no octet, so no block, is far below the row.
  if (!kScaled || block_inv == nullptr || far == 0 || low >= far - 1) {
    if (kMode != kStageCopy && tid == 0) row_inv[row] = inv;
    if constexpr (kV > 0) {
#pragma unroll
      for (int j = 0; j < kV; ++j)
        if (tid + threads * j < octets) put(v[j], tid + threads * j, inv);
    } else {
      for (uint32_t c = tid; c < octets; c += threads) {
        v[0].load(r, c, in_dim);
        put(v[0], c, inv);
      }
    }
    return;
  }
  if constexpr (kScaled) {
    float* const bi = block_inv + (size_t)row * ((in_dim + kQK - 1) / kQK);
    if (tid == 0) row_inv[row] = -inv;
    auto put_block = [&](const StageOctet<XD>& o, uint32_t c) {
      const int extra = block_extra(o);
      if (c >= octets) return;
      put(o, c, ldexpf(1.0f, exponent + extra));
      if (c % 32 == 0) bi[c / 32] = ldexpf(1.0f, -extra);
    };
    if constexpr (kV > 0) {
#pragma unroll
      for (int j = 0; j < kV; ++j) put_block(v[j], tid + threads * j);
    } else {
      for (uint32_t c = tid; c - tid < octets; c += threads) {
        if (c < octets)
          v[0].load(r, c, in_dim);
        else
          v[0].clear();
        put_block(v[0], c);
      }
    }
  }
}

template <int XD, int kMode>
static hipError_t launch_stage(const void* x, uint32_t m, uint32_t in_dim, uint32_t pitch,
                               float* row_inv, uint16_t* q, float* block_inv,
                               hipStream_t stream) {
  // An octet a thread for few rows (the round trip counts); for many, workgroups of 256,
  // several to a CU (2048 rows of 4096, bf16: 10.3 us), where they hold the row: past 16384
  // columns they would read it twice (IQ2_XXS matmuls of 2048 x 512 x 28672, staging
  // included, rows read twice / held: f32 289 / 250 us, bf16 139 / 124, f32 W8A8 192 / 147).
  const uint32_t octets = pitch / 8;
  const uint32_t threads = m > 512 && octets <= 256 * 8
                               ? 256
                               : std::min(kStageThreads, std::max(256u, (octets + 63) / 64 * 64));
  const uint32_t per = (octets + threads - 1) / threads;
  auto kern = per <= 1   ? &iq_stage_rows_kernel<XD, kMode, 1>
              : per <= 2 ? &iq_stage_rows_kernel<XD, kMode, 2>
              : per <= 4 ? &iq_stage_rows_kernel<XD, kMode, 4>
              : per <= 8 && threads == 256
                  ? &iq_stage_rows_kernel<XD, kMode, 8>
                  : &iq_stage_rows_kernel<XD, kMode, 0>;
  // (a launch holds fewer than 2^32 threads)
  for (uint32_t r0 = 0; r0 < m;) {
    const uint32_t rows = std::min(m - r0, kStageLaunchRows);
    hipLaunchKernelGGL(kern, dim3(rows), dim3(threads), 0, stream,
                       static_cast<const uint8_t*>(x) + (size_t)r0 * in_dim * (XD == 0 ? 4 : 2),
                       in_dim, pitch, row_inv + (kMode == kStageCopy ? 0 : r0),
                       block_inv ? block_inv + (size_t)r0 * ((in_dim + kQK - 1) / kQK) : nullptr,
                       q + (size_t)r0 * pitch * (kMode == kStagePair ? 2 : 1));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    r0 += rows;
  }
  return hipSuccess;
}

hipError_t launch_iq_stage_rows(const void* x, int x_dtype, bool w8a8, uint32_t m,
                                uint32_t in_dim, uint32_t pitch, float* row_inv, void* rows,
                                hipStream_t stream, float* block_inv) {
  uint16_t* const q = static_cast<uint16_t*>(rows);
  if (w8a8) {
    auto launch = x_dtype == 0   ? &launch_stage<0, kStageW8A8>
                  : x_dtype == 1 ? &launch_stage<1, kStageW8A8>
                                 : &launch_stage<2, kStageW8A8>;
    return launch(x, m, in_dim, pitch, row_inv, q, nullptr, stream);
  }
  auto launch = x_dtype == 0   ? &launch_stage<0, kStagePair>
                : x_dtype == 1 ? &launch_stage<1, kStageCopy>
                               : &launch_stage<2, kStageScaled>;
  return launch(x, m, in_dim, pitch, row_inv, q, block_inv, stream);
}

}  // namespace cmk
