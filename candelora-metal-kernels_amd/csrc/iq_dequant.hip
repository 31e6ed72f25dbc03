// iq_dequant.hip — any of the four formats -> dense [out_dim, in_dim] in f16 / bf16 / f32.
//
// Replaces the reference kernels iq2_xxs_dequantize_f16 / iq2_xs_dequantize_f16 /
// iq2_s_dequantize_f16 / iq3_s_dequantize_f16 (src/metal_src/iq2_matmul.metal:868-950,
// element decodes :701-866), which run one thread per output element and re-read the
// block's scale and codes for each.  Here one thread owns one group of 8 weights (one
// codebook entry and its sign byte; IQ3_S: two entries of 4).
//
// Every output is the single round-to-nearest-even of the exact fp32 product
// dl * g * sign (at most 22 significant bits), dl = d * (0.5 + s) * 0.25 for the IQ2
// formats and d * (1 + 2 s) for IQ3_S, so it is bit-identical to the reference's
// half(float) conversion.
//
// Bound: HBM, by the writes (2 or 4 bytes per weight against 0.26 to 0.43 read).
// Neighbouring threads own neighbouring groups, so a wave's loads fall into a few
// lines and each of its 16-byte stores covers 1 KB of one row; a thread per
// 32-weight sub-block, as before, stored 64 lanes x 16 bytes at 64-byte strides.
// 14336 x 4096 to f16: IQ2_S 259 -> 33 us, IQ2_XXS 41 -> 33 us (4.1 and 3.9 TB/s; a
// large copy reaches 5.2).  Rows whose outputs cannot take 16-byte
// stores (in_dim not a multiple of 8, or an unaligned out) go through LDS: a
// workgroup decodes 2048 columns of a row there and stores them in dwords at the
// output's own alignment (4001 x 4093 to f16: 80 -> 19 us; storing each element by
// itself took one 2-byte store per weight).
#include <type_traits>

#include "iq2xxs_device.h"
#include "iq2xxs_kernels.h"
#include "iq_variants_format.h"

namespace cmk {

static __constant__ uint16_t kDequantXsCodes[512] = {CMK_IQ2XS_GRID_CODES};
static __constant__ uint16_t kDequantSCodes[1024] = {CMK_IQ2S_GRID_CODES};
static __constant__ uint16_t kDequant3sCodes[512] = {CMK_IQ3S_GRID_CODES};

// V: 0 = IQ2_XXS, 1 = IQ2_XS, 2 = IQ2_S, 3 = IQ3_S.
template <int V>
struct DequantFmt {
  static constexpr uint32_t kBytes = V == 3 ? 104 : V == 2 ? 72 : 64;
  static constexpr uint32_t kScales = V == 3 ? 6 : V == 0 ? 2 : 10;
  static constexpr uint32_t kGrid = V == 0 ? 256 : V == 2 ? 1024 : 512;
};

// Codebook entries as magnitude bytes (IQ3_S: four, in the low half).
template <int V>
__device__ __forceinline__ void build_dequant_grid(uint64_t* grid) {
  for (uint32_t e = threadIdx.x; e < DequantFmt<V>::kGrid; e += blockDim.x) {
    if constexpr (V == 3) {
      const uint32_t c = kDequant3sCodes[e];
      uint32_t v = 0;
#pragma unroll
      for (int j = 0; j < 4; ++j) v |= (2u * ((c >> (3 * j)) & 7u) + 1u) << (8 * j);
      grid[e] = v;
    } else {
      grid[e] = grid_entry_from_code(V == 0 ? kGridCodesDev[e]
                                            : V == 1 ? kDequantXsCodes[e] : kDequantSCodes[e]);
    }
  }
}

template <bool kAligned>
__device__ __forceinline__ uint32_t dequant_u16(const uint8_t* p) {
  if constexpr (kAligned) return *reinterpret_cast<const uint16_t*>(p);
  return (uint32_t)p[0] | ((uint32_t)p[1] << 8);
}

// Signs of a ksigns index: the eighth makes their number even.
__device__ __forceinline__ uint32_t dequant_ksigns(uint32_t i) {
  return i | ((__popc(i) & 1u) << 7);
}

// The eight weights of group g (0..31) of block `block`.  kAligned: weight_bytes
// 8-byte and weight_scales 2-byte aligned (every block size is a multiple of 8 / 2).
template <int V, bool kAligned>
__device__ __forceinline__ void decode_group(const uint8_t* __restrict__ wb,
                                             const uint8_t* __restrict__ ws, uint64_t block,
                                             uint32_t g, const uint64_t* grid, float* v) {
  using F = DequantFmt<V>;
  const uint8_t* q = wb + block * F::kBytes;
  const uint8_t* sc = ws + block * F::kScales;
  const float d = half_bits_to_float((uint16_t)dequant_u16<kAligned>(sc));
  const uint32_t sb = g >> 2, w = g & 3;
  uint64_t mag;
  uint32_t sgn;
  float dl;
  if constexpr (V == 0) {
    static_assert(kAligned, "IQ2_XXS buffers are aligned");
    const uint32_t aux_s = *reinterpret_cast<const uint32_t*>(q + 8 * sb + 4);
    mag = grid[q[8 * sb + w]];
    sgn = dequant_ksigns((aux_s >> (7 * w)) & 0x7Fu);
    dl = (d * (0.5f + (float)(aux_s >> 28))) * 0.25f;
  } else if constexpr (V == 1) {
    const uint32_t code = dequant_u16<kAligned>(q + 2 * g);
    mag = grid[code & 0x1FFu];
    sgn = dequant_ksigns(code >> 9);
    dl = (d * (0.5f + (float)((sc[2 + sb] >> (4 * (w >> 1))) & 0x0Fu))) * 0.25f;
  } else if constexpr (V == 2) {
    mag = grid[q[g] | (((uint32_t)q[64 + sb] >> (2 * w)) & 3u) << 8];
    sgn = q[32 + g];
    dl = (d * (0.5f + (float)((sc[2 + sb] >> (4 * (w >> 1))) & 0x0Fu))) * 0.25f;
  } else {
    const uint32_t lo = dequant_u16<kAligned>(q + 2 * g);
    const uint32_t hi = (uint32_t)q[64 + sb] >> (2 * w);
    mag = grid[(lo & 0xFFu) | (hi & 1u) << 8] | grid[(lo >> 8) | (hi & 2u) << 7] << 32;
    sgn = q[72 + g];
    dl = d * (1.0f + 2.0f * (float)((sc[2 + (sb >> 1)] >> (4 * (sb & 1))) & 0x0Fu));
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const float m = dl * (float)((mag >> (8 * j)) & 0xFFu);
    v[j] = ((sgn >> j) & 1u) ? -m : m;
  }
}

__device__ __forceinline__ uint32_t dequant_bf16_rne(float v) {
  uint32_t b = __float_as_uint(v);
  if ((b & kAbsMask) > kInfBits) return ((b >> 16) & 0x8000u) | 0x7FC0u;
  b += 0x7FFFu + ((b >> 16) & 1u);
  return b >> 16;
}

// The eight weights as 16-bit patterns, two to a word: kind 1 = f16, 2 = bf16.  The
// hardware's conversion to bf16 rounds to nearest even and differs from the
// reference's rule for NaN only, which all eight weights of a group are or none is.
template <int kind>
__device__ __forceinline__ void dequant_pack(const float* v, uint32_t* p) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if constexpr (kind == 1) {
      p[k] = (uint32_t)__half_as_ushort(__float2half_rn(v[2 * k])) |
             (uint32_t)__half_as_ushort(__float2half_rn(v[2 * k + 1])) << 16;
    } else {
      typedef __bf16 bf2 __attribute__((ext_vector_type(2)));
      const bf2 b = {(__bf16)v[2 * k], (__bf16)v[2 * k + 1]};
      p[k] = __builtin_bit_cast(uint32_t, b);
    }
  }
  if constexpr (kind == 2) {
    if (v[0] != v[0]) {
#pragma unroll
      for (int k = 0; k < 4; ++k)
        p[k] = dequant_bf16_rne(v[2 * k]) | dequant_bf16_rne(v[2 * k + 1]) << 16;
    }
  }
}

constexpr uint32_t kDequantThreads = 256;

// kind: 0 = f32 out, 1 = f16 out, 2 = bf16 out.  in_dim % 8 == 0 and out 16-byte
// aligned: a group goes out as one 16-byte (f32: two) store.
template <int V, int kind, bool kAligned>
__global__ __launch_bounds__(kDequantThreads) void iq_dequant_kernel(
    const uint8_t* __restrict__ wb, const uint8_t* __restrict__ ws, void* __restrict__ out,
    uint64_t total, uint32_t groups_per_row, uint32_t bpr, uint32_t per_block) {
  __shared__ uint64_t grid[DequantFmt<V>::kGrid];
  build_dequant_grid<V>(grid);
  __syncthreads();
  // per_block consecutive groups: the row of the first one once per workgroup, the
  // others' from it in 32 bits
  const uint64_t g0 = (uint64_t)blockIdx.x * per_block;
  const uint64_t row0 = g0 / groups_per_row;
  const uint32_t rem0 = (uint32_t)(g0 - row0 * groups_per_row);
  const uint32_t count = (uint32_t)(total - g0 < per_block ? total - g0 : per_block);
#pragma unroll 2
  for (uint32_t i = threadIdx.x; i < count; i += kDequantThreads) {
    const uint32_t at = rem0 + i, r = at / groups_per_row, g = at - r * groups_per_row;
    float v[8];
    decode_group<V, kAligned>(wb, ws, (row0 + r) * bpr + (g >> 5), g & 31, grid, v);
    if constexpr (kind == 0) {
      float4* o = static_cast<float4*>(out) + 2 * (g0 + i);
      o[0] = make_float4(v[0], v[1], v[2], v[3]);
      o[1] = make_float4(v[4], v[5], v[6], v[7]);
    } else {
      uint32_t p[4];
      dequant_pack<kind>(v, p);
      static_cast<uint4*>(out)[g0 + i] = make_uint4(p[0], p[1], p[2], p[3]);
    }
  }
}

// Any in_dim and any out aligned to its element: a workgroup takes 2048 columns of a
// row at a time, a group per thread, through LDS.  16-bit outputs leave as dwords
// that are aligned in out; an odd first or last element as a 2-byte store.
constexpr uint32_t kDequantSegment = 8 * kDequantThreads;

template <int V, int kind, bool kAligned>
__global__ __launch_bounds__(kDequantThreads) void iq_dequant_ragged_kernel(
    const uint8_t* __restrict__ wb, const uint8_t* __restrict__ ws, void* __restrict__ out,
    uint32_t out_dim, uint32_t in_dim, uint32_t bpr) {
  using T = typename std::conditional<kind == 0, float, uint16_t>::type;
  __shared__ uint64_t grid[DequantFmt<V>::kGrid];
  __shared__ __align__(16) T seg[kDequantSegment];
  build_dequant_grid<V>(grid);
  const uint32_t segs = (in_dim - 1) / kDequantSegment + 1;
  const uint64_t total = (uint64_t)out_dim * segs;
  for (uint64_t s = blockIdx.x; s < total; s += gridDim.x) {
    const uint64_t row = s / segs;
    const uint32_t c0 = (uint32_t)(s - row * segs) * kDequantSegment;
    const uint32_t n = in_dim - c0 < kDequantSegment ? in_dim - c0 : kDequantSegment;
    __syncthreads();  // the codebook, or the previous segment's stores
    if (8 * threadIdx.x < n) {
      const uint32_t g = c0 / 8 + threadIdx.x;
      float v[8];
      decode_group<V, kAligned>(wb, ws, row * bpr + (g >> 5), g & 31, grid, v);
      if constexpr (kind == 0) {
#pragma unroll
        for (int j = 0; j < 8; ++j) seg[8 * threadIdx.x + j] = v[j];
      } else {
        uint32_t p[4];
        dequant_pack<kind>(v, p);
        reinterpret_cast<uint4*>(seg)[threadIdx.x] = make_uint4(p[0], p[1], p[2], p[3]);
      }
    }
    __syncthreads();
    T* const o = static_cast<T*>(out) + row * in_dim + c0;
    if constexpr (kind == 0) {
      for (uint32_t i = threadIdx.x; i < n; i += kDequantThreads) o[i] = seg[i];
    } else {
      const uint32_t odd = (reinterpret_cast<uintptr_t>(o) >> 1) & 1u;  // (n >= 1)
      const uint32_t pairs = (n - odd) / 2;
      for (uint32_t i = threadIdx.x; i < pairs; i += kDequantThreads)
        reinterpret_cast<uint32_t*>(o + odd)[i] =
            (uint32_t)seg[odd + 2 * i] | (uint32_t)seg[odd + 2 * i + 1] << 16;
      if (threadIdx.x == 0 && odd) o[0] = seg[0];
      if (threadIdx.x == 1 && odd + 2 * pairs < n) o[n - 1] = seg[n - 1];
    }
  }
}

template <int V, int kind, bool kAligned>
static hipError_t launch_dequant_t(const uint8_t* wb, const uint8_t* ws, void* out,
                                   uint32_t out_dim, uint32_t in_dim, int num_cus,
                                   hipStream_t stream) {
  const uint32_t bpr = (uint32_t)(((uint64_t)in_dim + kQK - 1) / kQK);
  if (in_dim % 8 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0) {
    // 8 to 64 groups a thread: enough to pay for the codebook, and at least eight
    // workgroups for every CU where the matrix has them
    const uint64_t total = (uint64_t)out_dim * (in_dim / 8);
    uint64_t per_thread = total / ((uint64_t)kDequantThreads * 8 * (uint64_t)num_cus);
    per_thread = per_thread < 8 ? 8 : per_thread > 64 ? 64 : per_thread;
    uint64_t per_block = per_thread * kDequantThreads;
    // (a grid holds 2^31 - 1 workgroups; total < 2^61 keeps this within 32 bits)
    while ((total + per_block - 1) / per_block > 0x40000000u) per_block *= 2;
    hipLaunchKernelGGL((iq_dequant_kernel<V, kind, kAligned>),
                       dim3((uint32_t)((total + per_block - 1) / per_block)),
                       dim3(kDequantThreads), 0, stream, wb, ws, out, total, in_dim / 8, bpr,
                       (uint32_t)per_block);
    return hipGetLastError();
  }
  const uint64_t segs = (uint64_t)out_dim * ((in_dim - 1) / kDequantSegment + 1);
  const uint64_t cap = (uint64_t)num_cus * 16;
  hipLaunchKernelGGL((iq_dequant_ragged_kernel<V, kind, kAligned>),
                     dim3((uint32_t)(segs < cap ? segs : cap)), dim3(kDequantThreads), 0, stream,
                     wb, ws, out, out_dim, in_dim, bpr);
  return hipGetLastError();
}

template <int V, bool kAligned>
static hipError_t launch_dequant_kind(const uint8_t* wb, const uint8_t* ws, void* out,
                                      int out_kind, uint32_t out_dim, uint32_t in_dim,
                                      int num_cus, hipStream_t stream) {
  switch (out_kind) {
    case 0:
      return launch_dequant_t<V, 0, kAligned>(wb, ws, out, out_dim, in_dim, num_cus, stream);
    case 1:
      return launch_dequant_t<V, 1, kAligned>(wb, ws, out, out_dim, in_dim, num_cus, stream);
    default:
      return launch_dequant_t<V, 2, kAligned>(wb, ws, out, out_dim, in_dim, num_cus, stream);
  }
}

template <int V>
static hipError_t launch_dequant_v(const uint8_t* wb, const uint8_t* ws, void* out, int out_kind,
                                   uint32_t out_dim, uint32_t in_dim, int num_cus,
                                   hipStream_t stream) {
  if (reinterpret_cast<uintptr_t>(wb) % 8 == 0 && reinterpret_cast<uintptr_t>(ws) % 2 == 0)
    return launch_dequant_kind<V, true>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
  if constexpr (V == 0)  // (cmk_iq2_dequantize refuses unaligned IQ2_XXS buffers)
    return hipErrorInvalidValue;
  else
    return launch_dequant_kind<V, false>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
}

hipError_t launch_iq_dequant(int variant, const uint8_t* wb, const uint8_t* ws, void* out,
                             int out_kind, uint32_t out_dim, uint32_t in_dim, int num_cus,
                             hipStream_t stream) {
  switch (variant) {
    case 0:
      return launch_dequant_v<0>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
    case 1:
      return launch_dequant_v<1>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
    case 2:
      return launch_dequant_v<2>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
    case 3:
      return launch_dequant_v<3>(wb, ws, out, out_kind, out_dim, in_dim, num_cus, stream);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace cmk
