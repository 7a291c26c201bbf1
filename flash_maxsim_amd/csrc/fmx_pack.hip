// Packing documents, and making operand rows ready. Packing: the token rows of padded docs [B, Ld, d], doc b's first
// lengths[b], back to back on groups of four rows. No counterpart in the
// reference, whose docs are always padded.
//
// layout_kernel turns lengths into where each doc starts, pack_kernel moves
// the rows. Each is one launch where tensor ops take a dozen over index
// tensors several times the size of the rows they move.
#include "fmx_device.h"
#include "fmx_kernels.h"

namespace fmx {
namespace {

constexpr int kLayoutThreads = 1024;
constexpr int kLayoutPer = 4;  // consecutive docs per thread and step

// Lengths clamped to [0, Ld], the exclusive prefix sum of their groups of four
// rows, and totals[0] = rows in all, totals[1] = the longest length. One
// workgroup walks the docs in order, kLayoutThreads * kLayoutPer a step, its
// sums meeting through LDS: a step is bound by its two barriers, and the whole
// by launch latency (5000 docs 7 us).
__global__ void __launch_bounds__(kLayoutThreads) layout_kernel(const int32_t* lengths, int64_t B, int32_t Ld,
                                                                int32_t* out, int64_t* tok_group, int64_t* totals) {
  __shared__ int64_t wsum[kLayoutThreads / 64];
  __shared__ int wmax[kLayoutThreads / 64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int64_t carry = 0;
  int longest = 0;
  for (int64_t b0 = 0; b0 < B; b0 += kLayoutThreads * kLayoutPer) {
    const int64_t b = b0 + (int64_t)threadIdx.x * kLayoutPer;
    int len[kLayoutPer];
    int64_t sum = 0;
#pragma unroll
    for (int i = 0; i < kLayoutPer; ++i) {
      const int l = b + i < B ? lengths[b + i] : 0;
      len[i] = l < 0 ? 0 : (l > Ld ? Ld : l);
    }
#pragma unroll
    for (int i = 0; i < kLayoutPer; ++i) {
      sum += ((int64_t)len[i] + 3) >> 2;
      longest = len[i] > longest ? len[i] : longest;
    }
    int64_t incl = sum;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int64_t v = __shfl_up(incl, o);
      if (lane >= o) incl += v;
    }
    if (lane == 63) wsum[wave] = incl;
    __syncthreads();
    int64_t at = carry + incl - sum;
    for (int w = 0; w < kLayoutThreads / 64; ++w) {
      if (w < wave) at += wsum[w];
      carry += wsum[w];
    }
    __syncthreads();  // wsum is rewritten by the next step
#pragma unroll
    for (int i = 0; i < kLayoutPer; ++i) {
      if (b + i < B) {
        out[b + i] = len[i];
        tok_group[b + i] = at;
      }
      at += ((int64_t)len[i] + 3) >> 2;
    }
  }
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int v = __shfl_xor(longest, o);
    longest = v > longest ? v : longest;
  }
  if (lane == 0) wmax[wave] = longest;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kLayoutThreads / 64; ++w) longest = wmax[w] > longest ? wmax[w] : longest;
    totals[0] = 4 * carry;
    totals[1] = longest;
  }
}

// Copies in units of U (the widest that rows, strides and addresses are
// multiples of). A workgroup takes kPackBlock consecutive units of one packed
// doc, whose rows are contiguous there; rows past the doc's length, up to its
// group's end, are zeros. Bound by memory: 10799 docs of 197 x 128 fp16 (545 MB
// read and as many written) 2012 -> 201 us, 5.4 TB/s.
// NT: both sides non-temporal, for docs the last-level cache would not hold.
constexpr int kPackIter = 4, kPackBlock = 256 * kPackIter;

template <typename U, bool NT>
__global__ void __launch_bounds__(256) pack_kernel(const U* src, int64_t sb, int64_t sl, int64_t B, int64_t Ld,
                                                   uint32_t upr, uint32_t magic, const int32_t* lengths,
                                                   const int64_t* tok_group, int64_t tok_rows, U* dst) {
  const int64_t base = (int64_t)blockIdx.x * kPackBlock;
  const int64_t row0 = base / upr;
  const uint32_t off0 = (uint32_t)(base - row0 * upr);
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    int64_t len = ld_uniform(lengths + b);
    len = len < 0 ? 0 : (len > Ld ? Ld : len);
    const int64_t end = ((len + 3) & ~(int64_t)3) * upr;  // units of the packed doc
    if (base >= end) continue;
    const int64_t out0 = 4 * ld_uniform(tok_group + b);
    const U* s = src + b * sb;
    U v[kPackIter];
#pragma unroll
    for (int k = 0; k < kPackIter; ++k) {
      const uint32_t o = off0 + k * 256 + threadIdx.x;
      const uint32_t r = magic ? __umulhi(o, magic) : o / upr;
      const int64_t j = row0 + r;
      v[k] = U{};
      if (j < len) {
        const U* p = s + j * sl + (o - r * upr);
        if constexpr (NT) {
          v[k] = __builtin_nontemporal_load(p);
        } else {
          v[k] = *p;
        }
      }
    }
#pragma unroll
    for (int k = 0; k < kPackIter; ++k) {
      const int64_t i = base + k * 256 + threadIdx.x;
      const uint32_t o = off0 + k * 256 + threadIdx.x;
      const int64_t row = out0 + row0 + (magic ? __umulhi(o, magic) : o / upr);
      if (i < end && row >= 0 && row < tok_rows) {
        U* p = dst + out0 * upr + i;
        if constexpr (NT) {
          __builtin_nontemporal_store(v[k], p);
        } else {
          *p = v[k];
        }
      }
    }
  }
}

template <typename U>
hipError_t launch_pack_units(const PackArgs& a, hipStream_t s) {
  const int64_t upr = a.row_bytes / (int64_t)sizeof(U);
  const int64_t gx = (((a.Ld + 3) & ~(int64_t)3) * upr + kPackBlock - 1) / kPackBlock;
  if (upr > INT32_MAX - 2 * kPackBlock || gx > 0x7fffff) return hipErrorInvalidValue;
  const int64_t gy = a.B < 65535 ? a.B : 65535;
  // o / upr by a multiplication while o * upr < 2^32 (o < upr + kPackBlock)
  const uint32_t magic = upr > 1 && upr <= 32768 ? (uint32_t)(((uint64_t)1 << 32) / (uint64_t)upr) + 1 : 0;
  const bool nt = a.tok_rows * a.row_bytes >= ((int64_t)1 << 28);
  auto kern = nt ? pack_kernel<U, true> : pack_kernel<U, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, static_cast<const U*>(a.src),
                     a.s_stride_b / (int64_t)sizeof(U), a.s_stride_l / (int64_t)sizeof(U), a.B, a.Ld, (uint32_t)upr,
                     magic, a.lengths, a.tok_group, a.tok_rows, static_cast<U*>(a.dst));
  return hipGetLastError();
}

// Operand rows cast to fp16 (round to nearest even, as torch's cast) or kept, and
// padded with zeros to a multiple of 8 elements, in one pass where torch casts,
// then pads (training step of 32 x 32 tokens over 256 fp32 docs of up to 180 x
// 128 105 -> 86 us with the gradients written in fp32); rows past a doc's length
// are left out, as nothing reads them. A thread takes kConvIter groups of four
// elements, each load and store of a wave contiguous (eight elements a thread
// left every fp32 load at a 32-byte stride: 8872 docs of 297 x 128 under 206
// tokens 515 -> 499 us). NT: non-temporal loads, for sources the last-level cache
// would not hold (there 507 -> 500; 500 docs of 100 x 128, 18.6 -> 21.9, keep the
// default). NTS: so the stores, for copies that it would not hold (502 -> 484;
// 2000 docs of 300 x 1024 849 -> 814, of 300 x 128, 154 MB, 101 -> 111).
// SRC: 0 fp16 or any 2-byte type kept, 1 bf16, 2 fp32. WIDE: groups are aligned
// and do not straddle d, one load each.
constexpr int kConvIter = 4;

template <int SRC, bool WIDE, bool NT, bool NTS>
__global__ void __launch_bounds__(256) convert_kernel(const void* src, int64_t sb, int64_t sl, int32_t Ld, uint32_t d,
                                                      uint32_t gpr, int64_t B, const int32_t* lengths, u32x2_t* dst) {
  const uint32_t x0 = blockIdx.x * (256 * kConvIter) + threadIdx.x;  // groups of a doc
  for (int64_t b = blockIdx.y; b < B; b += gridDim.y) {
    int32_t len = Ld;
    if (lengths) {
      len = ld_uniform(lengths + b);
      len = len < 0 ? 0 : (len > Ld ? Ld : len);
    }
    const uint32_t n = (uint32_t)len * gpr;
    if (x0 - threadIdx.x >= n) continue;  // uniform
    u32x4_t v[kConvIter];  // 2-byte sources: two words
#pragma unroll
    for (int k = 0; k < kConvIter; ++k) {
      // Groups past the doc repeat its last one and groups past d the row's: the
      // loads are unconditional, so all are in flight together.
      const uint32_t x = x0 + k * 256 < n ? x0 + k * 256 : n - 1, j = x / gpr, k0 = (x - j * gpr) * 4;
      const int64_t row = b * sb + (int64_t)j * sl;
      if constexpr (WIDE) {
        const bool pad = k0 >= d;
        const int64_t e0 = row + (pad ? d - 4 : k0);
        if constexpr (SRC == 2) {
          const u32x4_t* p = reinterpret_cast<const u32x4_t*>(static_cast<const uint32_t*>(src) + e0);
          v[k] = NT ? __builtin_nontemporal_load(p) : *p;
        } else {
          const u32x2_t* p = reinterpret_cast<const u32x2_t*>(static_cast<const uint16_t*>(src) + e0);
          const u32x2_t w = NT ? __builtin_nontemporal_load(p) : *p;
          v[k] = u32x4_t{w[0], w[1], 0u, 0u};
        }
        if (pad) v[k] = u32x4_t{0u, 0u, 0u, 0u};
      } else {
        v[k] = u32x4_t{0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if constexpr (SRC == 2) {
            v[k][e] = k0 + e < d ? static_cast<const uint32_t*>(src)[row + k0 + e] : 0u;
          } else {
            const uint32_t h = k0 + e < d ? static_cast<const uint16_t*>(src)[row + k0 + e] : 0u;
            v[k][e >> 1] |= h << (16 * (e & 1));
          }
        }
      }
    }
    auto half = [](float f) { return (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)f); };
#pragma unroll
    for (int k = 0; k < kConvIter; ++k) {
      const uint32_t x = x0 + k * 256;
      if (x >= n) continue;
      u32x2_t o;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (SRC == 2) {
          // (copies: a vector subscript inside a bit cast takes the first element)
          const uint32_t lo = v[k][2 * i], hi = v[k][2 * i + 1];
          o[i] = half(__builtin_bit_cast(float, lo)) | (half(__builtin_bit_cast(float, hi)) << 16);
        } else if constexpr (SRC == 1) {
          o[i] = half(bf16_bits_to_float(v[k][i] & 0xffffu)) | (half(bf16_bits_to_float(v[k][i] >> 16)) << 16);
        } else {
          o[i] = v[k][i];
        }
      }
      u32x2_t* p = dst + b * ((int64_t)Ld * gpr) + x;
      if constexpr (NTS) {
        __builtin_nontemporal_store(o, p);
      } else {
        *p = o;
      }
    }
  }
}

template <int SRC>
hipError_t launch_convert_src(ConvertArgs a, hipStream_t s) {
  constexpr int esz = SRC == 2 ? 4 : 2;
  const int64_t gpr = a.dp / 4;
  if (a.Ld * gpr > INT32_MAX - 4096) return hipErrorInvalidValue;
  const bool nt = a.B * a.Ld * a.d * esz >= ((int64_t)1 << 28);
  const bool nts = nt && a.B * a.Ld * a.dp * 2 >= ((int64_t)1 << 28);
  // docs back to back, all rows of them: one doc, without a part-filled workgroup each
  if (!a.lengths && a.s_stride_b == a.Ld * a.s_stride_l && a.B * a.Ld <= (INT32_MAX - 4096) / gpr) {
    a.Ld *= a.B;
    a.B = 1;
  }
  const uint64_t bits = reinterpret_cast<uintptr_t>(a.src) / esz | (uint64_t)a.s_stride_b | (uint64_t)a.s_stride_l |
                        (uint64_t)a.d;
  const int64_t gy = a.B < 65535 ? a.B : 65535, gx = (a.Ld * gpr + 256 * kConvIter - 1) / (256 * kConvIter);
  auto kern = convert_kernel<SRC, false, false, false>;
  if ((bits & 3) == 0)
    kern = nts  ? convert_kernel<SRC, true, true, true>
           : nt ? convert_kernel<SRC, true, true, false>
                : convert_kernel<SRC, true, false, false>;
  hipLaunchKernelGGL(kern, dim3((unsigned)gx, (unsigned)gy), dim3(256), 0, s, a.src, a.s_stride_b, a.s_stride_l,
                     (int32_t)a.Ld, (uint32_t)a.d, (uint32_t)gpr, a.B, a.lengths, static_cast<u32x2_t*>(a.dst));
  return hipGetLastError();
}

}  // namespace

hipError_t launch_convert(const ConvertArgs& a, hipStream_t s) {
  return a.f32 ? launch_convert_src<2>(a, s) : a.bf16 ? launch_convert_src<1>(a, s) : launch_convert_src<0>(a, s);
}

hipError_t launch_layout(const int32_t* lengths, int64_t B, int32_t Ld, int32_t* out, int64_t* tok_group,
                         int64_t* totals, hipStream_t s) {
  hipLaunchKernelGGL(layout_kernel, dim3(1), dim3(kLayoutThreads), 0, s, lengths, B, Ld, out, tok_group, totals);
  return hipGetLastError();
}

hipError_t launch_pack(const PackArgs& a, hipStream_t s) {
  const uint64_t bits = (uint64_t)a.row_bytes | (uint64_t)a.s_stride_b | (uint64_t)a.s_stride_l |
                        reinterpret_cast<uintptr_t>(a.src) | reinterpret_cast<uintptr_t>(a.dst);
  if ((bits & 15) == 0) return launch_pack_units<u32x4_t>(a, s);
  if ((bits & 3) == 0) return launch_pack_units<uint32_t>(a, s);
  if ((bits & 1) == 0) return launch_pack_units<uint16_t>(a, s);
  return launch_pack_units<uint8_t>(a, s);
}

}  // namespace fmx
