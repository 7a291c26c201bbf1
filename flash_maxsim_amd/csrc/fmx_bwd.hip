// Argmax backward of MaxSim (single or batched queries over shared docs).
//
// Replaces _maxsim_bwd_dQ_kernel and _maxsim_bwd_dD_kernel (reference
// flash_maxsim/flash_maxsim.py:153-188) with the same mathematics, extended to
// Nq queries and doc lengths (a = argmax, g = upstream gradient of scores):
//   dQ[qi, q, :] = sum_b g[qi, b] * D[b, a[qi*B + b, q], :]
//   dD[b, j, :]  = sum_{(qi, q) : a[qi*B + b, q] = j} g[qi, b] * Q[qi, q, :]
// Docs of length 0 (every similarity masked, score -inf) take no part, as in
// autograd through the masked naive MaxSim.
// Differences by design:
//  * dQ is a two-stage gather-reduce: doc chunks accumulate fp32 partials in a
//    caller workspace, then a second kernel adds the chunks in order. The
//    reference runs one program per query token looping over every doc.
//  * dD is written exactly once per element by the doc's workgroup (zeros for
//    rows no query token picked, the fp32 sum for picked rows, in (query,
//    token) order), so there is no torch.zeros_like memset and no fp16
//    atomics; results are bitwise deterministic.
#include <type_traits>

#include "fmx_device.h"
#include "fmx_kernels.h"

namespace fmx {
namespace {

template <bool BF>
struct Elem;
template <>
struct Elem<false> {
  static __device__ __forceinline__ float to_f(uint16_t v) { return (float)__builtin_bit_cast(_Float16, v); }
  static __device__ __forceinline__ uint16_t from_f(float x) {
    return __builtin_bit_cast(uint16_t, (_Float16)x);
  }
};
template <>
struct Elem<true> {
  static __device__ __forceinline__ float to_f(uint16_t v) {
    return __builtin_bit_cast(float, (uint32_t)v << 16);
  }
  static __device__ __forceinline__ uint16_t from_f(float x) {
    return __builtin_bit_cast(uint16_t, (__bf16)x);
  }
};

// Gradient rows as they are stored: 2-byte elements with d % 8 == 0 (OUT_H8),
// 2-byte elements of any d, or fp32. A lane has eight elements of a row: eight
// in a row, or for fp32 two quads L quads apart, so that each store
// instruction covers whole lines.
enum Out : int { OUT_H8, OUT_H, OUT_F32 };

// Loads elements p0 .. p0+3 and p1 .. p1+3 of a 2-byte row as fp32, p0 < d: one
// 16-byte load where they are adjacent (rows start 16-byte aligned, a multiple
// of 8 elements apart). Elements at or past d may be anything; they reach only
// sums that are not stored.
template <bool BF, int OUT>
__device__ __forceinline__ void load8(const uint16_t* row, int p0, int p1, float (&x)[8]) {
  u32x4_t v;
  if constexpr (OUT == OUT_F32) {
    const u32x2_t a = *reinterpret_cast<const u32x2_t*>(row + p0), b = *reinterpret_cast<const u32x2_t*>(row + p1);
    v = u32x4_t{a[0], a[1], b[0], b[1]};
  } else {
    v = *reinterpret_cast<const u32x4_t*>(row + p0);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    x[2 * e] = Elem<BF>::to_f(v[e] & 0xffffu);
    x[2 * e + 1] = Elem<BF>::to_f(v[e] >> 16);
  }
}

// Stores those elements (the ones below d) of a gradient row; 16-byte stores of
// 2-byte elements need d % 8 == 0 so that every row of the contiguous output
// starts 16-byte aligned, 8-byte ones (and 16-byte ones of fp32) d % 4 == 0
// (backward of 18 queries of 32 tokens over 2000 docs of 1048 x 100: 512 -> 165
// us with whole-row loads and these). dD is written once and read only by the
// optimiser later: non-temporal stores stream it out instead of leaving it
// dirty in the caches, where its write-back would compete with the next
// forward's reads.
template <bool BF, int OUT>
__device__ __forceinline__ void store8(void* out_row, int p0, int p1, int d, const float (&x)[8]) {
  if constexpr (OUT == OUT_F32) {
    float* row = static_cast<float*>(out_row);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int p = h ? p1 : p0;
      if ((d & 3) == 0) {
        if (p < d)
          __builtin_nontemporal_store(f32x4_t{x[4 * h], x[4 * h + 1], x[4 * h + 2], x[4 * h + 3]},
                                      reinterpret_cast<f32x4_t*>(row + p));
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (p + e < d) row[p + e] = x[4 * h + e];
      }
    }
    return;
  }
  uint16_t* row = static_cast<uint16_t*>(out_row);
  u32x4_t v;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    v[i] = (uint32_t)Elem<BF>::from_f(x[2 * i]) | ((uint32_t)Elem<BF>::from_f(x[2 * i + 1]) << 16);
  if constexpr (OUT == OUT_H8) {
    __builtin_nontemporal_store(v, reinterpret_cast<u32x4_t*>(row + p0));
  } else if ((d & 3) == 0) {
    __builtin_nontemporal_store(u32x2_t{v[0], v[1]}, reinterpret_cast<u32x2_t*>(row + p0));
    if (p1 < d) __builtin_nontemporal_store(u32x2_t{v[2], v[3]}, reinterpret_cast<u32x2_t*>(row + p1));
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if (p0 + e < d) row[p0 + e] = Elem<BF>::from_f(x[e]);
  }
}

__device__ __forceinline__ int clamp_index(int j, int Ld) { return j < 0 ? 0 : (j >= Ld ? Ld - 1 : j); }

__device__ __forceinline__ int doc_len(const BwdArgs& a, int b) {
  if (!a.lengths) return a.Ld;
  const int l = a.lengths[b];
  return l < 0 ? 0 : (l > a.Ld ? a.Ld : l);
}

// Stage 1 of dQ: one thread per (query token row r = qi*Lq + q, 8-wide k
// chunk), one grid row per chunk of docs; ws[chunk][r][k] = sum over the
// chunk's docs, in order. Docs go in batches of DB: the batch's argmax, upstream
// gradients and lengths are loaded together, then its DB row chunks of D, so a
// thread has DB gathers in flight instead of one (a doc at a time costs two
// dependent memory round trips, and config 5's threads walk 32 docs each).
// Positions past the chunk read its last doc again and, like empty docs, are
// skipped (not multiplied by zero: a row may hold NaN padding); whether a doc
// counts depends on the doc alone, so the skip is uniform over the wave.
template <bool BF>
__device__ __forceinline__ void dq_partial_block(const BwdArgs& a, int64_t bx, int by) {
  constexpr int DB = 8;
  const int nkc = (a.d + 7) >> 3;
  const int64_t rows = (int64_t)a.Nq * a.Lq;
  const int64_t tid = bx * 256 + threadIdx.x;
  if (tid >= rows * nkc) return;
  const int64_t r = tid / nkc;
  const int k0 = (int)(tid - r * nkc) * 8;
  const int qi = (int)(r / a.Lq), q = (int)(r - (int64_t)qi * a.Lq);
  const int per = (a.B + a.nchunk - 1) / a.nchunk;
  const int b0 = by * per;
  const int b1 = min(a.B, b0 + per);
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  const uint16_t* D = static_cast<const uint16_t*>(a.D);
  const int32_t* am = a.argmax + (int64_t)qi * a.B * a.Lq + q;
  const float* g = a.grad + (int64_t)qi * a.g_n;
  for (int bb = b0; bb < b1; bb += DB) {
    int j[DB];
    float gb[DB];
    int bi[DB];
#pragma unroll
    for (int u = 0; u < DB; ++u) {
      bi[u] = bb + u < b1 ? bb + u : b1 - 1;
      j[u] = am[(int64_t)bi[u] * a.Lq];
      gb[u] = g[(int64_t)bi[u] * a.g_b];
    }
    bool live[DB];
#pragma unroll
    for (int u = 0; u < DB; ++u) {
      live[u] = bb + u < b1;
      if (a.lengths) live[u] = live[u] && ld_uniform(a.lengths + bi[u]) > 0;
      j[u] = clamp_index(j[u], a.Ld);
    }
    float x[DB][8];
#pragma unroll
    for (int u = 0; u < DB; ++u) {
      const uint16_t* row = D + (int64_t)bi[u] * a.sd_b + (int64_t)j[u] * a.sd_l;
      load8<BF, OUT_H8>(row, k0, k0 + 4, x[u]);
    }
#pragma unroll
    for (int u = 0; u < DB; ++u)
      if (live[u])
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] = fmaf(gb[u], x[u][e], acc[e]);
  }
  float* out = a.ws + ((int64_t)by * rows + r) * a.d + k0;
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (k0 + e < a.d) out[e] = acc[e];
}

// Stage 2 of dQ: dQ[r][k] = sum over chunks (in order) of ws[chunk][r][k].
template <bool BF, int OUT>
__device__ __forceinline__ void dq_sum_block(const BwdArgs& a, int64_t block) {
  const int64_t n = (int64_t)a.Nq * a.Lq * a.d;
  const int64_t i = block * 256 + threadIdx.x;
  if (i >= n) return;
  float s = 0.f;
#pragma unroll 8
  for (int c = 0; c < a.nchunk; ++c) s += a.ws[(int64_t)c * n + i];  // chunk order: deterministic
  if constexpr (OUT == OUT_F32) {
    static_cast<float*>(a.dQ)[i] = s;
  } else {
    static_cast<uint16_t*>(a.dQ)[i] = Elem<BF>::from_f(s);
  }
}

constexpr int kEntryBits = 13;  // entries of one chunk < 2^13 (kDdChunk)
constexpr uint32_t kNoRow = 0xffffffffu;
constexpr int kDdMaxPasses = 4;  // workgroup row passes per dD writer slab, at most
// LDS of an index workgroup: its keys, and with the counting sort four
// counters per doc row, which fit beside 8192 keys up to Ld = 2044.
constexpr size_t kDdIndexLds = 65536 - 64;
constexpr size_t dd_count_bytes(int64_t Ld) { return (size_t)Ld * 4 * sizeof(uint32_t); }

// dD index, one workgroup per (doc, chunk of kDdChunk consecutive (query,
// token) entries): the chunk's entries sorted by the doc row they picked, in
// entry order within a row. Written to the workspace:
//   ent[b][e0 + p]     chunk-local entry of sorted position p (uint16)
//   rows[c][b][j]      first sorted position | count << 16 of row j within
//                      chunk c, or kNoRow.
// Chunks hold consecutive entries, so a row's entries taken chunk by chunk
// are in entry order. Docs of length 0 pick no rows.
//
// A stable counting sort: wave w takes the w-th quarter of the entries and
// counts its rows in its own LDS counters; a scan over (row, wave) turns the
// counts into positions; then each wave places its entries 64 at a time, a
// lane's place among the lanes of its row found by ballots over the bits of
// the row number. What bounds it is the number of barriers and dependent LDS
// round trips per workgroup, as one doc's entries rarely fill more than one
// workgroup per CU: four barriers here, where a bitonic sort of the keys takes
// one per step, 55 for 1024 entries (32 queries of 32 tokens over 256 docs of
// up to 180 tokens: 44.0 -> 6.7 us).
__device__ __forceinline__ void dd_index_count(const BwdArgs& a, int b, int chunk, uint32_t* smem) {
  const int NL = a.Nq * a.Lq;
  const int e0 = chunk * kDdChunk;
  const int n = NL - e0 < kDdChunk ? NL - e0 : kDdChunk;  // entries of this chunk
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool empty = a.lengths && doc_len(a, b) == 0;
  uint32_t* keys = smem;                // [sort_n] the row each entry picked
  uint32_t* pos = smem + a.sort_n;      // [4][Ld] counts, then next positions
  __shared__ uint32_t wtot[4];
  for (int i = threadIdx.x; i < 4 * a.Ld; i += 256) pos[i] = 0u;
  __syncthreads();
  const int seg = (n + 255) / 256 * 64;  // entries per wave
  const int p0 = wave * seg, p1 = empty ? p0 : (p0 + seg < n ? p0 + seg : n);
  uint32_t* mypos = pos + wave * a.Ld;
  for (int p = p0 + lane; p < p1; p += 64) {
    const int e = e0 + p;
    const int qi = e / a.Lq, q = e - qi * a.Lq;
    const int j = clamp_index(a.argmax[((int64_t)qi * a.B + b) * a.Lq + q], a.Ld);
    keys[p] = (uint32_t)j;
    atomicAdd(&mypos[j], 1u);
  }
  __syncthreads();
  // each thread scans `per` consecutive rows
  const int per = (a.Ld + 255) / 256;
  const int j0 = threadIdx.x * per, j1 = j0 + per < a.Ld ? j0 + per : a.Ld;
  uint32_t sum = 0u;
  for (int j = j0; j < j1; ++j) sum += pos[j] + pos[a.Ld + j] + pos[2 * a.Ld + j] + pos[3 * a.Ld + j];
  uint32_t incl = sum;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const uint32_t v = __shfl_up(incl, o);
    if (lane >= o) incl += v;
  }
  if (lane == 63) wtot[wave] = incl;
  __syncthreads();
  uint32_t at = incl - sum;
  for (int w = 0; w < wave; ++w) at += wtot[w];
  uint32_t* rows = a.dd_rows + ((int64_t)chunk * a.B + b) * a.Ld;
  for (int j = j0; j < j1; ++j) {
    const uint32_t first = at;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const uint32_t c = pos[w * a.Ld + j];
      pos[w * a.Ld + j] = at;
      at += c;
    }
    rows[j] = at > first ? first | ((at - first) << 16) : kNoRow;
  }
  __syncthreads();
  uint16_t* ent = a.dd_ent + (int64_t)b * NL + e0;
  const int nbits = a.Ld > 1 ? 32 - __builtin_clz((unsigned)(a.Ld - 1)) : 0;
  for (int pb = p0; pb < p1; pb += 64) {  // uniform over the wave
    const int p = pb + lane;
    const bool in = p < p1;
    const uint32_t j = in ? keys[p] : 0u;
    uint64_t same = __builtin_amdgcn_ballot_w64(in);  // lanes of this lane's row
    for (int bit = 0; bit < nbits; ++bit) {
      const bool one = (j >> bit) & 1u;
      const uint64_t ones = __builtin_amdgcn_ballot_w64(one);
      same &= one ? ones : ~ones;
    }
    if (in) {
      const uint32_t base = mypos[j];
      const int before = __builtin_popcountll(same & (((uint64_t)1 << lane) - 1));
      ent[base + before] = (uint16_t)p;
      // the row's last lane moves its next position on, once every lane has read it
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (same >> lane == 1u) mypos[j] = base + before + 1;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  }
}

// The same by a bitonic sort of the keys row << 13 | (e - e0) in LDS, for docs
// whose row counters do not fit there (kDdIndexLds).
__device__ __forceinline__ void dd_index_sort(const BwdArgs& a, int b, int chunk, uint32_t* keys) {
  const int NL = a.Nq * a.Lq;
  const int e0 = chunk * kDdChunk;
  const int n = NL - e0 < kDdChunk ? NL - e0 : kDdChunk;  // entries of this chunk
  const bool empty = a.lengths && doc_len(a, b) == 0;
  for (int p = threadIdx.x; p < a.sort_n; p += 256) {
    uint32_t key = kNoRow;
    if (p < n && !empty) {
      const int e = e0 + p;
      const int qi = e / a.Lq, q = e - qi * a.Lq;
      const int j = clamp_index(a.argmax[((int64_t)qi * a.B + b) * a.Lq + q], a.Ld);
      key = ((uint32_t)j << kEntryBits) | (uint32_t)p;
    }
    keys[p] = key;
  }
  __syncthreads();
  for (int size = 2; size <= a.sort_n; size <<= 1) {
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      for (int p = threadIdx.x; p < a.sort_n / 2; p += 256) {
        const int i = 2 * stride * (p / stride) + (p % stride);
        const int j = i + stride;
        const bool asc = (i & size) == 0;
        const uint32_t x = keys[i], y = keys[j];
        if ((x > y) == asc) {
          keys[i] = y;
          keys[j] = x;
        }
      }
      __syncthreads();
    }
  }
  uint16_t* ent = a.dd_ent + (int64_t)b * NL + e0;
  for (int p = threadIdx.x; p < n; p += 256) ent[p] = (uint16_t)(keys[p] & ((1u << kEntryBits) - 1));
  uint32_t* rows = a.dd_rows + ((int64_t)chunk * a.B + b) * a.Ld;
  for (int j = threadIdx.x; j < a.Ld; j += 256) {
    // first sorted position with row >= j (keys of empty slots are kNoRow)
    const uint32_t lo_key = (uint32_t)j << kEntryBits;
    int lo = 0, hi = n;
    while (lo < hi) {
      const int mid = (lo + hi) >> 1;
      if (keys[mid] < lo_key) lo = mid + 1; else hi = mid;
    }
    uint32_t info = kNoRow;
    if (lo < n && (keys[lo] >> kEntryBits) == (uint32_t)j) {
      int cnt = 1;
      while (lo + cnt < n && (keys[lo + cnt] >> kEntryBits) == (uint32_t)j) ++cnt;
      info = (uint32_t)lo | ((uint32_t)cnt << 16);
    }
    rows[j] = info;
  }
}

// dD writer: rows of [B, Ld, d] in memory order, a slab of consecutive rows
// per workgroup, so the stores stream like a fill of the whole tensor. A row
// no entry picked is zeros; a picked row is the fp32 sum over its entries, in
// entry order, of g[qi, b] * Q[qi, q]. Lanes cover a row's 8-wide k chunks:
// L = min(64, pow2 >= chunks) lanes per row, 64 / L rows per wave pass.
//
// Sparse rows (one query) are bound by the stores, and take one entry at a
// time. DENSE, rows that many entries picked (a batch of queries over short
// docs: 200 a row), are a serial chain, as the sum keeps entry order: the L
// lanes of a row therefore fetch L entries at a time, each lane one entry's
// number, Q row and gradient, the next L while the current ones are summed, and
// the Q rows themselves come up to kDdAhead at a time (an entry at a time is a
// chain of three memory round trips each: 32 queries of 32 tokens over 256 docs
// of up to 180 tokens 84 -> 25 us). Rows of one or two entries gain nothing
// from that, so a wave whose rows all have so few takes them singly here too.
// kDdAhead: eight rows ahead cost a third of the waves (five per SIMD, seven
// with four: 1000 docs of 512 x 1024 under 256 tokens 357 -> 323 us, 4000 of
// 300 x 128 under 200 144 -> 128; the smallest batches 35 -> 38).
constexpr int kDdAhead = 4;
template <bool BF, bool DENSE, int OUT>
__device__ __forceinline__ void dd_write_block(const BwdArgs& a, int64_t slab) {
  const int nkc = (a.d + 7) >> 3;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int lsh = 0;
  while ((1 << lsh) < nkc && lsh < 6) ++lsh;
  const int L = 1 << lsh;
  const int rpw = 64 >> lsh;               // rows per wave pass
  const int sub = lane >> lsh;             // this lane's row within the pass
  const int kc0 = lane & (L - 1);
  const int64_t total = (int64_t)a.B * a.Ld;
  const int64_t r0 = slab * a.dd_slab;
  const int64_t r1 = r0 + a.dd_slab < total ? r0 + a.dd_slab : total;
  const int step = 4 * rpw;
  // the lane's elements p0 .. p0+3 and p1 .. p1+3 of the row's part from 8 * kb on
  auto at = [&](int kb, int h) { return OUT == OUT_F32 ? 8 * kb + 4 * (h * L + kc0) : 8 * (kb + kc0) + 4 * h; };
  int64_t r = r0 + wave * rpw + sub;
  int b = (int)(r / a.Ld);
  int j = (int)(r - (int64_t)b * a.Ld);
  const int NL = a.Nq * a.Lq;
  const uint16_t* Q = static_cast<const uint16_t*>(a.Q);
  const float zero[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // The row-index entries of all of this lane's passes (a slab is at most
  // kDdMaxPasses of them) are loaded up front, so their round trips overlap.
  uint32_t infos[kDdMaxPasses];
#pragma unroll
  for (int p = 0; p < kDdMaxPasses; ++p) {
    const int64_t rp = r + (int64_t)p * step;
    infos[p] = rp < r1 ? a.dd_rows[rp] : kNoRow;
  }
#pragma unroll
  for (int p = 0; p < kDdMaxPasses; ++p, r += step) {
    if (r >= r1) break;
    void* orow = static_cast<char*>(a.dD) + r * a.d * (OUT == OUT_F32 ? 4 : 2);
    const uint32_t info0 = infos[p];
    if (a.dd_chunks == 1 && info0 == kNoRow) {
      for (int kb = 0; at(kb, 0) < a.d; kb += 64) store8<BF, OUT>(orow, at(kb, 0), at(kb, 1), a.d, zero);
    } else if (!DENSE || (a.dd_chunks == 1 &&
                          __builtin_amdgcn_ballot_w64(info0 != kNoRow && (info0 >> 16) > 2u) == 0)) {
      for (int kb = 0; at(kb, 0) < a.d; kb += 64) {
        const int p0 = at(kb, 0), p1 = at(kb, 1);
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        // the row's entries chunk by chunk: entry order overall
        for (int ch = 0; ch < a.dd_chunks; ++ch) {
          const uint32_t info = ch == 0 ? info0 : a.dd_rows[(int64_t)ch * total + r];
          if (info == kNoRow) continue;
          const int e0 = ch * kDdChunk;
          const uint16_t* ent = a.dd_ent + (int64_t)b * NL + e0 + (info & 0xffffu);
          const int n = (int)(info >> 16);
          for (int i = 0; i < n; ++i) {
            const int e = e0 + ent[i];
            const int qi = e / a.Lq, q = e - qi * a.Lq;
            const float g = a.grad[(int64_t)qi * a.g_n + (int64_t)b * a.g_b];
            float x[8];
            load8<BF, OUT>(Q + (int64_t)qi * a.sq_n + (int64_t)q * a.sq_l, p0, p1 < a.d ? p1 : p0, x);
#pragma unroll
            for (int k = 0; k < 8; ++k) acc[k] = fmaf(g, x[k], acc[k]);
          }
        }
        store8<BF, OUT>(orow, p0, p1, a.d, acc);
      }
    } else if constexpr (DENSE) {
      // every lane of the row takes part in each step below, those past its
      // last k chunk too (they fetch entries; their loads repeat chunk 0)
      for (int kb = 0; kb < nkc; kb += 64) {
        const int p0 = at(kb, 0), p1 = at(kb, 1);
        const bool live = p0 < a.d;
        const int l0 = live ? p0 : 0, l1 = p1 < a.d ? p1 : l0;  // places to load from
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        // the row's entries chunk by chunk: entry order overall
        for (int ch = 0; ch < a.dd_chunks; ++ch) {
          const uint32_t info = ch == 0 ? info0 : a.dd_rows[(int64_t)ch * total + r];
          if (info == kNoRow) continue;
          const int e0 = ch * kDdChunk;
          const uint16_t* ent = a.dd_ent + (int64_t)b * NL + e0 + (info & 0xffffu);
          const int n = (int)(info >> 16);
          // entry i0 + kc0 of the row: its Q row's offset in 8-element units
          // (query strides are multiples of 8) and its gradient
          auto fetch = [&](int i0, uint32_t& off, float& g) __attribute__((always_inline)) {
            off = 0u;
            g = 0.f;
            if (i0 + kc0 < n) {
              const int e = e0 + ent[i0 + kc0];
              const int qi = e / a.Lq, q = e - qi * a.Lq;
              off = (uint32_t)(((int64_t)qi * a.sq_n + (int64_t)q * a.sq_l) >> 3);
              g = a.grad[(int64_t)qi * a.g_n + (int64_t)b * a.g_b];
            }
          };
          auto add = [&](auto count_tag, uint32_t off, float g, int u0) __attribute__((always_inline)) {
            constexpr int U = decltype(count_tag)::value;
            float x[U][8], gu[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
              const int src = (lane & ~(L - 1)) + u0 + u;
              const uint16_t* row = Q + (int64_t)lane_fetch(off, src) * 8;
              gu[u] = __builtin_bit_cast(float, lane_fetch(__builtin_bit_cast(uint32_t, g), src));
              load8<BF, OUT>(row, l0, l1, x[u]);
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
              for (int k = 0; k < 8; ++k) acc[k] = fmaf(gu[u], x[u][k], acc[k]);
          };
          uint32_t off, noff = 0u;
          float g, ng = 0.f;
          fetch(0, off, g);
          for (int i0 = 0; i0 < n; i0 += L) {
            const int m = n - i0 < L ? n - i0 : L;
            if (i0 + L < n) fetch(i0 + L, noff, ng);
            int u0 = 0;
            for (; u0 + kDdAhead <= m; u0 += kDdAhead) add(std::integral_constant<int, kDdAhead>{}, off, g, u0);
            for (; u0 + 2 <= m; u0 += 2) add(std::integral_constant<int, 2>{}, off, g, u0);
            if (u0 < m) add(std::integral_constant<int, 1>{}, off, g, u0);
            off = noff;
            g = ng;
          }
        }
        if (live) store8<BF, OUT>(orow, p0, p1, a.d, acc);
      }
    }
    j += step;
    while (j >= a.Ld) {
      j -= a.Ld;
      ++b;
    }
  }
}

// The backward is two launches. Each carries a small part of one gradient
// beside the large part of the other, which it does not depend on, so the
// small parts cost neither a launch nor time of their own:
//   front: the dQ gather (the first n_gather workgroups) and the dD index,
//   back:  the dQ sum (the first n_sum workgroups) and the dD writer.
// The gather and the writer do not share a launch: reads of D beside the
// stores of dD lower the rate of both (interleaved in one grid 15 % slower; on
// two streams 4 % slower than this with 1000 docs of 512 x 1024, and its event
// waits cost 20 us where dD is 77 MB, 41.8 -> 24.0 us). The gather comes first and
// the index workgroups start as it leaves room. One dynamic LDS size serves both
// parts, so the gather's workgroups reserve the index's up to 64 KB too; that still
// costs less than a launch for each. Both gradients, gather first / index first /
// two launches (us), and the index's LDS: 64 x 64 tokens over 1000 docs of 1100 x
// 128 237 / 296 / 269, 34 KB; over 64 of 2000 x 128 57.8 / 55.5 / 66.4, 48 KB; 128 x
// 64 over 300 of 300 x 128 177 / 183 / 208, 38 KB; 32 over 5000 of 300 x 128 94 / 102
// / 106, 5 KB.
template <bool BF, bool COUNT>
__global__ void __launch_bounds__(256) bwd_front_kernel(BwdArgs a, unsigned n_gather, unsigned gather_x,
                                                        unsigned index0) {
  extern __shared__ uint32_t smem[];
  const unsigned x = blockIdx.x;
  if (x < n_gather) {
    // wave-uniform on purpose: the chunk's lengths then come by scalar loads
    const int by = __builtin_amdgcn_readfirstlane((int)(x / gather_x));
    dq_partial_block<BF>(a, x - (unsigned)by * gather_x, by);
  } else {
    const unsigned y = index0 + (x - n_gather);
    const int b = (int)(y % (unsigned)a.B), chunk = (int)(y / (unsigned)a.B);
    if constexpr (COUNT) {
      dd_index_count(a, b, chunk, smem);
    } else {
      dd_index_sort(a, b, chunk, smem);
    }
  }
}

template <bool BF, bool DENSE, int OUT>
__global__ void __launch_bounds__(256) bwd_back_kernel(BwdArgs a, unsigned n_sum) {
  const unsigned x = blockIdx.x;
  if (x < n_sum) {
    dq_sum_block<BF, OUT>(a, x);
  } else {
    dd_write_block<BF, DENSE, OUT>(a, x - n_sum);
  }
}

// Which writer: the dense one from an entry a row, or from two entries to five
// rows where docs have lengths, whose entries then crowd fewer rows. dD alone,
// one entry at a time against dense (us), docs all long / of U[Ld/32, Ld]
// tokens, 128 MiB of dD at d = 128:
//   300 tokens, entries a row 0.21: 36.3 / 33.9 against 41.4 / 36.7, 0.43: 43.7
//   / 40.9 against 47.8 / 40.3, 0.85: 54.0 / 51.8 against 53.0 / 44.2, 1.7: 69.6
//   / 74.0 against 59.1 / 51.6, 6.8: 158 / 206 against 104 / 103;
//   77 tokens, 27: 451 / 745 against 236 / 291; d = 1024 and 300 tokens, 3.4:
//   70 / 177 against 51 / 55.
// Rows of one chunk have one lane, which nothing is fetched ahead for: one entry at
// a time (d = 8, 32 x 32 over 100 ragged docs of 60 tokens 538 -> 312 us, d = 12 251
// against 269).
// The dense writer keeps the place of a Q row in 32 bits, in units of 8 elements;
// queries that span more than 2^35 elements (views far apart) take the other.
inline bool dd_dense(const BwdArgs& a) {
  if (a.d <= 8 || a.sq_n < 0 || (a.Nq - 1) * a.sq_n + a.Lq * a.sq_l > ((int64_t)1 << 35)) return false;
  return 5 * (int64_t)a.Nq * a.Lq > (a.lengths ? 2 : 5) * (int64_t)a.Ld;
}

// Unused LDS that keeps the writer, a stream of stores, to seven workgroups per
// CU: more spread the stores over more of dD than the memory takes well, fewer
// leave it waiting (step of 1000 docs of 512 x 1024, eight to five workgroups:
// 410-420, 396, 402, 415 us). dD alone over 13 other shapes of d = 64 to 384, fp16
// and fp32, long and ragged, against none: within 2 % for most, from 121 -> 105 us
// (256 tokens over 2000 ragged docs of 1100 x 128) and 44.6 -> 39.7 (8 x 32 over 500
// of 1000 x 100) to 104 -> 112 (the former docs all long).
constexpr size_t kWriterLds = 23000;
constexpr int64_t kBwdMaxBlocks = ((int64_t)1 << 24) - 1;  // workgroups of 256 threads per launch

template <bool BF>
hipError_t launch_front(const BwdArgs& a, int64_t n_index, int64_t n_gather, hipStream_t s) {
  if (n_index + n_gather == 0) return hipSuccess;
  if (n_index > UINT32_MAX) return hipErrorInvalidValue;
  const size_t keys = n_index ? (size_t)a.sort_n * sizeof(uint32_t) : 0;
  const bool count = keys + dd_count_bytes(a.Ld) <= kDdIndexLds;
  const size_t lds = n_index ? keys + (count ? dd_count_bytes(a.Ld) : 0) : 0;
  auto kern = count ? bwd_front_kernel<BF, true> : bwd_front_kernel<BF, false>;
  const int64_t gather_x = n_gather ? n_gather / a.nchunk : 1;
  // one launch, and more for the index workgroups past a launch's limit
  for (int64_t first = 0; n_gather || first < n_index; n_gather = 0) {
    const int64_t room = kBwdMaxBlocks - n_gather, rest = n_index - first;
    const int64_t n = rest < room ? rest : room > 0 ? room : 0;
    hipLaunchKernelGGL(kern, dim3((unsigned)(n_gather + n)), dim3(256), lds, s, a, (unsigned)n_gather,
                       (unsigned)gather_x, (unsigned)first);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    first += n;
  }
  return hipSuccess;
}

template <bool BF>
hipError_t launch_back(const BwdArgs& a, int64_t n_sum, int64_t n_write, hipStream_t s) {
  if (n_sum + n_write == 0) return hipSuccess;
  if (n_sum + n_write > kBwdMaxBlocks && n_sum && n_write) {
    const hipError_t e = launch_back<BF>(a, n_sum, 0, s);
    return e != hipSuccess ? e : launch_back<BF>(a, 0, n_write, s);
  }
  const bool dense = dd_dense(a);
  auto kern = (a.d & 7) == 0 ? (dense ? bwd_back_kernel<BF, true, OUT_H8> : bwd_back_kernel<BF, false, OUT_H8>)
                             : (dense ? bwd_back_kernel<BF, true, OUT_H> : bwd_back_kernel<BF, false, OUT_H>);
  if constexpr (!BF) {
    if (a.out_f32) kern = dense ? bwd_back_kernel<BF, true, OUT_F32> : bwd_back_kernel<BF, false, OUT_F32>;
  }
  hipLaunchKernelGGL(kern, dim3((unsigned)(n_sum + n_write)), dim3(256),
                     kWriterLds, s, a, (unsigned)n_sum);
  return hipGetLastError();
}

template <bool BF>
hipError_t launch_bwd_t(const BwdArgs& a, hipStream_t s) {
  const bool do_dd = a.dD && a.B > 0;
  const int64_t rows = (int64_t)a.Nq * a.Lq;
  const int64_t n_index = do_dd ? (int64_t)a.B * a.dd_chunks : 0;
  const int64_t n_gather = a.dQ ? (rows * ((a.d + 7) >> 3) + 255) / 256 * a.nchunk : 0;
  const int64_t n_sum = a.dQ ? (rows * a.d + 255) / 256 : 0;
  const int64_t n_write = do_dd ? ((int64_t)a.B * a.Ld + a.dd_slab - 1) / a.dd_slab : 0;
  const hipError_t e = launch_front<BF>(a, n_index, n_gather, s);
  return e != hipSuccess ? e : launch_back<BF>(a, n_sum, n_write, s);
}

}  // namespace

// Doc chunks of the dQ gather: about 2^17 (row, k-chunk, doc-chunk) threads,
// at most 64 chunks, at least 8 docs each. Each thread keeps 8 gathers in
// flight, so fewer, longer chunks keep the loads going with less partial-sum
// traffic (config 5, 8 chunks: step 437 us; 16: 439; 32: 444).
int bwd_dq_chunks(int B, int rows, int d) {
  if (B <= 0) return 1;
  const int64_t per_chunk = (int64_t)rows * ((d + 7) / 8);
  int64_t n = ((int64_t)1 << 17) / (per_chunk > 0 ? per_chunk : 1);
  const int64_t by_docs = (B + 7) / 8;
  if (n > by_docs) n = by_docs;
  if (n > 64) n = 64;
  if (n < 1) n = 1;
  return (int)n;
}

// Sort size of one dD index chunk: a power of two >= the chunk's entries.
int bwd_sort_n(int64_t entries) {
  int n = 64;
  while (n < entries && n < kDdChunk) n <<= 1;
  return n;
}

int64_t bwd_dd_chunks(int64_t entries) { return entries > 0 ? (entries + kDdChunk - 1) / kDdChunk : 1; }

// Workspace of the dD index: rows [chunks, B, Ld] uint32, then ent [B, entries] uint16.
size_t bwd_dd_index_bytes(int64_t B, int64_t entries, int64_t Ld) {
  const size_t rows = (size_t)bwd_dd_chunks(entries) * (size_t)B * (size_t)Ld * sizeof(uint32_t);
  return rows + (((size_t)B * (size_t)entries * sizeof(uint16_t) + 255) & ~(size_t)255);
}

// Rows per dD writer workgroup: about 16 KB of output, a whole number of
// the workgroup's row passes (4 waves x 64 / L rows, L lanes per row), at
// most kDdMaxPasses of them.
int bwd_dd_slab(int d) {
  const int nkc = (d + 7) / 8;
  int lsh = 0;
  while ((1 << lsh) < nkc && lsh < 6) ++lsh;
  const int pass = 4 * (64 >> lsh);
  int rows = 16384 / (2 * d);
  if (rows < pass) rows = pass;
  if (rows > kDdMaxPasses * pass) rows = kDdMaxPasses * pass;
  return (rows + pass - 1) / pass * pass;
}

hipError_t launch_bwd(int kind, const BwdArgs& a, hipStream_t s) {
  switch (kind) {
    case KIND_F16: return launch_bwd_t<false>(a, s);
    case KIND_BF16: return launch_bwd_t<true>(a, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fmx
