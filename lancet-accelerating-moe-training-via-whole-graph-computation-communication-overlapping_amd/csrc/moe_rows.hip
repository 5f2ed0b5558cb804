// Row movers: scatter of token rows into the [E,C,M] expert buffer, weighted gather-combine
// back, partition merge of masks and buffers, and the gradients of both.  All are pure HBM streaming: rows
// shared by part of a wave, a wave or several, 16-byte accesses, every output byte written once (but for the
// bytes that two granules of a row share which ends inside one: written twice, with the same value).
#include "launchers.hpp"
#include "common.hpp"
#include "../../include/lancet_hip.h"
#include <algorithm>

namespace lancet {

constexpr int kRowsPerBlock = kTile / kWave;  // waves per workgroup; a wave moves a row or a share of one
constexpr int kTailRows = 16;                 // rows zero-filled by one tail workgroup

// A load that is issued where it stands: the compiler moves an ordinary one down to its use, behind other waits and
// branches.  (A relaxed atomic of the narrowest scope is the same instruction.)
template <typename T>
__device__ __forceinline__ T ld_now(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WAVEFRONT);
}

// 2^q lanes share a row: part of a wave, a wave or several.  (Rows of less than a wave used to take a whole one: rows of
// 512 bytes, 131072 of them, decode top-1 41 -> 24 us, decode_dx 54 -> 30, decode_dg 39 -> 22, scatter 29 -> 23; rows of 1 KB
// at two granules per lane, 262144 of them, decode 83 -> 69.)  The thread's row, its place among the row's lanes and the
// distance in granules between the ones it moves.  Neighbouring lanes and waves move neighbouring granules in row order:
// short waves in row order keep the chip-wide streams close to address order, which the memory system rewards.
struct RowShare {
  int r, v, step;
};
__device__ __forceinline__ RowShare row_share(int q, uint32_t block) {
  const uint64_t t = static_cast<uint64_t>(block) * kTile + threadIdx.x;
  RowShare h;
  h.r = static_cast<int>(t >> q);
  h.step = 1 << q;
  h.v = static_cast<int>(static_cast<uint32_t>(t) & static_cast<uint32_t>(h.step - 1));
  return h;
}
__device__ __forceinline__ RowShare row_share(int q) { return row_share(q, blockIdx.x); }
// sum over the row's lanes inside a wave
__device__ __forceinline__ float share_sum(float x, int q) {
  if (q >= 6) return wave_sum(x);
  for (int o = 1 << q >> 1; o > 0; o >>= 1) x += __shfl_xor(x, o, kWave);
  return x;
}

// How a row is cut into the pieces its lanes move:
//   kWhole16  16-byte granules, rows and pointers aligned to them;
//   kAny16    rows of at least 16 bytes that end anywhere and start wherever their elements are aligned: 16-byte
//             granules at unaligned addresses (the hardware takes them), the last one drawn back so that it ends with
//             the row.  Its first bytes are then moved twice, with the same values.  At 10007 rows of 1003 bf16 values
//             (60 experts, top-2) the scatter takes 13 us this way and 44 an element per lane, the decode 10 and 26;
//   kElem2 / kElem4  one element per lane: rows of less than 16 bytes.
// Loads: non-temporal (ld), except where rows come twice (ld_keep: the top-2 decode_dx reads every token row for both
// slots, 402 -> 380 us at 65536 x 4096 bf16 and 39 -> 33 at 16384 x 1024 fp32; top-1 reads it once, 199 against 206) and
// in the scatter (65536 x 4096 top-2 312 -> 307, 16384 x 2048 top-2 40 -> 36, nowhere slower).  The decode and the dot
// products read every row once: 259 against 280 and 321 against 346 us with plain loads.  Stores are non-temporal
// (plain: scatter 304 there, but 38 against 33 at 16384 x 1024 fp32 and 211 against 203 top-1).  Unaligned granules
// share lines with their neighbours and are accessed plainly (10007 x 1003 bf16 scatter 13 against 16 us).
enum RowMode { kWhole16, kAny16, kElem2, kElem4 };
typedef u32x4 u32x4_any __attribute__((aligned(2)));

template <int MODE>
struct Granule {
  typedef u32x4 V;
  static __device__ __forceinline__ uint32_t at(int v, uint32_t) { return 16u * static_cast<uint32_t>(v); }
  static __device__ __forceinline__ V ld(const char* p) { return __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p)); }
  static __device__ __forceinline__ V ld_keep(const char* p) { return *reinterpret_cast<const u32x4*>(p); }
  static __device__ __forceinline__ void st(LANCET_GLOBAL char* p, V x) { __builtin_nontemporal_store(x, (LANCET_GLOBAL u32x4*)p); }
  static __device__ __forceinline__ V zero() { return u32x4{0u, 0u, 0u, 0u}; }
};
template <>
struct Granule<kAny16> {
  typedef u32x4 V;
  static __device__ __forceinline__ uint32_t at(int v, uint32_t row_bytes) { return min(16u * static_cast<uint32_t>(v), row_bytes - 16u); }
  static __device__ __forceinline__ V ld(const char* p) { return *reinterpret_cast<const u32x4_any*>(p); }
  static __device__ __forceinline__ V ld_keep(const char* p) { return ld(p); }
  static __device__ __forceinline__ void st(LANCET_GLOBAL char* p, V x) { *(LANCET_GLOBAL u32x4_any*)p = x; }
  static __device__ __forceinline__ V zero() { return u32x4{0u, 0u, 0u, 0u}; }
};
// 16-byte granules of a row of 16 bytes or more (up to 4 GB, where adding first would wrap)
__device__ __forceinline__ int granules_of(uint32_t row_bytes) { return static_cast<int>((row_bytes - 1u) / 16u + 1u); }
template <typename E>
struct GranuleElem {
  typedef E V;
  static __device__ __forceinline__ uint32_t at(int v, uint32_t) { return static_cast<uint32_t>(sizeof(E)) * static_cast<uint32_t>(v); }
  static __device__ __forceinline__ V ld(const char* p) { return __builtin_nontemporal_load(reinterpret_cast<const E*>(p)); }
  static __device__ __forceinline__ V ld_keep(const char* p) { return ld(p); }
  static __device__ __forceinline__ void st(LANCET_GLOBAL char* p, V x) { __builtin_nontemporal_store(x, (LANCET_GLOBAL E*)p); }
  static __device__ __forceinline__ V zero() { return E(0); }
};
template <>
struct Granule<kElem2> : GranuleElem<uint16_t> {};
template <>
struct Granule<kElem4> : GranuleElem<uint32_t> {};

// ---------------------------------------------------------------------------------------
// encode_forward: out[idx, loc, :] = data[s, :]; rows no token lands on are zero.
// Replaces cudaMemsetAsync + atomicAdd per element of
// src/op/dialect/cuda/kernels/tutel_moe_dispatch.cu:61-81,461-484.
// ---------------------------------------------------------------------------------------
struct ScatterArgs {
  const char* data;
  char* out;
  const int32_t* idx;         // [K*S]
  const int32_t* loc;         // [K*S]
  const int32_t* dest;        // [K*S] or null: destination row e * C + location (-1: none) in ONE word per slot,
                              // instead of idx / loc / avail_used / row_base
  const int32_t* avail_used;  // [E] or null
  const int32_t* row_base;    // [E] or null: row of expert e that location 0 maps to
  const int32_t* rows_lo;     // [E] or null
  const int32_t* rows_hi;     // [E] or null (no tail fill)
  int S, E, C, K;
  int slot_stride;            // distance between the slots of one token in idx / loc (S, or the whole batch's
                              // token count when this call moves a token range of a larger mask)
  uint32_t row_bytes;
  int row_vecs;               // granules per row
  int q;                      // 2^q lanes share one token row
  int token_blocks;
  int tail_chunks;            // tail workgroups per expert
  int tail_groups;            // eights of tail workgroups that stand among the tokens', 0 = all stand behind them
  int tail_every;             // ... one in this many eights, two at least
  uint32_t tail_inverse;      // 2^32 / tail_every, rounded up
};

constexpr int kXcds = 8;  // workgroups go round them: what comes in turns comes in eights, or a few XCDs do all of it

template <int MODE, int K, bool DEST = false>
__global__ __launch_bounds__(kTile) void scatter_rows_kernel(ScatterArgs a) {
  typedef Granule<MODE> G;
  typedef typename G::V V;
  int token = static_cast<int>(blockIdx.x), tail = token - a.token_blocks;  // tail: negative in a workgroup of tokens
  if (a.tail_groups) {
    // (a division would stand in front of every workgroup's first load: top-1 scatters with tails that are mostly empty 1.03 against 1.06
    // of the time they take with the tails behind)
    const int eight = token / kXcds, turn = static_cast<int>(__umulhi(static_cast<uint32_t>(eight), a.tail_inverse));
    const bool clears = turn < a.tail_groups && eight - turn * a.tail_every == a.tail_every - 1;
    tail = clears ? turn * kXcds + token % kXcds : -1;
    token -= kXcds * min(turn, a.tail_groups);
  }
  if (tail < 0) {
    const RowShare h = row_share(a.q, static_cast<uint32_t>(token));
    const int s = h.r, step = h.step;
    int v = h.v;
    if (s >= a.S) return;
    // The row's granules do not depend on the routing, only their destinations do: the first loads of the row
    // go out before idx / loc are known, so that a wave waits for the longer of the two latencies and not for
    // their sum (a dropped token's row is then read for nothing).  338 -> 333 us at the headline shape.
    const char* src = a.data + static_cast<size_t>(s) * a.row_bytes;
    const bool has0 = v < a.row_vecs, has1 = v + step < a.row_vecs;
    const uint32_t o0 = G::at(v, a.row_bytes), o1 = G::at(v + step, a.row_bytes);
    V x0 = G::zero(), x1 = G::zero();
    if (has0) x0 = G::ld_keep(src + o0);
    if (has1) x1 = G::ld_keep(src + o1);
    // destinations picked at run time: typed as global memory so the stores are not flat.  (The routing words of a
    // row are the same for every lane; loading them through the scalar cache, or forming the row addresses on the
    // scalar unit from vector-loaded words, was measured slower: 346 and 340 us against 333 at the headline shape.)
    LANCET_GLOBAL char* dst[K];
    int es[K], ls[K];
    if (!DEST) {
#pragma unroll
      for (int j = 0; j < K; ++j) {
        es[j] = ld_now(a.idx + static_cast<size_t>(j) * a.slot_stride + s);
        ls[j] = ld_now(a.loc + static_cast<size_t>(j) * a.slot_stride + s);
      }
    }
    int nd = 0;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (DEST) {
        const int d = a.dest[static_cast<size_t>(j) * a.slot_stride + s];
        dst[j] = as_global(a.out);
        if (d >= 0 && d < a.E * a.C) dst[nd++] = as_global(a.out + static_cast<size_t>(d) * a.row_bytes);
        continue;
      }
      const int e = es[j];
      int l = ls[j];
      bool ok = (e >= 0) & (e < a.E) & (l >= 0) & (l < a.C);
      if (ok && a.avail_used) ok = l < a.C - a.avail_used[e];
      dst[j] = as_global(a.out);
      if (ok && a.row_base) {
        l += a.row_base[e];
        ok = l < a.C;
      }
      if (ok) dst[nd++] = as_global(a.out + (static_cast<size_t>(e) * a.C + l) * a.row_bytes);
    }
    if (nd == 0) return;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      if (j < nd) {
        if (has0) G::st(dst[j] + o0, x0);
        if (has1) G::st(dst[j] + o1, x1);
      }
    }
    for (v += 2 * step; v < a.row_vecs; v += step) {
      const uint32_t o = G::at(v, a.row_bytes);
      const V x = G::ld_keep(src + o);
#pragma unroll
      for (int j = 0; j < K; ++j)
        if (j < nd) G::st(dst[j] + o, x);
    }
  } else {
    // tail: zero rows [used, C) of expert e, kTailRows rows per workgroup and turn
    const int e = tail / a.tail_chunks;
    const int ch = tail - e * a.tail_chunks;
    if (e >= a.E) return;  // the last eight may be more than there are
    const int used = a.rows_hi[e] - (a.rows_lo ? a.rows_lo[e] : 0);
    // the rows lie one behind the other: one run of granules, or one per row where the run's length takes more than 32 bits
    const uint32_t rows = a.row_bytes <= 0xffffffffu / kTailRows ? kTailRows : 1;
    const uint32_t C = static_cast<uint32_t>(a.C), stride = static_cast<uint32_t>(a.tail_chunks) * kTailRows;
    for (uint32_t first = static_cast<uint32_t>(max(used, 0)) + static_cast<uint32_t>(ch) * kTailRows; first < C; first += stride) {
      const uint32_t last = min(first + kTailRows, C);
      for (uint32_t r = first; r < last; r += rows) {
        LANCET_GLOBAL char* run = as_global(a.out + (static_cast<size_t>(e) * a.C + r) * a.row_bytes);
        const uint32_t bytes = min(rows, last - r) * a.row_bytes;
        const uint32_t n = static_cast<uint32_t>((bytes + sizeof(V) - 1) / sizeof(V));
        for (uint32_t v = threadIdx.x; v < n; v += kTile) G::st(run + G::at(v, bytes), G::zero());
      }
    }
  }
}

__global__ void zero_bytes_kernel(u32x4* p, size_t nvec, uint8_t* tail, size_t ntail) {
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  const u32x4 z = {0u, 0u, 0u, 0u};
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < nvec; i += stride)
    __builtin_nontemporal_store(z, p + i);
  if (blockIdx.x == 0 && threadIdx.x < ntail) tail[threadIdx.x] = 0;
}

// ---------------------------------------------------------------------------------------
// decode_forward: out[s,:] = sum_j gates[j*S+s] * expert_out[idx, loc, :], fp32 products and
// sum (no fused multiply-add, so that the result is one well-defined rounding sequence), one
// rounding to the storage type.  Replaces tutel_moe_dispatch.cu:46-55,110-116,511-521.
// ---------------------------------------------------------------------------------------
template <int DT>
struct Codec;
template <>
struct Codec<LANCET_F32> {
  typedef uint32_t S;  // scalar storage
  static constexpr int kPerVec = 4;
  static __device__ __forceinline__ float get(S x) { return __uint_as_float(x); }
  static __device__ __forceinline__ S put(float f) { return __float_as_uint(f); }
};
template <>
struct Codec<LANCET_BF16> {
  typedef uint16_t S;
  static constexpr int kPerVec = 8;
  static __device__ __forceinline__ float get(S x) { return bf16_to_f32(x); }
  static __device__ __forceinline__ S put(float f) { return static_cast<S>(f32_to_bf16(f)); }
};
template <>
struct Codec<LANCET_F16> {
  typedef uint16_t S;
  static constexpr int kPerVec = 8;
  static __device__ __forceinline__ float get(S x) { return f16_to_f32(x); }
  static __device__ __forceinline__ S put(float f) { return static_cast<S>(f32_to_f16(f)); }
};

// One IEEE multiply / add each, never contracted into a fused multiply-add (the operators of
// the HIP headers' __fmul_rn/__fadd_rn carry the translation unit's contraction setting).
__device__ __forceinline__ float mul_rn(float a, float b) {
#pragma clang fp contract(off)
  return a * b;
}
__device__ __forceinline__ float add_rn(float a, float b) {
#pragma clang fp contract(off)
  return a + b;
}

template <int DT, int K>
__device__ __forceinline__ u32x4 combine_vec(const u32x4 (&x)[K], const float (&g)[K]) {
#pragma clang fp contract(off)
  typedef Codec<DT> Cd;
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (Cd::kPerVec == 4) {
      float acc = mul_rn(g[0], Cd::get(x[0][i]));
      if (K == 2) acc = add_rn(acc, mul_rn(g[1], Cd::get(x[1][i])));
      r[i] = Cd::put(acc);
    } else {
      float lo = mul_rn(g[0], Cd::get(static_cast<typename Cd::S>(x[0][i] & 0xffffu)));
      float hi = mul_rn(g[0], Cd::get(static_cast<typename Cd::S>(x[0][i] >> 16)));
      if (K == 2) {
        lo = add_rn(lo, mul_rn(g[1], Cd::get(static_cast<typename Cd::S>(x[1][i] & 0xffffu))));
        hi = add_rn(hi, mul_rn(g[1], Cd::get(static_cast<typename Cd::S>(x[1][i] >> 16))));
      }
      r[i] = static_cast<uint32_t>(Cd::put(lo)) | (static_cast<uint32_t>(Cd::put(hi)) << 16);
    }
  }
  return r;
}

// A gate value as it lies in memory: the aligned word that holds it.  (A 16-bit value's word may reach two bytes past
// either end of the array, never past an aligned word of it.)
struct GateWord {
  uint32_t w, shift;
  __device__ __forceinline__ void load(const void* p, size_t i, int gd) {
    const char* at = static_cast<const char*>(p) + (i << (gd == 0 ? 2 : 1));
    const uint32_t odd = static_cast<uint32_t>(reinterpret_cast<uintptr_t>(at)) & 2u;
    w = ld_now(reinterpret_cast<const uint32_t*>(at - odd));
    shift = odd * 8u;
  }
  __device__ __forceinline__ float value(int gd) const {
    const uint32_t h = w >> shift;
    return gd == 0 ? __uint_as_float(w) : gd == 1 ? bf16_to_f32(h) : f16_to_f32(h & 0xffffu);
  }
};

// routing words and combine weights of a token's K slots
template <int K>
struct RowWords {
  int e[K], l[K];
  GateWord g[K];
  bool unit;  // no gates: every weight is one
  int gd;
  __device__ __forceinline__ void load(const int32_t* idx, const int32_t* loc, const void* gates, int gate_dtype, int stride, int s) {
    load_dest(idx, gates, gate_dtype, stride, s);
#pragma unroll
    for (int j = 0; j < K; ++j) l[j] = ld_now(loc + static_cast<size_t>(j) * stride + s);
  }
  __device__ __forceinline__ void load_dest(const int32_t* dest, const void* gates, int gate_dtype, int stride, int s) {
    unit = gates == nullptr;
    gd = unit ? 0 : gate_dtype;
    const void* gp = unit ? static_cast<const void*>(dest) : gates;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      e[j] = ld_now(dest + static_cast<size_t>(j) * stride + s);
      l[j] = 0;
      g[j].load(gp, static_cast<size_t>(j) * stride + s, gd);
    }
  }
  __device__ __forceinline__ float weight(int j, bool ok) const { return ok ? (unit ? 1.f : g[j].value(gd)) : 0.f; }
};

// (Granules per lane: one for top-2, two for top-1, so that a wave has two row loads in flight either way.  65536 x 4096
// bf16: top-2 264 us with one, 270 with two, 273 with four; top-1 193 / 177 / 188.  Two for top-2 as well where a row of
// more than a wave would leave lanes idle, which is to say where it has no power of two of granules: 32768 x 2560 bf16 105.1
// with one, 83.6 with two, 32768 x 3072 113.0 and 98.3, 32768 x 4096 130.0 and 132.3.)
struct DecodeArgs {
  const void* expert_out;
  const void* gates;     // [K*S] of gate_dtype; null = all ones (moe_encode_dx)
  int gate_dtype;
  const int32_t* idx;    // [K*S]
  const int32_t* loc;    // [K*S]
  const int32_t* dest;   // [K*S] or null: row e * C + location of the slot (-1: none) instead of idx / loc
  void* out;             // [S, M]
  int S, M, E, C;
  int slot_stride;       // distance between the slots of one token in gates / idx / loc
  int q;                 // 2^q lanes share one token row
};

template <int DT, int K, int MODE, bool DEST = false>
__global__ __launch_bounds__(kTile) void decode_rows_kernel(DecodeArgs a) {
  typedef Codec<DT> Cd;
  const RowShare h = row_share(a.q);
  const int s = h.r, step = h.step;
  if (s >= a.S) return;
  // Everything a row's addresses and weights come from is asked for at once and without a branch in between: asked
  // for one after the other, each behind the test of the one before, the three words of a slot are three round trips
  // to memory in front of the row's own.
  RowWords<K> words;
  if (DEST) words.load_dest(a.dest, a.gates, a.gate_dtype, a.slot_stride, s);
  else words.load(a.idx, a.loc, a.gates, a.gate_dtype, a.slot_stride, s);
  size_t row[K];
  bool ok[K];
  bool any = false;
#pragma unroll
  for (int j = 0; j < K; ++j) {
    if (DEST) {
      ok[j] = (words.e[j] >= 0) & (words.e[j] < a.E * a.C);
      row[j] = ok[j] ? static_cast<size_t>(words.e[j]) : 0;
    } else {
      ok[j] = (words.e[j] >= 0) & (words.e[j] < a.E) & (words.l[j] >= 0) & (words.l[j] < a.C);
      row[j] = ok[j] ? (static_cast<size_t>(words.e[j]) * a.C + words.l[j]) : 0;
    }
    any = any || ok[j];
  }
  if constexpr (MODE == kWhole16 || MODE == kAny16) {
    typedef Granule<MODE> G;
    const uint32_t row_bytes = static_cast<uint32_t>(a.M) * static_cast<uint32_t>(sizeof(typename Cd::S));
    const int row_vecs = granules_of(row_bytes);
    LANCET_GLOBAL char* dst = as_global(static_cast<char*>(a.out) + static_cast<size_t>(s) * row_bytes);
    const char* src[K];
#pragma unroll
    for (int j = 0; j < K; ++j) src[j] = static_cast<const char*>(a.expert_out) + row[j] * row_bytes;
    const u32x4 z = {0u, 0u, 0u, 0u};
    int v = h.v;
    if (!any) {
      for (; v < row_vecs; v += step) G::st(dst + G::at(v, row_bytes), z);
      return;
    }
    // two granules in flight per slot; the weights are looked at behind the first loads
    u32x4 xa[K], xb[K];
    const auto load = [&](int u) {
#pragma unroll
      for (int j = 0; j < K; ++j) {
        xa[j] = xb[j] = z;
        if (ok[j] && u < row_vecs) xa[j] = G::ld(src[j] + G::at(u, row_bytes));
        if (ok[j] && u + step < row_vecs) xb[j] = G::ld(src[j] + G::at(u + step, row_bytes));
      }
    };
    load(v);
    float g[K];
#pragma unroll
    for (int j = 0; j < K; ++j) g[j] = words.weight(j, ok[j]);
    for (;;) {
      if (v < row_vecs) G::st(dst + G::at(v, row_bytes), combine_vec<DT, K>(xa, g));
      if (v + step < row_vecs) G::st(dst + G::at(v + step, row_bytes), combine_vec<DT, K>(xb, g));
      v += 2 * step;
      if (v >= row_vecs) break;
      load(v);
    }
  } else {
    typedef typename Cd::S St;
    St* dst = static_cast<St*>(a.out) + static_cast<size_t>(s) * a.M;
    const St* base = static_cast<const St*>(a.expert_out);
    float g[K];
#pragma unroll
    for (int j = 0; j < K; ++j) g[j] = words.weight(j, ok[j]);
    for (int i = h.v; i < a.M; i += step) {
#pragma clang fp contract(off)
      float acc = ok[0] ? mul_rn(g[0], Cd::get(base[row[0] * a.M + i])) : 0.f;
      if (K == 2) acc = add_rn(acc, ok[1] ? mul_rn(g[1], Cd::get(base[row[1] * a.M + i])) : 0.f);
      dst[i] = Cd::put(acc);
    }
  }
}

// ---------------------------------------------------------------------------------------
// merge_masks / redispatch.  Both need kept[p][e] = number of tokens of partition p routed to
// expert e; one counting pass over the masks (the reference re-counts with a tree reduction in
// each of its E blocks, tutel_moe_dispatch.cu:238-253,377-392).
// ---------------------------------------------------------------------------------------
constexpr int kCountPerThread = 4;

__global__ __launch_bounds__(kTile) void count_experts_kernel(PtrTable t, int S, int E, uint32_t* counts) {
  extern __shared__ uint32_t hist[];
  const int p = blockIdx.y;
  const int32_t* idx = static_cast<const int32_t*>(t.p[p]);
  for (int c = threadIdx.x; c < E; c += kTile) hist[c] = 0;
  __syncthreads();
  const int base = blockIdx.x * kTile * kCountPerThread;
#pragma unroll
  for (int k = 0; k < kCountPerThread; ++k) {
    const int i = base + k * kTile + threadIdx.x;
    if (i < S) {
      const int e = idx[i];
      if (e >= 0 && e < E) atomicAdd(&hist[e], 1u);
    }
  }
  __syncthreads();
  for (int c = threadIdx.x; c < E; c += kTile)
    if (hist[c]) atomicAdd(counts + static_cast<size_t>(p) * E + c, hist[c]);
}

// Partitions of up to kCountWhole tokens: one workgroup counts a partition alone, sixteen tokens a thread at most, so that
// nothing has to be cleared first and no counter is shared between workgroups.  Bound by the LDS atomics of its one CU,
// which run one after the other where they meet in a counter: every counter has kCountCopies copies side by side, one per
// lane modulo their number.  moe_merge_masks, four partitions, 64 experts, in us: clearing and counting in several
// workgroups / one workgroup with one copy / with sixteen
//   8192 tokens, even 6.4 / 5.2 / 5.1, seven in ten on one expert 6.6 / 9.4 / 5.4
//   16384 tokens, even 6.4 / 5.9 / 5.9, all on one expert 6.8 / 18.5 / 5.9
// (8 copies are up to 8 % slower there, 32 the same).  Beyond kCountWhole the one CU's share grows and the launches' does not.
constexpr int kCountWhole = 16384;
constexpr int kCountThreads = 1024;
constexpr int kCountCopies = 16;
static_assert(LANCET_MAX_EXPERTS * kCountCopies * sizeof(uint32_t) <= 32768, "LDS a launch may have by default, twice over");
__global__ __launch_bounds__(kCountThreads) void count_experts_whole_kernel(PtrTable t, int S, int E, uint32_t* counts) {
  extern __shared__ uint32_t hist[];
  const int p = blockIdx.x;
  const int32_t* idx = static_cast<const int32_t*>(t.p[p]);
  for (int c = threadIdx.x; c < E * kCountCopies; c += kCountThreads) hist[c] = 0;
  __syncthreads();
  constexpr int kBatch = 8;  // loads in flight per thread
  const int copy = threadIdx.x % kCountCopies;
  for (int i = threadIdx.x; i < S; i += kBatch * kCountThreads) {
    int e[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) e[k] = i + k * kCountThreads < S ? idx[i + k * kCountThreads] : -1;
#pragma unroll
    for (int k = 0; k < kBatch; ++k)
      if (e[k] >= 0 && e[k] < E) atomicAdd(&hist[e[k] * kCountCopies + copy], 1u);
  }
  __syncthreads();
  for (int c = threadIdx.x; c < E; c += kCountThreads) {
    uint32_t n = 0;
#pragma unroll
    for (int k = 0; k < kCountCopies; ++k) n += hist[c * kCountCopies + (k + c) % kCountCopies];  // (neighbours in other banks)
    counts[static_cast<size_t>(p) * E + c] = n;
  }
}

// out[0, p*S+i] = idx, out[1, p*S+i] = loc + sum_{q<p} kept[q][idx]; dropped -> (-1,-1)
// (tutel_moe_dispatch.cu:214-236).
__global__ __launch_bounds__(kTile) void merge_masks_kernel(PtrTable t, int P, int S, int E,
                                                            const uint32_t* counts, int32_t* out) {
  extern __shared__ uint32_t s_off[];
  const int p = blockIdx.y;
  for (int c = threadIdx.x; c < E; c += kTile) {
    uint32_t off = 0;
    for (int q = 0; q < p; ++q) off += counts[static_cast<size_t>(q) * E + c];
    s_off[c] = off;
  }
  __syncthreads();
  const int i = blockIdx.x * kTile + threadIdx.x;
  if (i >= S) return;
  const int32_t* il = static_cast<const int32_t*>(t.p[p]);
  const int e = il[i];
  const int l = il[S + i];
  const bool kept = e >= 0 && e < E;
  const size_t o = static_cast<size_t>(p) * S + i;
  out[o] = kept ? e : -1;
  out[static_cast<size_t>(P) * S + o] = kept ? l + static_cast<int>(s_off[e]) : -1;
}

// out[e, off_p[e] + r, :] = buf_p[e, r, :] for r < kept[p][e]; other rows zero
// (tutel_moe_dispatch.cu:365-408, which leaves them uninitialised).
template <int MODE>
__global__ __launch_bounds__(kTile) void redispatch_rows_kernel(PtrTable bufs, int P, int E, int C, uint32_t row_bytes,
                                                                int row_vecs, int wpr_shift,
                                                                const uint32_t* counts, char* out) {
  typedef Granule<MODE> G;
  typedef typename G::V V;
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const uint32_t gw = blockIdx.x * static_cast<uint32_t>(kRowsPerBlock) + w;
  const long r = gw >> wpr_shift;
  const int part = static_cast<int>(gw & ((1u << wpr_shift) - 1u));
  const int step = kWave << wpr_shift;
  if (r >= static_cast<long>(E) * C) return;
  const int e = static_cast<int>(r / C);
  const int c = static_cast<int>(r - static_cast<long>(e) * C);
  // which partition holds row c of expert e: lane q takes partition q's count (P <= 64), an inclusive scan
  // over the lanes gives every partition's row range, one ballot finds the owner
  const uint32_t k = lane < P ? counts[static_cast<size_t>(lane) * E + e] : 0u;
  uint32_t incl = k;
#pragma unroll
  for (int o = 1; o < kWave; o <<= 1) {
    const uint32_t t = __shfl_up(incl, o, kWave);
    if (lane >= o) incl += t;
  }
  const uint32_t excl = incl - k;
  const uint64_t owner = __ballot(lane < P && static_cast<uint32_t>(c) >= excl && static_cast<uint32_t>(c) < incl);
  LANCET_GLOBAL char* dst = as_global(out + static_cast<size_t>(r) * row_bytes);
  if (owner) {
    const int q = __ffsll(static_cast<unsigned long long>(owner)) - 1;
    const int off = static_cast<int>(__shfl(excl, q, kWave));
    const char* src = static_cast<const char*>(bufs.p[q]) + (static_cast<size_t>(e) * C + (c - off)) * row_bytes;
    int v = part * kWave + lane;
    for (; v + step < row_vecs; v += 2 * step) {
      const uint32_t o0 = G::at(v, row_bytes), o1 = G::at(v + step, row_bytes);
      const V x0 = G::ld(src + o0), x1 = G::ld(src + o1);
      G::st(dst + o0, x0);
      G::st(dst + o1, x1);
    }
    if (v < row_vecs) {
      const uint32_t o0 = G::at(v, row_bytes);
      G::st(dst + o0, G::ld(src + o0));
    }
  } else {
    for (int v = part * kWave + lane; v < row_vecs; v += step) G::st(dst + G::at(v, row_bytes), G::zero());
  }
}

// ---------------------------------------------------------------------------------------
// redispatch_expert_input: merge of P partitions of one local expert's all-to-all output, layout
// [C, G, M] (capacity row, source GPU, model dim).  For source g the partitions' received element
// streams (recv_cnts_p[g*LE + le] * scale elements each, stored from row 0 of partition p) are
// concatenated: stream element x lands at out[x / M, g, x % M]
// (redispatch_expert_input_kernel_CGM, tutel_moe_dispatch.cu:436-456, 586-598).  Rows past the merged
// stream are zero-filled (the reference leaves them as they were).  One wave per output row (c, g);
// whole rows are moved in 16-byte granules when every count is a multiple of M.
// ---------------------------------------------------------------------------------------
struct CountTable {
  const uint64_t* p[kMaxPartitions];
};

// EL = element storage type; VEC = rows and pointers allow 16-byte granules (the row-aligned case then
// moves whole rows with them; streams that are not row aligned always take the element path).
template <typename EL, bool VEC>
__global__ __launch_bounds__(kTile) void redispatch_expert_input_kernel(PtrTable bufs, CountTable cnts, int P,
                                                                        int le, int LE, int C, int M, int G,
                                                                        uint64_t scale, EL* out) {
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  const long r = static_cast<long>(blockIdx.x) * kRowsPerBlock + w;  // output row index c*G + g
  if (r >= static_cast<long>(C) * G) return;
  const int c = static_cast<int>(r / G);
  const int g = static_cast<int>(r - static_cast<long>(c) * G);
  EL* dst = out + static_cast<size_t>(r) * M;
  const uint64_t x0 = static_cast<uint64_t>(c) * M;  // first stream element of this row
  uint64_t cum = 0, cum0 = 0;
  int p0 = -1;
  bool rows_only = true;
  for (int q = 0; q < P; ++q) {
    const uint64_t n = cnts.p[q][static_cast<size_t>(g) * LE + le] * scale;
    rows_only = rows_only && (n % M == 0);
    if (p0 < 0 && x0 < cum + n) {
      p0 = q;
      cum0 = cum;
    }
    cum += n;
  }
  const uint64_t total = cum;
  constexpr int kPer = 16 / sizeof(EL);
  if (x0 >= total) {  // past the merged stream
    if (VEC) {
      const u32x4 z = {0u, 0u, 0u, 0u};
      for (int v = lane; v < M / kPer; v += kWave) st_stream(reinterpret_cast<u32x4*>(dst) + v, z);
    } else {
      for (int i = lane; i < M; i += kWave) dst[i] = EL(0);
    }
    return;
  }
  if (rows_only) {
    const uint64_t src_row = (x0 - cum0) / M;
    const bool readable = src_row < static_cast<uint64_t>(C);  // counts larger than the buffer read nothing
    const EL* src = static_cast<const EL*>(bufs.p[p0]) + (readable ? (src_row * G + g) * M : 0);
    if (VEC) {
      const u32x4 z = {0u, 0u, 0u, 0u};
      for (int v = lane; v < M / kPer; v += kWave)
        st_stream(reinterpret_cast<u32x4*>(dst) + v, readable ? ld_stream(reinterpret_cast<const u32x4*>(src) + v) : z);
    } else {
      for (int i = lane; i < M; i += kWave) dst[i] = readable ? src[i] : EL(0);
    }
    return;
  }
  // element-granular streams: every element finds its partition
  for (int i = lane; i < M; i += kWave) {
    const uint64_t x = x0 + i;
    EL val = EL(0);
    if (x < total) {
      uint64_t run = 0;
      for (int q = 0; q < P; ++q) {
        const uint64_t n = cnts.p[q][static_cast<size_t>(g) * LE + le] * scale;
        if (x < run + n) {
          const uint64_t y = x - run;
          const uint64_t sr = y / M;
          if (sr < static_cast<uint64_t>(C)) val = static_cast<const EL*>(bufs.p[q])[(sr * G + g) * M + (y - sr * M)];
          break;
        }
        run += n;
      }
    }
    dst[i] = val;
  }
}

// ---------------------------------------------------------------------------------------
// backward kernels.  moe_encode_dx is decode_rows_kernel with unit gates
// (encode_backward_data_kernel, tutel_moe_dispatch.cu:88-94).
// ---------------------------------------------------------------------------------------
// grad_gates[s, e] = dy[j*S+s] where e is token s's expert in slot j, else 0: the memset + scatter of
// encode_backward_gate_kernel (tutel_moe_dispatch.cu:96-105, 499-506) as one pass that writes every
// element once.
template <int K>
__global__ __launch_bounds__(kTile) void encode_dg_kernel(const void* dy, const int32_t* idx, int S, int E,
                                                          void* grad_gates, int gd) {
  const size_t n = static_cast<size_t>(S) * E;
  for (size_t i = blockIdx.x * static_cast<size_t>(kTile) + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * kTile) {
    const int s = static_cast<int>(i / E);
    const int e = static_cast<int>(i - static_cast<size_t>(s) * E);
    float v = 0.f;
    if (idx[s] == e) v = ld_gate(dy, s, gd);
    if (K == 2 && idx[S + s] == e) v = ld_gate(dy, static_cast<size_t>(S) + s, gd);
    st_gate(grad_gates, i, v, gd);
  }
}

// src[e*C + l] = slot-token id (j*S + s) of the token that owns row (e, l); rows nobody owns keep what lies there.
__global__ __launch_bounds__(kTile) void inverse_map_kernel(const int32_t* idx, const int32_t* loc, int n, int E,
                                                            int C, int32_t* src) {
  const int i = blockIdx.x * kTile + threadIdx.x;
  if (i >= n) return;
  const int e = idx[i], l = loc[i];
  if (e >= 0 && e < E && l >= 0 && l < C) src[static_cast<size_t>(e) * C + l] = i;
}

// The slot-token that owns a row, or -1.  A map that was not cleared beforehand is checked (kClearedRows): an entry counts if the
// slot it names is routed to that row, which whatever else lies there is not.  f(i) asks for what else is needed of the slot named
// together with its routing words: behind them it would be one more round trip in front of the row.
template <typename F>
__device__ __forceinline__ int row_owner(const int32_t* src, size_t row, const int32_t* idx, const int32_t* loc, int n, int E, int C, bool checked, F f) {
  const int i = src[row];
  if (i < 0 || i >= n) return -1;
  if (!checked) {
    f(i);
    return i;
  }
  const int e = idx[i], l = loc[i];
  f(i);
  return e >= 0 && e < E && l >= 0 && l < C && static_cast<size_t>(e) * C + l == row ? i : -1;
}

// grad_expert_out[e, l, :] = gates[i] * dy[s, :] for the slot-token i = src[e*C+l] (s = i mod S), zero
// for rows nobody owns: decode_backward_data_kernel (tutel_moe_dispatch.cu:118-124, 523-533) without
// the memset + atomicAdd; every output byte is written once.
template <int DT, int MODE, int K>
__global__ __launch_bounds__(kTile) void decode_dx_rows_kernel(const void* dy, const void* gates, int gd,
                                                               const int32_t* src, const int32_t* idx, const int32_t* loc,
                                                               void* out, int S, int M, int E, int C, long rows, int q, bool checked) {
  typedef Codec<DT> Cd;
  const RowShare h = row_share(q);
  const long r = h.r;
  const int step = h.step;
  if (r >= rows) return;
  // the weight first, then the row: with both asked for at once the reads crowd out the writes here (262144 x 512 bf16
  // top-1: 83 against 90 us)
  float g1[1] = {0.f};
  const int i = row_owner(src, static_cast<size_t>(r), idx, loc, K * S, E, C, checked, [&](int slot) { g1[0] = ld_gate(gates, slot, gd); });
  const size_t s = i >= 0 ? static_cast<size_t>(i % S) : 0;
  if constexpr (MODE == kWhole16 || MODE == kAny16) {
    typedef Granule<MODE> G;
    const uint32_t row_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(sizeof(typename Cd::S));
    const int row_vecs = granules_of(row_bytes);
    LANCET_GLOBAL char* dst = as_global(static_cast<char*>(out) + static_cast<size_t>(r) * row_bytes);
    const u32x4 z = {0u, 0u, 0u, 0u};
    int v = h.v;
    if (i < 0) {
      for (; v < row_vecs; v += step) G::st(dst + G::at(v, row_bytes), z);
      return;
    }
    const auto ld = [](const char* q) { return K == 2 ? G::ld_keep(q) : G::ld(q); };
    const char* sp = static_cast<const char*>(dy) + s * row_bytes;
    for (; v + step < row_vecs; v += 2 * step) {
      const uint32_t oa = G::at(v, row_bytes), ob = G::at(v + step, row_bytes);
      const u32x4 xa[1] = {ld(sp + oa)};
      const u32x4 xb[1] = {ld(sp + ob)};
      G::st(dst + oa, combine_vec<DT, 1>(xa, g1));
      G::st(dst + ob, combine_vec<DT, 1>(xb, g1));
    }
    if (v < row_vecs) {
      const uint32_t oa = G::at(v, row_bytes);
      const u32x4 xa[1] = {ld(sp + oa)};
      G::st(dst + oa, combine_vec<DT, 1>(xa, g1));
    }
  } else {
    typedef typename Cd::S St;
    St* dst = static_cast<St*>(out) + static_cast<size_t>(r) * M;
    const St* sp = static_cast<const St*>(dy) + s * M;
    for (int k = h.v; k < M; k += step)
      dst[k] = i >= 0 ? Cd::put(mul_rn(g1[0], Cd::get(sp[k]))) : Cd::put(0.f);
  }
}

// acc + the products of the elements of two granules, in order, one rounding per element.  (Spelled out: left to itself
// the compiler moves sums into the chains it finds, or takes fp16 elements two at a time.)
template <int DT>
__device__ __forceinline__ float dot_vec(const u32x4& x, const u32x4& y, float acc) {
#pragma clang fp contract(off)
  typedef Codec<DT> Cd;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (Cd::kPerVec == 4) {
      acc = __builtin_fmaf(Cd::get(x[k]), Cd::get(y[k]), acc);
    } else {
      acc = __builtin_fmaf(Cd::get(static_cast<typename Cd::S>(x[k] & 0xffffu)), Cd::get(static_cast<typename Cd::S>(y[k] & 0xffffu)), acc);
      acc = __builtin_fmaf(Cd::get(static_cast<typename Cd::S>(x[k] >> 16)), Cd::get(static_cast<typename Cd::S>(y[k] >> 16)), acc);
    }
  }
  return acc;
}
// The sum of the products of two granules.  Where a lane takes several granules of a row, each has a sum of its own (one
// chain over both has up to a fifth more error against 64 bits: rows of 256 fp16 values 8.5e-8, so 7.6e-8), which makes the
// sum over a row of up to 64 granules the same tree however many a lane takes.  Granules of rows that end inside one are
// summed in pairs, as such rows have long been walked by a lane per element, without a chain.
template <int DT, int MODE>
__device__ __forceinline__ float dot_granule(const u32x4& x, const u32x4& y) {
  if (MODE == kWhole16) return dot_vec<DT>(x, y, 0.f);
  typedef Codec<DT> Cd;
  const auto pair = [&](int k) {  // both elements of word k (fp32: of words k and k + 1)
    if (Cd::kPerVec == 4) return __builtin_fmaf(Cd::get(x[k]), Cd::get(y[k]), mul_rn(Cd::get(x[k + 1]), Cd::get(y[k + 1])));
    return __builtin_fmaf(Cd::get(static_cast<typename Cd::S>(x[k] & 0xffffu)), Cd::get(static_cast<typename Cd::S>(y[k] & 0xffffu)),
                          mul_rn(Cd::get(static_cast<typename Cd::S>(x[k] >> 16)), Cd::get(static_cast<typename Cd::S>(y[k] >> 16))));
  };
  if (Cd::kPerVec == 4) return add_rn(pair(0), pair(2));
  return add_rn(add_rn(pair(0), pair(1)), add_rn(pair(2), pair(3)));
}
// a granule with its first n bytes (whole elements) as zeros: the last granule of a row that was drawn back over bytes
// another lane has already counted.  (Of both factors of a product: zero times infinity is no zero.)
template <int DT>
__device__ __forceinline__ u32x4 drop_bytes(u32x4 x, uint32_t n) {
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    if (4u * k + 4u <= n) x[k] = 0u;
    else if (Codec<DT>::kPerVec == 8 && 4u * k + 2u == n) x[k] &= 0xffff0000u;
  }
  return x;
}

// grad_gates_s[i] = <expert_out[idx, loc, :], dy[s, :]> for slot-token i, 0 when the slot is dropped
// (decode_backward_gate_kernel, tutel_moe_dispatch.cu:126-157): at most a wave per slot-token, fp32 partial
// sums per lane, xor-tree over its lanes.
template <int DT, int MODE>
__global__ __launch_bounds__(kTile) void decode_dg_kernel(const void* dy, const void* expert_out,
                                                          const int32_t* idx, const int32_t* loc, void* out, int gd,
                                                          int S, int M, int E, int C, int n, int q) {
  typedef Codec<DT> Cd;
  const RowShare h = row_share(q);  // at most a wave
  const int i = h.r;
  if (i >= n) return;
  const int e = idx[i], l = loc[i];
  if (!((e >= 0) & (e < E) & (l >= 0) & (l < C))) {
    if (h.v == 0) st_gate(out, i, 0.f, gd);
    return;
  }
  const size_t s = static_cast<size_t>(i % S);
  const size_t row = static_cast<size_t>(e) * C + l;
  float acc = 0.f;
  if constexpr (MODE == kWhole16 || MODE == kAny16) {
    typedef Granule<MODE> G;
    const uint32_t row_bytes = static_cast<uint32_t>(M) * static_cast<uint32_t>(sizeof(typename Cd::S));
    const int row_vecs = granules_of(row_bytes);
    const char* a = static_cast<const char*>(expert_out) + row * row_bytes;
    const char* b = static_cast<const char*>(dy) + s * row_bytes;
    if (MODE == kWhole16 && h.step == kWave) {  // many granules per lane: its sum goes on from one to the next
      for (int v = h.v; v < row_vecs; v += kWave) {
        const uint32_t o = G::at(v, row_bytes);
        acc = dot_vec<DT>(G::ld(a + o), G::ld(b + o), acc);
      }
    } else {
      for (int v = h.v; v < row_vecs; v += h.step) {
        const uint32_t o = G::at(v, row_bytes);
        u32x4 x = G::ld(a + o), y = G::ld(b + o);
        if (MODE == kAny16 && o != 16u * static_cast<uint32_t>(v)) {
          const uint32_t n = 16u * static_cast<uint32_t>(v) - o;
          x = drop_bytes<DT>(x, n);
          y = drop_bytes<DT>(y, n);
        }
        acc = add_rn(acc, dot_granule<DT, MODE>(x, y));
      }
    }
  } else {
    typedef typename Cd::S St;
    const St* a = static_cast<const St*>(expert_out) + row * M;
    const St* b = static_cast<const St*>(dy) + s * M;
    for (int k = h.v; k < M; k += h.step) acc += Cd::get(a[k]) * Cd::get(b[k]);
  }
  acc = share_sum(acc, q);
  if (h.v == 0) st_gate(out, i, acc, gd);
}

// ---------------------------------------------------------------------------------------
// decode_dx and decode_dg of one decode in one pass: a token's row of dy is read once, multiplied with the expert rows
// its slots came from (the weights' gradients) and, times each weight, written to the same rows of the gradient.  As two
// ops the row is read four times for top-2: 3.0 instead of 4.6 GB at 65536 x 4096 bf16 top-2, 32 experts.
// Same products and roundings as decode_dx; the dot products of rows of more than 64 granules are summed in another order
// than decode_dg's.
// Workgroups behind the tokens' clear the rows no slot owns.  Which those are, they look up in the inverse map
// (decode_dx) or, in short batches, find out themselves by walking all slots, which saves the launch that makes
// the map (kScanSlots below).
// ---------------------------------------------------------------------------------------
struct DecodeGradArgs {
  const char* dy;          // [S, M]
  const char* expert_out;  // [E, C, M]
  const void* gates;       // [K*S] of gate_dtype
  const int32_t* idx;      // [K*S]
  const int32_t* loc;      // [K*S]
  const int32_t* owner;    // [E*C] slot-token that owns a row (row_owner); null: walk the slots
  char* d_expert_out;      // [E, C, M]
  void* d_gates;           // [K*S] of gate_dtype
  int checked;             // the map was not cleared
  int S, E, C, gate_dtype;
  uint32_t row_bytes;
  int row_vecs;            // granules per row
  int q;                   // 2^q lanes of one workgroup share a token
  int token_blocks;
  int tail_rows;           // rows looked at by one workgroup behind the tokens' (kWave at most)
  int tail_chunks;         // such workgroups per expert
};

// EARLY: every lane has granules of its token for two turns and more; the first two are asked for before the routing words.
template <int DT, int K, int MODE, bool EARLY>
__global__ __launch_bounds__(kTile) void decode_grad_kernel(DecodeGradArgs a) {
  typedef Codec<DT> Cd;
  typedef Granule<MODE> G;
  __shared__ float s_dot[kRowsPerBlock][K];
  __shared__ uint32_t s_owned[2];
  const int w = threadIdx.x / kWave;
  const int lane = threadIdx.x & (kWave - 1);
  if (static_cast<int>(blockIdx.x) >= a.token_blocks) {
    const int tb = blockIdx.x - a.token_blocks;
    const int e = tb / a.tail_chunks;
    const int first = (tb - e * a.tail_chunks) * a.tail_rows;
    const int last = min(first + a.tail_rows, a.C);
    // which of the rows are owned, a bit each: a wave that has rows looks all up at once, one chain of round trips instead of one per
    // row (65536 x 512 bf16 top-2 73.8 -> 71.1 us, 262144 x 512 top-1 173 -> 168)
    const int q = min(a.q, 6);
    uint64_t owned = 0;
    if (a.owner) {
      if (first + (w * kWave >> q) >= last) return;
      owned = __ballot(first + lane < last &&
                       row_owner(a.owner, static_cast<size_t>(e) * a.C + first + lane, a.idx, a.loc, K * a.S, a.E, a.C, a.checked, [](int) {}) >= 0);
    } else {
      if (threadIdx.x < 2) s_owned[threadIdx.x] = 0u;
      __syncthreads();
      for (int i = threadIdx.x; i < K * a.S; i += kTile) {
        const int l = a.loc[i];
        if (a.idx[i] == e && l >= first && l < last) atomicOr(&s_owned[(l - first) >> 5], 1u << ((l - first) & 31));
      }
      __syncthreads();
      owned = s_owned[0] | static_cast<uint64_t>(s_owned[1]) << 32;
    }
    for (int r = first + (static_cast<int>(threadIdx.x) >> q); r < last; r += kTile >> q) {
      if ((owned >> (r - first)) & 1u) continue;
      const size_t row = static_cast<size_t>(e) * a.C + r;
      LANCET_GLOBAL char* dst = as_global(a.d_expert_out + row * a.row_bytes);
      for (int v = threadIdx.x & ((1 << q) - 1); v < a.row_vecs; v += 1 << q) G::st(dst + G::at(v, a.row_bytes), G::zero());
    }
    return;
  }
  const RowShare h = row_share(a.q);
  const int s = h.r, step = h.step;
  float acc[K];
#pragma unroll
  for (int j = 0; j < K; ++j) acc[j] = 0.f;
  if (s < a.S) {
    const char* dy = a.dy + static_cast<size_t>(s) * a.row_bytes;
    int v = h.v;
    u32x4 early[2];
    if constexpr (EARLY) {
      early[0] = G::ld(dy + G::at(v, a.row_bytes));
      early[1] = G::ld(dy + G::at(v + step, a.row_bytes));
    }
    RowWords<K> words;
    words.load(a.idx, a.loc, a.gates, a.gate_dtype, a.S, s);
    bool ok[K];
    const char* src[K];
    LANCET_GLOBAL char* dst[K];
    bool any = false;
#pragma unroll
    for (int j = 0; j < K; ++j) {
      ok[j] = (words.e[j] >= 0) & (words.e[j] < a.E) & (words.l[j] >= 0) & (words.l[j] < a.C);
      const size_t at = ok[j] ? (static_cast<size_t>(words.e[j]) * a.C + words.l[j]) * a.row_bytes : 0;
      src[j] = a.expert_out + at;
      dst[j] = as_global(a.d_expert_out + at);
      any = any || ok[j];
    }
    if constexpr (MODE == kWhole16 || MODE == kAny16) {
      // two granules of the token and of each slot's row in flight
      for (; any && v < a.row_vecs; v += 2 * step) {
        const bool two = v + step < a.row_vecs;
        const uint32_t o[2] = {G::at(v, a.row_bytes), G::at(v + step, a.row_bytes)};
        u32x4 d[2], x[2][K];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          d[b] = G::zero();
          if (EARLY && v == h.v) d[b] = early[b];
          else if (b == 0 || two) d[b] = G::ld(dy + o[b]);
#pragma unroll
          for (int j = 0; j < K; ++j) {
            x[b][j] = G::zero();
            if (ok[j] && (b == 0 || two)) x[b][j] = G::ld(src[j] + o[b]);
          }
        }
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          if (b == 1 && !two) break;
          // for the dot products: without the bytes that another lane has as well
          u32x4 once = d[b];
          if (MODE == kAny16) {
            const uint32_t at = 16u * static_cast<uint32_t>(v + b * step);
            if (o[b] != at) {
              once = drop_bytes<DT>(once, at - o[b]);
#pragma unroll
              for (int j = 0; j < K; ++j) x[b][j] = drop_bytes<DT>(x[b][j], at - o[b]);
            }
          }
#pragma unroll
          for (int j = 0; j < K; ++j) {
            if (!ok[j]) continue;
            const u32x4 dd[1] = {d[b]};
            const float g[1] = {words.weight(j, true)};
            G::st(dst[j] + o[b], combine_vec<DT, 1>(dd, g));
            acc[j] = add_rn(acc[j], dot_granule<DT, MODE>(once, x[b][j]));
          }
        }
      }
    } else {
      for (; any && v < a.row_vecs; v += step) {
        const uint32_t o = G::at(v, a.row_bytes);
        const float d = Cd::get(static_cast<typename Cd::S>(G::ld(dy + o)));
#pragma unroll
        for (int j = 0; j < K; ++j) {
          if (!ok[j]) continue;
          acc[j] += d * Cd::get(static_cast<typename Cd::S>(G::ld(src[j] + o)));
          G::st(dst[j] + o, static_cast<typename G::V>(Cd::put(mul_rn(words.weight(j, true), d))));
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < K; ++j) acc[j] = share_sum(acc[j], a.q);
  if (a.q > 6) {  // the token's waves, all of this workgroup, in order
    if (lane == 0) {
#pragma unroll
      for (int j = 0; j < K; ++j) s_dot[w][j] = acc[j];
    }
    __syncthreads();
    if (h.v == 0) {
#pragma unroll
      for (int j = 0; j < K; ++j) {
        acc[j] = 0.f;
        for (int k = 0; k < (step / kWave); ++k) acc[j] += s_dot[w + k][j];
      }
    }
  }
  if (s < a.S && h.v == 0) {
#pragma unroll
    for (int j = 0; j < K; ++j) st_gate(a.d_gates, static_cast<size_t>(j) * a.S + s, acc[j], a.gate_dtype);
  }
}

// ---------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------
static inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// log2 of the number of lanes that share one row of `units` granules: as few as leave per_lane granules to each, at most
// 2^max_q, so few that the grid stays below 2^30 workgroups.
static inline int row_lanes(long units, long rows, int per_lane, int max_q = 10) {
  int q = 0;
  while (q < max_q && (static_cast<long>(per_lane) << q) < units) ++q;
  while (q > 0 && ((rows << q) + kTile - 1) / kTile > 0x3fffffffL) --q;
  return q;
}
// Few granules in all: the launch is over when its first loads are back, and a second granule per lane only makes the waves
// longer (rows of at most a wave, decode top-1, two / one: 1024 x 192 bf16 2.9 / 2.5 us, 8192 x 128 3.2 / 2.9; 4096 x 384 with
// half as many again 3.4 / 3.7).
static inline bool few_granules(long units, long rows) { return units * rows <= 131072; }
static inline long row_blocks(long rows, int q) { return ((rows << q) + kTile - 1) / kTile; }

// the way rows of row_bytes bytes in arrays at the given addresses are cut
static inline RowMode row_mode(size_t row_bytes, int elem_bytes, bool aligned) {
  if (row_bytes < 16) return elem_bytes == 4 ? kElem4 : kElem2;
  return row_bytes % 16 == 0 && aligned ? kWhole16 : kAny16;
}
// granules of such a row
static inline int row_granules(RowMode mode, size_t row_bytes, int elem_bytes) {
  return static_cast<int>(mode == kWhole16 || mode == kAny16 ? (row_bytes + 15) / 16 : row_bytes / elem_bytes);
}
// MODE as a compile-time constant inside `...` (the second form: for rows of a known type, whose elements have one size)
#define LANCET_CODED_ROW_SWITCH(DT, mode, ...)                         \
  switch (mode) {                                                      \
    case kWhole16: { constexpr int MODE = kWhole16; __VA_ARGS__; } break; \
    case kAny16: { constexpr int MODE = kAny16; __VA_ARGS__; } break;     \
    default: { constexpr int MODE = DT == LANCET_F32 ? kElem4 : kElem2; __VA_ARGS__; } break; \
  }
#define LANCET_ROW_SWITCH(mode, ...)                                   \
  switch (mode) {                                                      \
    case kWhole16: { constexpr int MODE = kWhole16; __VA_ARGS__; } break; \
    case kAny16: { constexpr int MODE = kAny16; __VA_ARGS__; } break;     \
    case kElem2: { constexpr int MODE = kElem2; __VA_ARGS__; } break;     \
    default: { constexpr int MODE = kElem4; __VA_ARGS__; } break;         \
  }

// The scatter of rows that several waves share (more than 1 KB) asks for LDS it does not use, which keeps 5 of its
// workgroups on a CU instead of 8: with all wave slots taken its reads crowd out its writes.  8 / 6 / 5 / 4 / 3 workgroups:
// 344 / 337 / 324 / 350 / 420 us at 65536 x 4096 bf16 top-2, 206 / 208 / 200 / 221 / 243 top-1, 165 against 160 at rows of
// 2048.  Rows of one wave want every slot: 90 / 92 / 99 / 108 us at 262144 x 512.  The gather kernels do not gain.
constexpr size_t kCuLds = 160 * 1024;
constexpr size_t kScatterLds = kCuLds / 6 + 1;  // six do not fit, however LDS is rounded up; five do

// Where the workgroups that clear the experts' tails stand.  Behind the tokens' they are an end of the launch that only
// writes, or, where nearly all find nothing to clear, a row of empty starts; among them they hide behind the rows' traffic, but an
// empty start there costs more than one at the end.  Among them pays for long rows, which need few workgroups of tails per byte, in
// passes that are long themselves.  Behind / among, us, tokens x bytes of a row, arrays that change from call to call:
//   top-1, 40 to 60 % of the buffer filled: 34818 x 2912 64.9 / 60.2, 57288 x 2864 77.5 / 73.8, 135909 x 896 64.1 / 60.9 (the same arrays again
//   and again 62 / 44, 68 / 58, 61 / 52); more filled than that: 141135 x 2352 171 / 170, 34914 x 3456 51.6 / 51.1, 218661 x 1552 120 / 125;
//   top-2, half filled: 19356 x 2112 28.3 / 25.3, 28776 x 2160 38.2 / 35.2, 160407 x 912 98.9 / 94.7; filled: 119178 x 2240 210 / 207, 42771 x 2528 65.4 /
//   68.5, 13773 x 6256 48.9 / 48.3; 16384 x 4096 half filled 40.8 / 36.4 for the whole encode.
// Not for shorter rows and passes: 86769 x 48 top-2 6.5 / 10.8, 83468 x 64 top-1 5.4 / 7.3, 38382 x 448 10.2 / 12.2, 37842 x 1152 34.4 / 39.6, 69009 x 1216
// top-1 37.1 / 39.3, 12474 x 1536 11.5 / 11.9; nor for top-1 rows of more than 4 KB, whose reads and writes are in balance without (65536 x 8192
// 211.2 / 214.0, 45919 x 4752 107 / 119); nor for rows that end inside a granule (10007 x 2006 24.8 / 25.6).  At most
// kMixedTails of them, each then with several turns: one eight in four at 65536 x 2048 93.2, one in five 90.0 (behind: 91.3).
constexpr size_t kMixedRowBytes = 1536, kMixedBytes = size_t(64) << 20;
constexpr size_t kMixedLongRowBytes = 768, kMixedLongBytes = size_t(256) << 20;
constexpr size_t kMixedTop1Bytes = 4096;
constexpr int kMixedTails = 8192;
constexpr long kMixedBlocks = 1L << 19;  // up to here the multiplication by tail_inverse divides exactly
static bool tails_among_tokens(size_t row_bytes, int S, int E, int C, int K) {
  const size_t pass = (static_cast<size_t>(S) + static_cast<size_t>(E) * C) * row_bytes;
  if (E > kMixedTails || (K == 1 && row_bytes > kMixedTop1Bytes)) return false;
  return (row_bytes >= kMixedRowBytes && pass >= kMixedBytes) || (row_bytes >= kMixedLongRowBytes && pass >= kMixedLongBytes);
}

hipError_t run_scatter_rows(const void* data, void* out, const int32_t* idx, const int32_t* loc,
                            const int32_t* avail_used, const int32_t* row_base, const int32_t* rows_lo,
                            const int32_t* rows_hi,
                            int S, int M, int E, int C, int K, int elem_bytes, hipStream_t st, int slot_stride,
                            const int32_t* dest) {
  const size_t row_bytes = static_cast<size_t>(M) * elem_bytes;
  if (row_bytes == 0) return hipSuccess;
  const RowMode mode = row_mode(row_bytes, elem_bytes, aligned16(data) && aligned16(out));
  if (dest && mode != kWhole16) return hipErrorInvalidValue;  // the one-word form is for rows of 16-byte granules
  ScatterArgs a;
  a.dest = dest;
  a.data = static_cast<const char*>(data);
  a.out = static_cast<char*>(out);
  a.idx = idx;
  a.loc = loc;
  a.avail_used = avail_used;
  a.row_base = row_base;
  a.rows_lo = rows_lo;
  a.rows_hi = rows_hi;
  a.S = S;
  a.E = E;
  a.C = C;
  a.K = K;
  a.slot_stride = slot_stride < 0 ? S : slot_stride;
  a.row_bytes = static_cast<uint32_t>(row_bytes);  // M < 2^30
  a.row_vecs = row_granules(mode, row_bytes, elem_bytes);
  a.q = row_lanes(a.row_vecs, S, 1);
  a.token_blocks = static_cast<int>(row_blocks(S, a.q));
  a.tail_chunks = rows_hi ? (C + kTailRows - 1) / kTailRows : 0;
  a.tail_groups = a.tail_every = 0, a.tail_inverse = 0u;
  long blocks = static_cast<long>(a.token_blocks) + static_cast<long>(a.tail_chunks) * E;
  if (a.tail_chunks && a.token_blocks && mode == kWhole16 && tails_among_tokens(row_bytes, S, E, C, K)) {
    const int chunks = std::min(a.tail_chunks, kMixedTails / E), groups = (chunks * E + kXcds - 1) / kXcds;
    const long mixed = static_cast<long>(a.token_blocks) + static_cast<long>(groups) * kXcds;
    const int every = static_cast<int>(mixed / kXcds / groups);
    if (every >= 2 && mixed <= kMixedBlocks) {  // (more tails than tokens would stand in front of them)
      a.tail_chunks = chunks, a.tail_groups = groups, a.tail_every = every;
      a.tail_inverse = static_cast<uint32_t>((0x100000000ull + static_cast<uint64_t>(every) - 1) / static_cast<uint64_t>(every));
      blocks = mixed;
    }
  }
  if (blocks == 0) return hipSuccess;
  const size_t lds = a.row_vecs > kWave ? kScatterLds : 0;
  if (dest) {
    if (K == 1) scatter_rows_kernel<kWhole16, 1, true><<<static_cast<unsigned>(blocks), kTile, lds, st>>>(a);
    else scatter_rows_kernel<kWhole16, 2, true><<<static_cast<unsigned>(blocks), kTile, lds, st>>>(a);
    return hipGetLastError();
  }
  LANCET_ROW_SWITCH(mode,
    if (K == 1) scatter_rows_kernel<MODE, 1><<<static_cast<unsigned>(blocks), kTile, lds, st>>>(a);
    else scatter_rows_kernel<MODE, 2><<<static_cast<unsigned>(blocks), kTile, lds, st>>>(a))
  return hipGetLastError();
}

hipError_t run_zero_bytes(void* p, size_t nbytes, hipStream_t st) {
  if (nbytes == 0) return hipSuccess;
  uint8_t* b = static_cast<uint8_t*>(p);
  // head bytes up to 16-byte alignment are cleared together with the tail by a second launch
  const size_t head = (16 - (reinterpret_cast<uintptr_t>(b) & 15u)) & 15u;
  const size_t h = std::min(head, nbytes);
  if (h) {
    zero_bytes_kernel<<<1, 64, 0, st>>>(nullptr, 0, b, h);
    b += h;
    nbytes -= h;
  }
  const size_t nvec = nbytes / 16;
  const size_t ntail = nbytes - nvec * 16;
  if (nvec || ntail) {
    // one granule per thread up to 2^22 workgroups (16 GiB), a loop beyond that
    const int blocks = static_cast<int>(std::min<size_t>((nvec + 255) / 256 + 1, size_t(1) << 22));
    zero_bytes_kernel<<<blocks, 256, 0, st>>>(reinterpret_cast<u32x4*>(b), nvec, b + nvec * 16, ntail);
  }
  return hipGetLastError();
}

template <int DT>
static hipError_t decode_launch(DecodeArgs a, int K, RowMode mode, hipStream_t st) {
  if (a.S == 0 || a.M == 0) return hipSuccess;
  constexpr int eb = sizeof(typename Codec<DT>::S);
  const int units = row_granules(mode, static_cast<size_t>(a.M) * eb, eb);
  const bool few = few_granules(units, a.S);
  const bool spare = units > kWave && (units & (units - 1)) != 0 && !few;
  a.q = row_lanes(units, a.S, K == 1 ? (few && units <= kWave ? 1 : 2) : (spare ? 2 : 1));
  const unsigned blocks = static_cast<unsigned>(row_blocks(a.S, a.q));
  if (a.dest) {
    if (mode != kWhole16) return hipErrorInvalidValue;
    if (K == 1) decode_rows_kernel<DT, 1, kWhole16, true><<<blocks, kTile, 0, st>>>(a);
    else decode_rows_kernel<DT, 2, kWhole16, true><<<blocks, kTile, 0, st>>>(a);
    return hipGetLastError();
  }
  LANCET_CODED_ROW_SWITCH(DT, mode,
    if (K == 1) decode_rows_kernel<DT, 1, MODE><<<blocks, kTile, 0, st>>>(a);
    else decode_rows_kernel<DT, 2, MODE><<<blocks, kTile, 0, st>>>(a))
  return hipGetLastError();
}

hipError_t run_decode_rows(const void* expert_out, const void* gates, int gate_dtype, const int32_t* idx,
                           const int32_t* loc, void* out, int S, int M, int E, int C, int K,
                           int dtype, hipStream_t st, int slot_stride, const int32_t* dest) {
  DecodeArgs a;
  a.dest = dest;
  a.expert_out = expert_out;
  a.gates = gates;
  a.gate_dtype = gate_dtype;
  a.idx = idx;
  a.loc = loc;
  a.out = out;
  a.S = S;
  a.M = M;
  a.E = E;
  a.C = C;
  a.slot_stride = slot_stride < 0 ? S : slot_stride;
  const int eb = dtype == LANCET_F32 ? 4 : 2;
  const RowMode mode = row_mode(static_cast<size_t>(M) * eb, eb, aligned16(expert_out) && aligned16(out));
  switch (dtype) {
    case LANCET_F32: return decode_launch<LANCET_F32>(a, K, mode, st);
    case LANCET_BF16: return decode_launch<LANCET_BF16>(a, K, mode, st);
    default: return decode_launch<LANCET_F16>(a, K, mode, st);
  }
}

hipError_t run_count_experts(const PtrTable& indlocs, int P, int S, int E, uint32_t* counts, hipStream_t st) {
  if (S <= kCountWhole) {
    if (P == 0 || E == 0) return hipSuccess;
    count_experts_whole_kernel<<<P, kCountThreads, E * kCountCopies * sizeof(uint32_t), st>>>(indlocs, S, E, counts);
    return hipGetLastError();
  }
  hipError_t err = run_fill_u32(counts, static_cast<size_t>(P) * E, 0u, st);
  if (err != hipSuccess) return err;
  dim3 grid((S + kTile * kCountPerThread - 1) / (kTile * kCountPerThread), P);
  count_experts_kernel<<<grid, kTile, E * sizeof(uint32_t), st>>>(indlocs, S, E, counts);
  return hipGetLastError();
}

hipError_t run_merge_masks(const PtrTable& indlocs, int P, int S, int E, const uint32_t* counts,
                           int32_t* out, hipStream_t st) {
  if (S == 0) return hipSuccess;
  dim3 grid((S + kTile - 1) / kTile, P);
  merge_masks_kernel<<<grid, kTile, E * sizeof(uint32_t), st>>>(indlocs, P, S, E, counts, out);
  return hipGetLastError();
}

hipError_t run_redispatch_rows(const PtrTable& bufs, int P, int M, int C, int E, const uint32_t* counts,
                               void* out, int elem_bytes, hipStream_t st) {
  const size_t row_bytes = static_cast<size_t>(M) * elem_bytes;
  const long rows = static_cast<long>(E) * C;
  if (rows == 0 || row_bytes == 0) return hipSuccess;
  bool aligned = aligned16(out);
  for (int p = 0; p < P; ++p) aligned = aligned && aligned16(bufs.p[p]);
  const RowMode mode = row_mode(row_bytes, elem_bytes, aligned);
  const int units = row_granules(mode, row_bytes, elem_bytes);
  const int shift = std::max(row_lanes(units, rows, 2), 6) - 6;  // whole waves per row, two granules per lane: 426 -> 408 us
  const unsigned blocks = static_cast<unsigned>(((rows << shift) + kRowsPerBlock - 1) / kRowsPerBlock);
  LANCET_ROW_SWITCH(mode, (redispatch_rows_kernel<MODE><<<blocks, kTile, 0, st>>>(
                              bufs, P, E, C, static_cast<uint32_t>(row_bytes), units, shift, counts, static_cast<char*>(out))))
  return hipGetLastError();
}

hipError_t run_encode_dg(const void* dy, const int32_t* idx, int S, int E, int K, int gate_dtype, void* grad_gates, hipStream_t st) {
  const size_t n = static_cast<size_t>(S) * E;
  if (n == 0) return hipSuccess;
  const int blocks = static_cast<int>(std::min<size_t>((n + kTile - 1) / kTile, 65536));
  if (K == 1) encode_dg_kernel<1><<<blocks, kTile, 0, st>>>(dy, idx, S, E, grad_gates, gate_dtype);
  else encode_dg_kernel<2><<<blocks, kTile, 0, st>>>(dy, idx, S, E, grad_gates, gate_dtype);
  return hipGetLastError();
}

// Rows of the buffer up to which the map is checked instead of cleared.  Clearing is a launch of 2 to 3 us, checking two words more to
// gather per row.  Cleared / checked, us: moe_decode_dx 16384 x 64 bf16 top-1 (20480 rows) 7.8 / 6.1, 32768 x 2048 (40960) 59.0 / 58.0,
// 65536 x 64 (81920) 10.7 / 9.0; 131072 x 16 (163840) 10.9 / 10.3, 107376 x 8 (214752) 8.3 / 6.5, 57693 x 928 top-2 (230820) 94.3 / 91.4, 119642 x 24 top-2 (239400)
// 20.4 / 18.9; 131072 x 64 (163840) 16.0 / 16.5, 262144 x 64 (327680) 25.9 / 27.3, 87380 x 576 top-2 (349520) 112.9 / 113.9, 1000000 x 64 80.3 / 95.4;
// moe_decode_grad 65536 x 1024 82.0 / 80.2, 26295 x 8 top-2 (105184) 9.4 / 7.4, 90630 x 552 top-2 (226610) 142.4 / 138.9, 262144 x 64 35.4 / 35.8.
constexpr long kClearedRows = 262144;

template <int DT>
static hipError_t decode_dx_launch(const void* dy, const void* gates, int gd, const int32_t* src, const int32_t* idx,
                                   const int32_t* loc, void* out, int S, int M, int E, int C, int K, RowMode mode, hipStream_t st) {
  const long rows = static_cast<long>(E) * C;
  constexpr int eb = sizeof(typename Codec<DT>::S);
  const int units = row_granules(mode, static_cast<size_t>(M) * eb, eb);
  const int q = row_lanes(units, rows, few_granules(units, rows) && units <= kWave ? 1 : 2);  // two granules per lane: 442 -> 408 us
  const unsigned blocks = static_cast<unsigned>(row_blocks(rows, q));
  LANCET_CODED_ROW_SWITCH(DT, mode,
    if (K == 1) decode_dx_rows_kernel<DT, MODE, 1><<<blocks, kTile, 0, st>>>(dy, gates, gd, src, idx, loc, out, S, M, E, C, rows, q, rows <= kClearedRows);
    else decode_dx_rows_kernel<DT, MODE, 2><<<blocks, kTile, 0, st>>>(dy, gates, gd, src, idx, loc, out, S, M, E, C, rows, q, rows <= kClearedRows))
  return hipGetLastError();
}

// the inverse map (row_owner)
static hipError_t run_inverse_map(const int32_t* idx, const int32_t* loc, int n, int E, int C, int32_t* src, hipStream_t st) {
  if (static_cast<long>(E) * C > kClearedRows) {
    const hipError_t err = run_fill_u32(reinterpret_cast<uint32_t*>(src), static_cast<size_t>(E) * C, 0xffffffffu, st);
    if (err != hipSuccess) return err;
  }
  if (n == 0) return hipSuccess;
  inverse_map_kernel<<<(n + kTile - 1) / kTile, kTile, 0, st>>>(idx, loc, n, E, C, src);
  return hipGetLastError();
}

hipError_t run_decode_dx(const void* dy, const void* gates, int gate_dtype, const int32_t* idx, const int32_t* loc, void* out,
                         int32_t* src_map, int S, int M, int E, int C, int K, int dtype, hipStream_t st) {
  const long rows = static_cast<long>(E) * C;
  if (rows == 0 || M == 0) return hipSuccess;
  const hipError_t err = run_inverse_map(idx, loc, K * S, E, C, src_map, st);
  if (err != hipSuccess) return err;
  const int eb = dtype == LANCET_F32 ? 4 : 2;
  const RowMode mode = row_mode(static_cast<size_t>(M) * eb, eb, aligned16(dy) && aligned16(out));
  switch (dtype) {
    case LANCET_F32: return decode_dx_launch<LANCET_F32>(dy, gates, gate_dtype, src_map, idx, loc, out, S, M, E, C, K, mode, st);
    case LANCET_BF16: return decode_dx_launch<LANCET_BF16>(dy, gates, gate_dtype, src_map, idx, loc, out, S, M, E, C, K, mode, st);
    default: return decode_dx_launch<LANCET_F16>(dy, gates, gate_dtype, src_map, idx, loc, out, S, M, E, C, K, mode, st);
  }
}

// Slots up to which the clearing workgroups of decode_grad_kernel walk all of them themselves instead of looking rows up in
// a map that the launch before it makes.  Map / walk by workgroups of 64 rows, us: 1024 slots, rows of 64 bf16, 4 experts 4.6 /
// 2.9 and 512 experts 4.9 / 3.0, rows of 2048 6.7 / 8.2 and 6.5 / 4.5; 4096 slots 5.0 / 4.3, 5.3 / 4.9, 13.0 / 15.1 and 12.7 / 11.2; 6000 slots
// rows of 2048 16.0 / 19.1 and 16.1 / 15.5.  Rows of less than 768 bytes, bytes and slots: top-1 144 x 4734 5.8 / 5.6, 48 x 5087 5.6 / 5.3, 16 x
// 5225 5.5 / 5.9, 304 x 6343 6.1 / 7.0; top-2, whose map takes twice the writes, 320 x 4832 7.0 / 6.0, 160 x 5664 6.9 / 5.9, 238 x 6418 7.3 / 6.2, 100 x
// 6982 6.8 / 6.4, 304 x 7426 7.6 / 8.5; longer rows 2102 x 4358 top-1 11.6 / 14.2, 1596 x 5214 top-2 10.7 / 11.7.
constexpr int kScanSlots = 4096, kScanShortSlots1 = 5000, kScanShortSlots2 = 6900;
constexpr size_t kScanShortRow = 768;
constexpr int kGradTailRows = 16;  // rows per clearing workgroup with the inverse map
constexpr int kGradScanRows = 64;  // ... that walks the slots
constexpr size_t kGradWideLds = kCuLds / 5 + 1;  // five workgroups do not fit, four do
constexpr size_t kMemoryCache = size_t(256) << 20;  // what the cache in front of the HBM holds

template <int DT>
static hipError_t decode_grad_launch(DecodeGradArgs a, int K, int M, RowMode mode, hipStream_t st) {
  constexpr int eb = sizeof(typename Codec<DT>::S);
  a.row_bytes = static_cast<uint32_t>(M) * eb;
  a.row_vecs = row_granules(mode, a.row_bytes, eb);
  // The waves of a token are of one workgroup.  Granules per lane, one / two: 65536 x 1024 bf16 top-2 132 / 139 us, rows of
  // 384 60 / 56, 262144 x 512 top-1 114 / 93, rows of 4096 the same; 10007 x 1003 top-2 (unaligned) 26 / 23.
  a.q = row_lanes(a.row_vecs, a.S, K == 2 && a.row_vecs > kWave && mode == kWhole16 ? 1 : 2, 8);
  a.token_blocks = static_cast<int>(row_blocks(a.S, a.q));
  a.tail_rows = a.owner ? kGradTailRows : kGradScanRows;
  a.tail_chunks = (a.C + a.tail_rows - 1) / a.tail_rows;
  const unsigned blocks = static_cast<unsigned>(a.token_blocks + static_cast<long>(a.tail_chunks) * a.E);
  if (blocks == 0) return hipSuccess;
  // top-1 rows of several waves: as in the scatter, 317 against 329 us at 65536 x 4096 bf16 (rows of one wave 182 / 151).
  // top-2 rows with half as many granules again as a workgroup has lanes, of which those keep twice the loads in flight, in passes that
  // come from the HBM: four workgroups on a CU instead of eight (20000 x 3072 bf16 122 against 126 us, 13357 x 11376 bytes 150 / 160, 6797 x
  // 6304 the same; of fewer granules, which most lanes have one of, eight are faster: 17248 x 5040 bytes 85 / 70, 28302 x 4480 129 / 101,
  // 16384 x 4096 66 / 49), and where all lanes have two granules of it the token's row is asked for before the routing words: both
  // together 549 / 570 at 65536 x 4096, 156 / 165 at 20000, 96 / 101 at 12000, 51.3 / 52.7 at 6000.  In the cache neither pays (4200 x
  // 4096 with half as many rows kept 29 / 25), nor the latter for rows of 384 granules (158 / 153) or top-1 (20000 x 4096 92 / 90).
  const bool wide = K == 2 && mode == kWhole16 && 2 * a.row_vecs >= 3 * kTile &&
                    (static_cast<size_t>(a.S) + 2 * static_cast<size_t>(a.E) * a.C) * a.row_bytes > kMemoryCache;
  const size_t lds = wide ? kGradWideLds : K == 1 && a.q > 6 ? kScatterLds : 0;
  if (wide && a.row_vecs >= 2 * kTile) {
    decode_grad_kernel<DT, 2, kWhole16, true><<<blocks, kTile, lds, st>>>(a);
    return hipGetLastError();
  }
  LANCET_CODED_ROW_SWITCH(DT, mode,
    if (K == 1) decode_grad_kernel<DT, 1, MODE, false><<<blocks, kTile, lds, st>>>(a);
    else decode_grad_kernel<DT, 2, MODE, false><<<blocks, kTile, lds, st>>>(a))
  return hipGetLastError();
}

hipError_t run_decode_grad(const void* dy, const void* expert_out, const void* gates, int gate_dtype, const int32_t* idx,
                           const int32_t* loc, void* d_expert_out, void* d_gates, int32_t* src_map, int S, int M, int E,
                           int C, int K, int dtype, hipStream_t st) {
  DecodeGradArgs a;
  a.dy = static_cast<const char*>(dy);
  a.expert_out = static_cast<const char*>(expert_out);
  a.gates = gates;
  a.gate_dtype = gate_dtype;
  a.idx = idx;
  a.loc = loc;
  a.d_expert_out = static_cast<char*>(d_expert_out);
  a.d_gates = d_gates;
  a.S = S;
  a.E = E;
  a.C = C;
  a.owner = nullptr;
  a.checked = 0;
  const int eb = dtype == LANCET_F32 ? 4 : 2;
  const int walked = static_cast<size_t>(M) * eb >= kScanShortRow ? kScanSlots : K == 1 ? kScanShortSlots1 : kScanShortSlots2;
  if (K * static_cast<long>(S) > walked && M > 0 && C > 0) {
    const hipError_t err = run_inverse_map(idx, loc, K * S, E, C, src_map, st);
    if (err != hipSuccess) return err;
    a.owner = src_map;
    a.checked = static_cast<long>(E) * C <= kClearedRows;
  }
  const RowMode mode = row_mode(static_cast<size_t>(M) * eb, eb, aligned16(dy) && aligned16(expert_out) && aligned16(d_expert_out));
  switch (dtype) {
    case LANCET_F32: return decode_grad_launch<LANCET_F32>(a, K, M, mode, st);
    case LANCET_BF16: return decode_grad_launch<LANCET_BF16>(a, K, M, mode, st);
    default: return decode_grad_launch<LANCET_F16>(a, K, M, mode, st);
  }
}

template <int DT>
static hipError_t decode_dg_launch(const void* dy, const void* expert_out, const int32_t* idx, const int32_t* loc,
                                   void* out, int gd, int S, int M, int E, int C, int n, RowMode mode, hipStream_t st) {
  constexpr int eb = sizeof(typename Codec<DT>::S);
  // two granules per lane from 512 bytes on (262144 x 512 bf16 top-1 53 -> 43 us, 65536 x 384 top-2 44 -> 33), one in
  // shorter rows (200000 x 64: 10.6 against 15.5) and, with rows of at most a wave, in launches of up to 262144 granules
  // (4096 x 512 bf16 top-1 3.2 against 3.7)
  const int units = row_granules(mode, static_cast<size_t>(M) * eb, eb);
  const int q = row_lanes(units, n, units >= 32 && !few_granules(units, n / 2) ? 2 : 1, 6);
  LANCET_CODED_ROW_SWITCH(DT, mode, (decode_dg_kernel<DT, MODE><<<static_cast<unsigned>(row_blocks(n, q)), kTile, 0, st>>>(dy, expert_out, idx, loc, out, gd, S, M, E, C, n, q)))
  return hipGetLastError();
}

hipError_t run_decode_dg(const void* dy, const void* expert_out, const int32_t* idx, const int32_t* loc, void* out,
                         int gate_dtype, int S, int M, int E, int C, int K, int dtype, hipStream_t st) {
  const int n = K * S;
  if (n == 0) return hipSuccess;
  const int eb = dtype == LANCET_F32 ? 4 : 2;
  const RowMode mode = row_mode(static_cast<size_t>(M) * eb, eb, aligned16(dy) && aligned16(expert_out));
  switch (dtype) {
    case LANCET_F32: return decode_dg_launch<LANCET_F32>(dy, expert_out, idx, loc, out, gate_dtype, S, M, E, C, n, mode, st);
    case LANCET_BF16: return decode_dg_launch<LANCET_BF16>(dy, expert_out, idx, loc, out, gate_dtype, S, M, E, C, n, mode, st);
    default: return decode_dg_launch<LANCET_F16>(dy, expert_out, idx, loc, out, gate_dtype, S, M, E, C, n, mode, st);
  }
}

hipError_t run_redispatch_expert_input(const PtrTable& bufs, const void* const* cnt_ptrs, int P, int le, int LE, int C,
                                       int M, int G, uint64_t scale, void* out, int elem_bytes, hipStream_t st) {
  const long rows = static_cast<long>(C) * G;
  if (rows == 0 || M == 0) return hipSuccess;
  CountTable ct;
  for (int q = 0; q < kMaxPartitions; ++q) ct.p[q] = q < P ? static_cast<const uint64_t*>(cnt_ptrs[q]) : nullptr;
  const unsigned blocks = static_cast<unsigned>((rows + kRowsPerBlock - 1) / kRowsPerBlock);
  const size_t row_bytes = static_cast<size_t>(M) * elem_bytes;
  bool vec = row_bytes % 16 == 0 && aligned16(out);
  for (int q = 0; q < P; ++q) vec = vec && aligned16(bufs.p[q]);
  if (elem_bytes == 4) {
    if (vec) redispatch_expert_input_kernel<uint32_t, true><<<blocks, kTile, 0, st>>>(bufs, ct, P, le, LE, C, M, G, scale, static_cast<uint32_t*>(out));
    else redispatch_expert_input_kernel<uint32_t, false><<<blocks, kTile, 0, st>>>(bufs, ct, P, le, LE, C, M, G, scale, static_cast<uint32_t*>(out));
  } else {
    if (vec) redispatch_expert_input_kernel<uint16_t, true><<<blocks, kTile, 0, st>>>(bufs, ct, P, le, LE, C, M, G, scale, static_cast<uint16_t*>(out));
    else redispatch_expert_input_kernel<uint16_t, false><<<blocks, kTile, 0, st>>>(bufs, ct, P, le, LE, C, M, G, scale, static_cast<uint16_t*>(out));
  }
  return hipGetLastError();
}

}  // namespace lancet
